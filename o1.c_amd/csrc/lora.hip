// GPU LoRA merge-on-load: W = bf16(float(W) + s * (up @ down)), fp32 delta.
// Replaces hd_lora_merge_gpu (lora_merge.cu:35-104). The delta never reaches
// HBM. Two kernels:
//  - lora_merge_stream_kernel (R <= 64, R % 4 == 0): persistent blocks
//    stream W through registers, rank product on the bf16 matrix cores
//    with fp32 operands split in three bf16 parts; one launch for up to
//    LM_TG targets;
//  - lora_merge_mfma_kernel (any other R): a block per 128 x 128 tile, rank
//    product on the fp32 matrix cores (v_mfma_f32_32x32x2_f32); one launch
//    per target.
#include <stdio.h>

#include <algorithm>
#include <map>
#include <vector>

#include "hd_common.hpp"
#include "../../include/hd_hip.h"
#include "../../include/hd_lora.h"

// A block owns a 128 x 128 tile of W (two blocks per CU); the rank
// product runs on v_mfma_f32_32x32x2_f32 (fp32 products, fp32 accumulation,
// as an SGEMM does). Wave w computes rows [32w, 32w+32) x all 128 columns
// (4 accumulators); MFMA A = up (row = output row), B = down (column = output
// column), so a lane holds 16 rows of one column and the read-modify-write of
// W is coalesced along the row.
#define LM_T 128
#define LM_RC 64
#define LM_SU (LM_T * (LM_RC + 1))          // up slice [row][r], +1: conflict-free column reads
#define LM_SD (LM_RC * (LM_T + 32))         // down slice [r][col], +32: the half-waves read
                                            // consecutive r rows in opposite bank halves
#define LM_ST (LM_T * (LM_T + 8))           // fp32 delta tile [row][col] for the W update
template <int OCC>
__global__ __launch_bounds__(256, OCC) void lora_merge_mfma_kernel(uint16_t *__restrict__ w,
                                                              const float *__restrict__ up,
                                                              const float *__restrict__ down, int N,
                                                              int K, int R, float scale) {
    __shared__ __attribute__((aligned(16))) float lds[LM_SU + LM_SD > LM_ST ? LM_SU + LM_SD : LM_ST];
    float *su = lds, *sd = lds + LM_SU;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = blockIdx.y * LM_T, k0 = blockIdx.x * LM_T;
    const int l32 = lane & 31, lh = lane >> 5;
    const bool full = n0 + LM_T <= N && k0 + LM_T <= K && R % 4 == 0 && K % 8 == 0;
    // W update chunks of this thread: 8 x 8 consecutive weights, loaded
    // before the rank product so their latency hides under it
    u32x4_t wch[8];
    if (full) {
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int c = threadIdx.x + t * 256, row = c / 16, col = (c % 16) * 8;
            wch[t] = *(const u32x4_t *)(w + (size_t)(n0 + row) * K + k0 + col);
        }
    }
    f32x16_t acc[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[j][e] = 0.f;
    for (int r0 = 0; r0 < R; r0 += LM_RC) {
        const int rc = min(LM_RC, R - r0);
        if (full && rc == LM_RC) {
            // all 16 loads in flight before the first LDS store
            float4 ua[8], da[8];
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const int i = threadIdx.x + t * 256;
                ua[t] = *(const float4 *)(up + (size_t)(n0 + i / (LM_RC / 4)) * R + r0 + (i % (LM_RC / 4)) * 4);
                da[t] = *(const float4 *)(down + (size_t)(r0 + i / (LM_T / 4)) * K + k0 + (i % (LM_T / 4)) * 4);
            }
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const int i = threadIdx.x + t * 256;
                float *u = su + (i / (LM_RC / 4)) * (LM_RC + 1) + (i % (LM_RC / 4)) * 4;
                u[0] = ua[t].x; u[1] = ua[t].y; u[2] = ua[t].z; u[3] = ua[t].w;
                *(float4 *)(sd + (i / (LM_T / 4)) * (LM_T + 32) + (i % (LM_T / 4)) * 4) = da[t];
            }
        } else {
            for (int i = threadIdx.x; i < LM_T * LM_RC; i += 256) {
                const int row = i / LM_RC, r = i % LM_RC;
                su[row * (LM_RC + 1) + r] =
                    (r < rc && n0 + row < N) ? up[(size_t)(n0 + row) * R + r0 + r] : 0.f;
            }
            for (int i = threadIdx.x; i < LM_RC * LM_T; i += 256) {
                const int r = i / LM_T, c = i % LM_T;
                sd[r * (LM_T + 32) + c] = (r < rc && k0 + c < K) ? down[(size_t)(r0 + r) * K + k0 + c] : 0.f;
            }
        }
        __syncthreads();
        auto step = [&](int r) {
            const float a = su[(wave * 32 + l32) * (LM_RC + 1) + r + lh];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float b = sd[(r + lh) * (LM_T + 32) + j * 32 + l32];
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[j], 0, 0, 0);
            }
        };
        if (rc == LM_RC) {
            // unrolled: the operand reads of later steps issue ahead of the
            // MFMAs instead of one LDS round trip per step
#pragma unroll
            for (int r = 0; r < LM_RC; r += 2) step(r);
        } else {
            for (int r = 0; r < rc; r += 2) step(r);
        }
        __syncthreads();
    }
    // delta tile to LDS, row-major (acc[j][e]: row (e/4)*8 + lh*4 + e%4 of the
    // wave's 32, column j*32 + l32); row stride 136 floats keeps the two
    // half-waves' rows (4 apart) in opposite bank halves
    float *st = lds;
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int e = 0; e < 16; e++)
            st[(wave * 32 + (e >> 2) * 8 + lh * 4 + (e & 3)) * (LM_T + 8) + j * 32 + l32] = acc[j][e];
    __syncthreads();
    if (full) {
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int c = threadIdx.x + t * 256, row = c / 16, col = (c % 16) * 8;
            const float4 d0 = *(const float4 *)(st + row * (LM_T + 8) + col);
            const float4 d1 = *(const float4 *)(st + row * (LM_T + 8) + col + 4);
            const float dv[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
            u32x4_t o;
#pragma unroll
            for (int e = 0; e < 4; e++)
                o[e] = pack_bf2(fmaf(scale, dv[2 * e], lo_bf(wch[t][e])),
                                fmaf(scale, dv[2 * e + 1], hi_bf(wch[t][e])));
            *(u32x4_t *)(w + (size_t)(n0 + row) * K + k0 + col) = o;
        }
    } else {
        for (int c = threadIdx.x; c < LM_T * LM_T; c += 256) {
            const int row = c / LM_T, col = c % LM_T, n = n0 + row, k = k0 + col;
            if (n < N && k < K) {
                const size_t o = (size_t)n * K + k;
                w[o] = f2bf(fmaf(scale, st[row * (LM_T + 8) + col], bf2f(w[o])));
            }
        }
    }
}

// Split-operand variant on the bf16 matrix cores. Each fp32 operand x is
// held as three bf16 parts x = x0 + x1 + x2 (x0 = bf16(x), x1 =
// bf16(x - x0), x2 = bf16(x - x0 - x1); both differences are exact in fp32),
// and the rank product keeps the six part products down to 2^-16 of the
// leading one: a0b0 + a0b1 + a1b0 + a0b2 + a1b1 + a2b0 (summed smallest
// first). What is dropped is below 2^-24 of |ab|, fp32's own rounding level,
// so the delta matches an fp32 SGEMM up to summation order. Six
// v_mfma_f32_32x32x16_bf16 per 16 ranks replace eight v_mfma_f32_32x32x2_f32,
// about 2.7x less matrix-core time: the merge becomes bound by the
// read-modify-write of W in HBM. Ranks are staged 32 at a time: the six part
// planes of the up slice and of the transposed down slice are staged in LDS.
__device__ __forceinline__ void split3(float x, uint16_t &h0, uint16_t &h1, uint16_t &h2) {
    h0 = f2bf(x);
    const float r1 = x - bf2f(h0);
    h1 = f2bf(r1);
    h2 = f2bf(r1 - bf2f(h1));
}

// Streaming merge for R <= 64 (R % 4 == 0, K % 8 == 0). Persistent blocks of 8
// waves, one per CU, walk contiguous runs of 256 x 64 tiles of W, so the launch
// is one stream of W reads and writes, which bounds it:
//  * wave w owns rows 32 w .. 32 w + 31 of a tile, MFMA A = down^T (rows:
//    columns k of W), B = up (columns: rows of W). The A rows take k in an order
//    that leaves a lane with 8 consecutive columns of one row: W goes from
//    memory to registers and back in 16-byte pieces, two tiles ahead, with no
//    pass through LDS, and a load covers 64 bytes of each of 16 rows (with
//    32 x 32 products it would be 32 bytes of 32 rows: 219 us instead of 198);
//  * the up rows of a wave are split into their three bf16 parts in registers,
//    once per row strip; only the down slice, which all waves share, is staged
//    in LDS: its part planes are written for the next tile while the current
//    tile's MFMAs run, into the other of two buffers;
//  * waves 4 .. 7 run half a tile behind waves 0 .. 3, so that on each SIMD one
//    wave updates and stores while the other multiplies (in step: 217 us).
// One layer's seven targets at R = 64, 386 MB of W read and written: 241 us ->
// 197 us per call, 177 us in the kernel = 4.4 TB/s (a copy here reaches 4.8).
// Before, 128 x 64 tiles with W, up and down all staged in LDS took one launch
// per shape, and five LDS passes over W. Without the MFMAs it would take 178 us.
// Every load and store is unconditional: offsets past the data read as zero
// or are dropped.
#define LT_N 256
#define LT_K 64
#define LT_LD 72   // plane row stride (bf16): 144-byte rows, conflict-free 16-byte reads
__device__ __forceinline__ __amdgpu_buffer_rsrc_t lt_rsrc(const void *base, uint32_t nbytes) {
    const uint64_t b = (uint64_t)base;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    return __builtin_amdgcn_make_buffer_rsrc((void *)(((uint64_t)hi << 32) | lo), 0,
                                             __builtin_amdgcn_readfirstlane(nbytes), 0x00020000);
}
// One launch merges up to LM_TG targets of any shapes, handed over by value:
// their tiles form one index space (target-major, then row strip, then column
// tile) that the blocks split evenly; first[g] is the first tile of target g.
#define LM_TG 32
struct LmTarget {
    uint16_t *w;
    const float *up;
    const float *down;
    float scale;
    int N, K, R, ntk, nstrip;
};
struct LmBatch {
    int n, total;
    int first[LM_TG];
    LmTarget t[LM_TG];
};
__global__ __launch_bounds__(512, 1) void lora_merge_stream_kernel(const LmBatch bt) {
    __shared__ __attribute__((aligned(16))) uint16_t dpl[2][3][LT_K * LT_LD];
#if defined(__HIP_DEVICE_COMPILE__)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lg = lane >> 4;
    const int tb = (int)((int64_t)blockIdx.x * bt.total / gridDim.x);
    const int te = (int)((int64_t)(blockIdx.x + 1) * bt.total / gridDim.x);
    if (tb >= te) return;
    const uint32_t OOB = 0x80000000u;
    struct TC {
        int g, tn, tk;   // target, row strip, column tile
        bool ok;         // the tile exists (t < te)
        LmTarget d;      // the target (wave-uniform)
    };
    auto tc_next = [&](TC c, int t_next) {
        c.tk++;
        if (c.tk == c.d.ntk) {
            c.tk = 0;
            c.tn++;
            if (c.tn == c.d.nstrip) {
                c.tn = 0;
                c.g++;
                c.d = bt.t[c.g < bt.n ? c.g : 0];   // past the last target: any valid entry
            }
        }
        c.ok = t_next < te;
        return c;
    };
    // piece p of four: row (p / 2) * 16 + l16, columns (p % 2) * 32 + lg * 8 .. +7
    auto w_off = [&](const TC &c, int p) -> uint32_t {
        const int gn = c.tn * LT_N + wave * 32 + (p / 2) * 16 + l16, gk = c.tk * LT_K + (p % 2) * 32 + lg * 8;
        return c.ok && gn < c.d.N && gk < c.d.K ? ((uint32_t)gn * (uint32_t)c.d.K + (uint32_t)gk) * 2u : OOB;
    };
    auto load_w = [&](const TC &c, u32x4_t (&w)[4]) {
        const __amdgpu_buffer_rsrc_t rw = lt_rsrc(c.d.w, (uint32_t)((size_t)c.d.N * c.d.K * 2));
#pragma unroll
        for (int p = 0; p < 4; p++)
            w[p] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, w_off(c, p), 0, 0));
    };
    // down slice of a tile: ranks rr, rr + 1, columns kc .. kc + 3
    const int kc = (tid % 16) * 4, rr = (tid / 16) * 2;
    auto load_down = [&](const TC &c, f32x4_t (&d)[2]) {
        const __amdgpu_buffer_rsrc_t rd = lt_rsrc(c.d.down, (uint32_t)((size_t)c.d.R * c.d.K * 4));
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int r = rr + j, gk = c.tk * LT_K + kc;
            const uint32_t o = c.ok && r < c.d.R && gk < c.d.K ? ((uint32_t)r * (uint32_t)c.d.K + (uint32_t)gk) * 4u : OOB;
            d[j] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rd, o, 0, 0));
        }
    };
    // down registers -> part planes of buffer b: column k = 32 kp + 8 g + 4 h + e
    // in plane row 32 kp + 16 h + 4 g + e
    const int krow = (kc & 32) | ((kc & 4) << 2) | ((kc & 24) >> 1);
    auto put_down = [&](const f32x4_t (&d)[2], int b) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            uint16_t h0[3], h1[3];
            split3(d[0][e], h0[0], h0[1], h0[2]);
            split3(d[1][e], h1[0], h1[1], h1[2]);
#pragma unroll
            for (int pl = 0; pl < 3; pl++)
                *(uint32_t *)(dpl[b][pl] + (krow + e) * LT_LD + rr) = (uint32_t)h0[pl] | ((uint32_t)h1[pl] << 16);
        }
    };
    // this lane's up rows in three parts: B operands, row nb*16 + l16, ranks
    // ks*32 + lg*8 .. +7
    bf16x8_t fb[2][2][3];
    auto load_up = [&](const TC &c) {
        const __amdgpu_buffer_rsrc_t ru = lt_rsrc(c.d.up, (uint32_t)((size_t)c.d.N * c.d.R * 4));
        f32x4_t u[4][2];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int gn = c.tn * LT_N + wave * 32 + (i / 2) * 16 + l16, r = (i % 2) * 32 + lg * 8 + j * 4;
                const uint32_t o = gn < c.d.N && r < c.d.R ? ((uint32_t)gn * (uint32_t)c.d.R + (uint32_t)r) * 4u : OOB;
                u[i][j] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(ru, o, 0, 0));
            }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            u32x4_t v[3];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                uint16_t h0[3], h1[3];
                split3(u[i][e >> 1][(e & 1) * 2], h0[0], h0[1], h0[2]);
                split3(u[i][e >> 1][(e & 1) * 2 + 1], h1[0], h1[1], h1[2]);
#pragma unroll
                for (int pl = 0; pl < 3; pl++) v[pl][e] = (uint32_t)h0[pl] | ((uint32_t)h1[pl] << 16);
            }
#pragma unroll
            for (int pl = 0; pl < 3; pl++) fb[i / 2][i % 2][pl] = __builtin_bit_cast(bf16x8_t, v[pl]);
        }
    };
    TC c0;                                // tile t
    int tfirst = 0;
    c0.g = 0;
#pragma unroll
    for (int g = 1; g < LM_TG; g++)
        if (g < bt.n && bt.first[g] <= tb) {
            c0.g = g;
            tfirst = bt.first[g];
        }
    c0.d = bt.t[c0.g];
    c0.tn = (tb - tfirst) / c0.d.ntk;
    c0.tk = (tb - tfirst) % c0.d.ntk;
    c0.ok = true;
    TC c1 = tc_next(c0, tb + 1);          // tile t + 1
    u32x4_t WA[4], WB[4];
    f32x4_t DA[2], DB[2];
    load_down(c0, DA);
    load_w(c0, WA);
    load_down(c1, DB);
    load_w(c1, WB);
    int up_g = c0.g, up_tn = c0.tn;       // the strip whose up rows are in registers
    load_up(c0);
    put_down(DA, tb & 1);
    // tile t splits down(t+1) (dsplit) for the next tile and loads down(t+2)
    // into the registers down(t) used (dload), and W(t+2) into those of W(t);
    // the loop runs two tiles per trip with the register sets swapped, so no
    // register holding a load in flight is ever copied
    auto step = [&](int t, u32x4_t (&w)[4], const f32x4_t (&dsplit)[2], f32x4_t (&dload)[2]) {
        // the planes of tile t are written; every wave is past the previous
        // tile's MFMAs (the other plane buffer is free)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (c0.g != up_g || c0.tn != up_tn) {
            load_up(c0);
            up_g = c0.g;
            up_tn = c0.tn;
        }
        const TC c2 = tc_next(c1, t + 2);
        load_down(c2, dload);
        const int b = t & 1;
        f32x4_t acc[4][2];   // [piece of W][half of its 8 columns]
#pragma unroll
        for (int kb = 0; kb < 4; kb++) {   // 32 (kb / 2) + 4 (kb % 2): the columns' kp and h
            // three accumulators by part-product order (2^-16: a2b0 a1b1 a0b2;
            // 2^-8: a1b0 a0b1; leading: a0b0), summed smallest first at the end
            f32x4_t as[2], am[2], al[2];
#pragma unroll
            for (int nb = 0; nb < 2; nb++) as[nb] = am[nb] = al[nb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            bf16x8_t fa[2][3];
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int p = 0; p < 3; p++)
                    fa[ks][p] = *(const bf16x8_t *)(dpl[b][p] + (kb * 16 + l16) * LT_LD + ks * 32 + lg * 8);
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const bf16x8_t *a = fa[ks];
#pragma unroll
                for (int i = 0; i < 6; i++)
#pragma unroll
                    for (int nb = 0; nb < 2; nb++) {
                        const bf16x8_t *bb = fb[nb][ks];
                        if (i == 0) as[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2], bb[0], as[nb], 0, 0, 0);
                        if (i == 1) am[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], bb[0], am[nb], 0, 0, 0);
                        if (i == 2) al[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], bb[0], al[nb], 0, 0, 0);
                        if (i == 3) as[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], bb[1], as[nb], 0, 0, 0);
                        if (i == 4) am[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], bb[1], am[nb], 0, 0, 0);
                        if (i == 5) as[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], bb[2], as[nb], 0, 0, 0);
                    }
            }
            // the next tile's down slice into the other plane buffer, under the MFMAs
            if (kb == 0) put_down(dsplit, b ^ 1);
#pragma unroll
            for (int nb = 0; nb < 2; nb++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[nb * 2 + kb / 2][kb % 2][e] = al[nb][e] + (am[nb][e] + as[nb][e]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const __amdgpu_buffer_rsrc_t rw = lt_rsrc(c0.d.w, (uint32_t)((size_t)c0.d.N * c0.d.K * 2));
#pragma unroll
        for (int p = 0; p < 4; p++) {
            u32x4_t o;
#pragma unroll
            for (int e = 0; e < 4; e++)
                o[e] = pack_bf2(fmaf(c0.d.scale, acc[p][e / 2][(e % 2) * 2], lo_bf(w[p][e])),
                                fmaf(c0.d.scale, acc[p][e / 2][(e % 2) * 2 + 1], hi_bf(w[p][e])));
            __builtin_amdgcn_raw_buffer_store_b128(o, rw, w_off(c0, p), 0, 0);
        }
        load_w(c2, w);
        c0 = c1;
        c1 = c2;
    };
    // waves 4..7 run half a tile behind: one group's loads, updates and stores
    // run beside the other group's MFMAs
    if (wave >= 4) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int t = tb; t < te; t += 2) {
        step(t, WA, DB, DA);
        if (t + 1 < te) step(t + 1, WB, DA, DB);
    }
    if (wave < 4) asm volatile("s_barrier" ::: "memory");
#endif
}

extern "C" hd_status hd_lora_merge_gpu(hd_lora_entry *entries, size_t count, void *stream) {
    if (count == 0) return HD_OK;
    if (!entries) {
        hd_set_error("lora: null entries");
        return HD_ERR_MISSING;
    }
    hipStream_t st = stream ? (hipStream_t)stream : hd_stream();
    // every entry is checked before the GPU is touched
    for (size_t i = 0; i < count; i++) {
        hd_lora_entry *e = &entries[i];
        if (!e->base_dev || !e->up_dev || !e->down_dev || e->rank == 0 || e->in_dim == 0 ||
            e->out_dim == 0) {
            hd_set_error("lora: entry %zu has a null pointer or zero dim", i);
            return HD_ERR_MISSING;
        }
        if (e->rank > 256) {
            hd_set_error("lora: entry %zu rank %u > 256", i, e->rank);
            return HD_ERR_UNSUPPORTED;
        }
    }
    // Batches. An entry's level is one past the highest level of the earlier
    // entries whose weights overlap its own (two adapters on one target merge
    // in entry order, as the reference's loop does); levels launch in order.
    // Within a level, the entries the streaming kernel takes (R <= 64, R % 4
    // == 0, K % 8 == 0, all operands under 2 GiB) go into one launch per LM_TG
    // of them; the others run the fp32 matrix-core kernel, one launch each.
    struct Range {
        uintptr_t lo, hi;
        bool operator<(const Range &o) const { return lo < o.lo; }
    };
    std::vector<Range> range(count);
    for (size_t i = 0; i < count; i++) {
        range[i].lo = (uintptr_t)entries[i].base_dev;
        range[i].hi = range[i].lo + (size_t)entries[i].out_dim * entries[i].in_dim * 2;
    }
    std::vector<Range> sorted = range;
    std::sort(sorted.begin(), sorted.end());
    bool overlap = false;   // sorted by start: two ranges overlap only if two neighbours do
    for (size_t i = 1; i < count; i++) overlap = overlap || sorted[i].lo < sorted[i - 1].hi;
    std::vector<int> levels(count, 0);
    std::map<int, std::vector<LmTarget>> stream_batches;   // by level
    std::vector<std::pair<int, size_t>> mfma_entries;      // (level, entry)
    int nlevels = 0;
    for (size_t i = 0; i < count; i++) {
        hd_lora_entry *e = &entries[i];
        int level = 0;
        for (size_t j = 0; overlap && j < i; j++)
            if (range[j].lo < range[i].hi && range[i].lo < range[j].hi && level <= levels[j]) level = levels[j] + 1;
        levels[i] = level;
        nlevels = level + 1 > nlevels ? level + 1 : nlevels;
        const int N = (int)e->out_dim, K = (int)e->in_dim, R = (int)e->rank;
        const float scale = e->multiplier * e->alpha / (float)e->rank;   // lora_merge.cu:54
        const bool stream_ok = R <= 64 && R % 4 == 0 && K % 8 == 0 &&
                               (size_t)N * K * 2 < ((size_t)1 << 31) && (size_t)N * R * 4 < ((size_t)1 << 31) &&
                               (size_t)K * R * 4 < ((size_t)1 << 31);
        if (stream_ok)
            stream_batches[level].push_back(LmTarget{(uint16_t *)e->base_dev, (const float *)e->up_dev,
                                                     (const float *)e->down_dev, scale, N, K, R,
                                                     (int)hd_cdiv(K, LT_K), (int)hd_cdiv(N, LT_N)});
        else
            mfma_entries.push_back({level, i});
    }
    int cus = 0, dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    hd_status status = HD_OK;
    for (int level = 0; level < nlevels && status == HD_OK; level++) {
        const std::vector<LmTarget> tg = stream_batches.count(level) ? stream_batches[level] : std::vector<LmTarget>();
        for (size_t i0 = 0; i0 < tg.size(); i0 += LM_TG) {
            // tiles of a target: N K < 2^30, and N, K < 2^27 (up and down under 2 GiB
            // at R >= 4), so ceil(N / 256) ceil(K / 64) < 2^16 + 2^19 + 2^21 + 1;
            // LM_TG of them stay under 2^27
            LmBatch bt;
            bt.n = (int)(tg.size() - i0 < LM_TG ? tg.size() - i0 : LM_TG);
            bt.total = 0;
            for (int g = 0; g < bt.n; g++) {
                bt.t[g] = tg[i0 + g];
                bt.first[g] = bt.total;
                bt.total += bt.t[g].ntk * bt.t[g].nstrip;
            }
            for (int g = bt.n; g < LM_TG; g++) {   // never read as targets
                bt.t[g] = bt.t[0];
                bt.first[g] = bt.total;
            }
            lora_merge_stream_kernel<<<(unsigned)(bt.total < cus ? bt.total : cus), 512, 0, st>>>(bt);
        }
        for (auto &m : mfma_entries) {
            if (m.first != level || status != HD_OK) continue;
            hd_lora_entry *e = &entries[m.second];
            const int N = (int)e->out_dim, K = (int)e->in_dim, R = (int)e->rank;
            const float scale = e->multiplier * e->alpha / (float)e->rank;
            dim3 grid(hd_cdiv(K, LM_T), hd_cdiv(N, LM_T));
            lora_merge_mfma_kernel<2><<<grid, 256, 0, st>>>((uint16_t *)e->base_dev, (const float *)e->up_dev,
                                                            (const float *)e->down_dev, N, K, R, scale);
        }
        hipError_t err = hipGetLastError();
        if (status == HD_OK && err != hipSuccess) {
            hd_set_error("lora: merge launch failed: %s", hipGetErrorString(err));
            status = HD_ERR_RUNTIME;
        }
    }
    if (!stream_batches.empty()) (void)hipStreamSynchronize(st);
    return status;
}

// Flash attention for gfx950 (head_dim 128, GQA, fp32 online softmax) and
// the hd_sdpa_* plan API that replaces the reference's cuDNN-frontend SDPA
// (src/cuda/hd_cudnn_sdpa.cu), plus the small eager attention used for
// validation (attn.cu:22-173 semantics).
//
// Kernel layout (one wave = 32 query rows of one head, 4 waves per block):
//  * S^T = K . Q^T with v_mfma_f32_32x32x16_bf16: the MFMA output puts one
//    query per lane (lane % 32) and 16 key positions per lane, so the row
//    max / row sum need a single xor-32 exchange;
//  * O^T = V^T . P^T: the output accumulator also keeps one query per lane,
//    so the online-softmax rescale is a per-lane scalar;
//  * P^T feeds the second MFMA straight from the S^T registers. The key
//    order inside each 16-key group that this implies (lane half h holds keys
//    h*4..h*4+3 and 8+h*4..8+h*4+3) is matched by storing V^T with bits 2
//    and 3 of the key index swapped ("vt" layout below), so every operand
//    fetch is one 16-byte LDS read;
//  * K and V^T tiles go global -> LDS with buffer_load_dwordx4 ... lds into two
//    buffers (64 keys per tile), XOR-swizzled by row.
// The 8-wave blocks run flash_pp16_kernel: the same online softmax on
// v_mfma_f32_16x16x32_bf16 tiles, split into alternating MFMA and softmax
// phases with the two waves of each SIMD one phase apart (four LDS tile
// buffers, loads two tiles ahead).
//
// vt layout: [B, Hkv, 128, S_pad] bf16, S_pad = round_up(S, 64), key s
// stored at column perm16(s) = s with bits 2 and 3 exchanged, padding zero.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <math.h>

#include "hd_common.hpp"
#include "flash_rows.hpp"
#include "../../include/hd_hip.h"
#include "../../include/hd_sdpa.h"

#define FA_D 128
#define FA_BQ 128      // queries per block (4 waves x 32)
#define FA_BK 64       // keys per tile
#define FA_TAU 8.0f    // lazy-rescale threshold (log2 units)
#define FA_MAX_SPLIT 16 // most key chunks of a tail unit
#define FA_PP_MIN 1024 // shortest sequence that the 8-wave blocks take
#define FA_PP_MIN_DENSE 256   // with a dense mask
#ifndef FA_PF
#define FA_PF 8        // LDS fragment reads in flight ahead of the MFMAs (ping-pong kernel)
#endif

__host__ __device__ __forceinline__ int perm16(int s) {
    return (s & ~12) | ((s & 4) << 1) | ((s & 8) >> 1);
}
static inline int64_t fa_spad(int64_t s) { return (s + FA_BK - 1) / FA_BK * FA_BK; }

// Two bits per 32-row x 64-key tile of a dense mask: "mixed" 0 where every
// value is zero (adding it changes nothing) or every value is "dead": so low
// that mask / scale + score is -inf for any finite score. Two arrays [ceil(S/32)]
// [ceil(S/2048)], mixed then dead, bit t % 32 of word t / 32 for key tile t. The
// mask is the same for every head, so one pass over it here saves the heads'
// blocks reading the tiles that need no values (a mask is usually causal text
// rows, dead right of the diagonal, above zero rows). One wave per (strip, 8
// key tiles: one byte); a lane reads 8 consecutive keys of 4 rows per tile, all
// 32 loads in flight. Reads past S are moved back into the row: a tile may
// then count as mixed that is not, never the reverse. S >= 8.
__global__ __launch_bounds__(64) void fa_mask_bits_kernel(const uint16_t *mask, uint8_t *mixed, uint8_t *dead,
                                                          int S, float inv_scale) {
    const int lane = threadIdx.x;
    u32x4_t v[8][4];
#pragma unroll
    for (int k = 0; k < 8; k++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int kv = min((int)(blockIdx.x * 8 + k) * 64 + (lane & 7) * 8, S - 8);
            const int row = min((int)blockIdx.y * 32 + i * 8 + (lane >> 3), S - 1);
            __builtin_memcpy(&v[k][i], mask + (size_t)row * S + kv, 16);   // an odd S: any even address
        }
    uint32_t m = 0, d = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        uint32_t any = 0;
        bool low = true;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                any |= v[k][i][e];
                // a quarter of the product still overflows: finite scores cannot bring it back
                low = low && lo_bf(v[k][i][e]) * (0.25f * inv_scale) < -3.4028235e38f &&
                      hi_bf(v[k][i][e]) * (0.25f * inv_scale) < -3.4028235e38f;
            }
        const bool all_low = __builtin_amdgcn_ballot_w64(!low) == 0;
        if (all_low) d |= 1u << k;
        else if (__builtin_amdgcn_ballot_w64((any & 0x7fff7fffu) != 0)) m |= 1u << k;
    }
    if (lane == 0) {
        const size_t at = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
        mixed[at] = (uint8_t)m;
        dead[at] = (uint8_t)d;
    }
}

struct FaArgs {
    const uint16_t *q;     // [B,Hq,S,D]
    const uint16_t *k;     // [B,Hkv,S,D]
    const uint16_t *vt;    // [B,Hkv,D,S_pad] (perm16 columns)
    const uint16_t *mask;  // optional [S,S] additive bf16
    uint16_t *out;         // seq-major [B,S,Hq*D] or head-major [B,Hq,S,D]
    int S, S_pad, Hq, Hkv;
    int ar_len;            // rows < ar_len: causal
    int q_row_begin;       // first query row of the launch (its q tiles start here)
    int q_row_end;         // only rows < q_row_end are computed/written
    float scale_log2;      // scale * log2(e)
    float inv_scale;       // 1 / scale (mask values are added to raw scores)
    int out_seq_major;
    int out_rows;          // rows per sequence in `out` (S, or fewer for a staging buffer)
    // tail split: blocks [0, n_whole) each run one (b, head, q tile) unit over
    // all keys; the units from n_whole on run as `split` chunks of the key
    // tiles each (n_chunks blocks), writing unnormalised partials to `part`
    // (merged afterwards). flash_pp16_kernel<FA_CAUSAL>: the blocks after the
    // chunks are the units of the causal rows [0, ar_len), the units before
    // them cover rows [q_row_begin, q_row_end), which see every key
    int n_whole, split, n_chunks;
    float *part;           // [n_chunks][FA_BQ][FA_D] O, then [..][FA_BQ] (m, l)
    // from here on not read by the plain kernels: a further cache line of
    // arguments costs a block ~0.5 us at its start
    int batch;
    FaRows full, causal;   // flash_pp16_kernel: row tiling of the two kinds of units
    const uint32_t *mask_bits;   // FA_DENSE, may be null: see fa_mask_bits_kernel
};

// 16-byte buffer load straight to LDS against a wave-uniform descriptor
// (base, nbytes); the descriptor type exists in the device pass only
__device__ __forceinline__ void fa_buf_load16(const void *base, int nbytes, uint32_t voff, uint32_t soff,
                                              HD_LDS void *dst) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint64_t b = (uint64_t)base;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(((uint64_t)hi << 32) | lo), 0, __builtin_amdgcn_readfirstlane(nbytes), 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, voff, soff, 0, 0);
#endif
}

__device__ __forceinline__ void fa_wait_vm0() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// max / sum with the lane 32 positions away (v_permlane32_swap exchanges
// the two 32-lane halves; max/sum of the pair is the same in both lanes)
__device__ __forceinline__ float xor32_max(float v) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor32_sum(float v) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Blocks are dispatched to the 8 XCDs round-robin (block b to XCD b % 8):
// give each XCD a contiguous range of linear ids instead, so the blocks one
// XCD runs at a time share their kv heads' K / V^T in that XCD's L2.
__device__ __forceinline__ int fa_xcd_remap(int b, int nb) {
    const int per = nb / 8, rem = nb % 8;
    const int xcd = b % 8, idx = b / 8;
    return xcd * per + (xcd < rem ? xcd : rem) + idx;
}

// NWV waves per block (4: two blocks per CU; 8: one block of 256 queries
// per CU sharing one copy of the K / V^T tiles); 32 queries per wave either way.
template <bool MASKED, int NWV>
__global__ __launch_bounds__(NWV * 64, 8 / NWV) void flash_fwd_kernel(FaArgs a) {
    constexpr int BQ = NWV * 32, LPW = 16 / NWV;   // queries per block, loads per wave per tile
    __shared__ __attribute__((aligned(1024))) uint16_t smem[2 * (FA_BK * FA_D + FA_D * FA_BK)];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, h = lane >> 5;

    // block -> (b, head, q tile). Query heads sharing one kv head get
    // consecutive linear ids so they run close together in time.
    const int nqt = (a.q_row_end - a.q_row_begin + BQ - 1) / BQ;
    const int group = a.Hq / a.Hkv;
    int lin = blockIdx.x, chunk = -1, item = 0;
    if (lin >= a.n_whole) {
        item = lin - a.n_whole;
        chunk = item % a.split;
        lin = a.n_whole + item / a.split;
    } else {
        lin = fa_xcd_remap(lin, a.n_whole);
    }
    const int g = lin % group; lin /= group;
    const int qt = lin % nqt; lin /= nqt;
    const int hk = lin % a.Hkv;
    const int b = lin / a.Hkv;
    const int hq = hk * group + g;

    const int qb = a.q_row_begin + qt * BQ;          // the block's first query row
    const int q0 = qb + wave * 32;
    const int my_q = q0 + l32;                       // this lane's query row
    const bool causal_block = qb < a.ar_len;
    // keys needed by this block
    int kv_end = a.S;
    if (causal_block) {
        int last_row = min(qb + BQ, a.q_row_end) - 1;
        if (last_row < a.ar_len) kv_end = last_row + 1;
    }
    int t_begin = 0, t_end = (kv_end + FA_BK - 1) / FA_BK;
    if (chunk >= 0) {
        const int nt = t_end;
        t_begin = chunk * nt / a.split;
        t_end = (chunk + 1) * nt / a.split;
    }

    // ---- Q fragments (B operand of S^T), held for the whole loop ---------
    const uint16_t *qrow = a.q + (((size_t)b * a.Hq + hq) * a.S + min(my_q, a.S - 1)) * FA_D;
    bf16x8_t qf[8];
#pragma unroll
    for (int ks = 0; ks < 8; ks++) qf[ks] = *(const bf16x8_t *)(qrow + ks * 16 + h * 8);

    // ---- loader addressing ------------------------------------------------
    const uint16_t *kbase = a.k + ((size_t)b * a.Hkv + hk) * (size_t)a.S * FA_D;
    const uint16_t *vbase = a.vt + ((size_t)b * a.Hkv + hk) * (size_t)FA_D * a.S_pad;
    // K tile: 64 rows x 16 chunks; wave instr i covers rows 4*(wave*4+i) ..+4
    // V^T tile: 128 rows x 8 chunks; wave instr i covers rows 8*(wave*4+i) ..+8
    // LDS slots are XOR-swizzled so the 16 rows one ds_read_b128 phase
    // touches land in 16 distinct 16-byte bank groups: chunk ^ (row & 15)
    // for the 256-byte K rows, chunk ^ ((row >> 1) & 7) for the 128-byte V^T
    // rows (two rows per 64-bank line)
    uint16_t *Ks0 = smem, *Vs0 = smem + 2 * FA_BK * FA_D;
    // buffer loads straight to LDS: per-lane byte offsets fixed for the
    // block, the tile advance goes in the scalar offset; K rows past S read
    // as zero (their scores are masked: S % 64 != 0 selects the masked
    // kernel), V^T columns are zero-padded to S_pad
    const int kbytes = a.S * FA_D * 2, vbytes = FA_D * a.S_pad * 2;
    uint32_t k_vo[LPW], v_vo[LPW];
#pragma unroll
    for (int i = 0; i < LPW; i++) {
        const int krow = (wave * LPW + i) * 4 + (lane >> 4);
        k_vo[i] = (uint32_t)(krow * FA_D + (((lane & 15) ^ (krow & 15)) * 8)) * 2;
        const int vrow = (wave * LPW + i) * 8 + (lane >> 3);
        v_vo[i] = (uint32_t)(vrow * a.S_pad + (((lane & 7) ^ ((vrow >> 1) & 7)) * 8)) * 2;
    }
    auto issue = [&](int t, int buf) {
        uint16_t *Ks = Ks0 + buf * FA_BK * FA_D, *Vs = Vs0 + buf * FA_D * FA_BK;
#pragma unroll
        for (int i = 0; i < LPW; i++)
            fa_buf_load16(kbase, kbytes, k_vo[i], (uint32_t)t * FA_BK * FA_D * 2,
                          (HD_LDS void *)(Ks + (wave * LPW + i) * 512));
#pragma unroll
        for (int i = 0; i < LPW; i++)
            fa_buf_load16(vbase, vbytes, v_vo[i], (uint32_t)t * FA_BK * 2,
                          (HD_LDS void *)(Vs + (wave * LPW + i) * 512));
    };

    f32x16_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[i][r] = 0.f;
    float m_run = -1e30f, l_run = 0.f;

    issue(t_begin, t_begin & 1);
    fa_wait_vm0();
    __syncthreads();
    for (int t = t_begin; t < t_end; t++) {
        const int buf = t & 1;
        if (t + 1 < t_end) issue(t + 1, buf ^ 1);
        const uint16_t *Ks = Ks0 + buf * FA_BK * FA_D, *Vs = Vs0 + buf * FA_D * FA_BK;

        // S^T for 64 keys: two 32-key tiles
        f32x16_t s[2];
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) s[j][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int row = j * 32 + l32;
                const int c = ((ks * 2 + h) ^ (row & 15)) * 8;
                bf16x8_t kf = *(const bf16x8_t *)(Ks + row * FA_D + c);
                s[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], s[j], 0, 0, 0);
            }
        }

        // tile max on raw scores (the positive scale commutes with max)
        const int kv0 = t * FA_BK;
        // masking is decided per tile and wave: keys past S, causal rows
        // whose diagonal falls in the tile, or a dense mask
        const bool need_mask = MASKED && (a.mask != nullptr || kv0 + FA_BK > a.S ||
                                          (q0 < a.ar_len && kv0 + FA_BK - 1 > q0));
        float mt = -INFINITY;
        // the wave-uniform test is taken once per tile, so tiles without
        // masked keys run exactly the unmasked kernel's max loop
        if (need_mask) {
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    float v = s[j][r];
                    const int kv = kv0 + j * 32 + (r >> 2) * 8 + h * 4 + (r & 3);
                    bool dead = kv >= a.S || (my_q < a.ar_len && kv > my_q);
                    if (a.mask && !dead && my_q < a.S)
                        v += bf2f(a.mask[(size_t)my_q * a.S + kv]) * a.inv_scale;
                    if (dead) v = -INFINITY;
                    s[j][r] = v;
                    mt = fmaxf(mt, v);
                }
        } else {
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) mt = fmaxf(mt, s[j][r]);
        }
        mt = xor32_max(mt);
        // Lazy rescale: the running max only moves when some row's tile max
        // exceeds it by more than 2^FA_TAU in probability terms, so the O
        // rescale is rare after the first tiles; p stays <= 2^FA_TAU.
        if (__builtin_amdgcn_ballot_w64((mt - m_run) * a.scale_log2 > FA_TAU)) {
            const float m_new = fmaxf(m_run, mt);
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * a.scale_log2);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[i][r] *= alpha;
        }
        const float mc = -m_run * a.scale_log2;
        bf16x8_t pf[4];
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int hh = 0; hh < 2; hh++) {
                bf16x8_t pv;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    float p = __builtin_amdgcn_exp2f(fmaf(s[j][hh * 8 + e], a.scale_log2, mc));
                    l_run += p;
                    pv[e] = (__bf16)p;
                }
                pf[j * 2 + hh] = pv;
            }
        // O^T += V^T . P^T over 4 steps of 16 keys
#pragma unroll
        for (int st = 0; st < 4; st++) {
#pragma unroll
            for (int dt = 0; dt < 4; dt++) {
                const int row = dt * 32 + l32;
                const int c = ((st * 2 + h) ^ ((row >> 1) & 7)) * 8;
                bf16x8_t vf = *(const bf16x8_t *)(Vs + row * FA_BK + c);
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[st], o[dt], 0, 0, 0);
            }
        }
        fa_wait_vm0();
        __syncthreads();
    }

    // ---- normalise and store ----------------------------------------------
    const float l_tot = xor32_sum(l_run);
    if (chunk >= 0) {
        // partial: O relative to this chunk's running max, with (m, l)
        float *po = a.part + ((size_t)item * BQ + wave * 32 + l32) * FA_D;
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int gq = 0; gq < 4; gq++) {
                const int d = dt * 32 + gq * 8 + h * 4;
                *(f32x4_t *)(po + d) = {o[dt][gq * 4], o[dt][gq * 4 + 1], o[dt][gq * 4 + 2],
                                        o[dt][gq * 4 + 3]};
            }
        if (h == 0) {
            float2 *pml = (float2 *)(a.part + (size_t)a.n_chunks * BQ * FA_D);
            pml[(size_t)item * BQ + wave * 32 + l32] = make_float2(m_run, l_tot);
        }
        return;
    }
    const float inv = 1.0f / l_tot;
    if (my_q >= a.q_row_end) return;
    uint16_t *dst;
    if (a.out_seq_major)
        dst = a.out + (((size_t)b * a.out_rows + my_q) * a.Hq + hq) * FA_D;
    else
        dst = a.out + (((size_t)b * a.Hq + hq) * a.out_rows + my_q) * FA_D;
    // Lanes l and l + 32 hold the low and high 4 columns of each 8-column
    // chunk of row l. For each pair of chunks (g0, g1) one swap across the
    // half-waves gives lane l all of chunk g0 and lane l + 32 all of g1, so
    // each lane writes 16-byte chunks (8 stores of 16 bytes, not 16 of 8).
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
        for (int gp = 0; gp < 2; gp++) {
            const int g0 = 2 * gp, g1 = g0 + 1;
            const u32x2_t p0 = {pack_bf2(o[dt][g0 * 4] * inv, o[dt][g0 * 4 + 1] * inv),
                                pack_bf2(o[dt][g0 * 4 + 2] * inv, o[dt][g0 * 4 + 3] * inv)};
            const u32x2_t p1 = {pack_bf2(o[dt][g1 * 4] * inv, o[dt][g1 * 4 + 1] * inv),
                                pack_bf2(o[dt][g1 * 4 + 2] * inv, o[dt][g1 * 4 + 3] * inv)};
            // the half this lane gives away: chunk g1's low half (lane l) or
            // chunk g0's high half (lane l + 32)
            const uint32_t z0 = h ? p0[0] : p1[0], z1 = h ? p0[1] : p1[1];
            const auto s0 = __builtin_amdgcn_permlane32_swap(z0, z0, false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(z1, z1, false, false);
            const uint32_t r0 = h ? s0[0] : s0[1], r1 = h ? s1[0] : s1[1];
            const u32x4_t v = h ? (u32x4_t){r0, r1, p1[0], p1[1]} : (u32x4_t){p0[0], p0[1], r0, r1};
            *(u32x4_t *)(dst + dt * 32 + (h ? g1 : g0) * 8) = v;
        }
}

// Ping-pong form of the 8-wave kernel. Each wave alternates an MFMA phase
// (O += P(t-1) V(t-1) and S(t) = K(t) Q^T) with a softmax phase
// (max, lazy rescale, exp2, P(t): VALU only). Waves w and w + 4 share a SIMD;
// waves 4..7 run one phase behind waves 0..3, so on every SIMD one wave's
// softmax issues while the other wave's MFMAs run. A block barrier closes
// every phase. K / V^T tiles go through four LDS buffers, loaded two tiles
// ahead: the buffer tile t + 2 goes to was last read in phase M(t-1), which
// both wave groups have finished when the first group starts M(t).
// (the scheduling fences keep register-only work, e.g. the exp2 of a softmax
// phase, from being moved across the barrier into the neighbouring phase)
__device__ __forceinline__ void fa_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// The ping-pong kernel (the automatic 8-wave choice) on 16x16x32 tiles: the
// phases, barriers, LDS buffers and loads above; each wave's 32 queries are
// two 16-query blocks, and every product runs on
// v_mfma_f32_16x16x32_bf16 (under the power limit the matrix cores sustain
// more FLOP/s with it on random operands than with 32x32x16):
//  * S^T = K Q^T: 4 MFMAs of 16 keys per tile and query block, each summing
//    4 steps of 32 head dimensions. The K rows feeding output row i of
//    MFMA u are key(u, i) = (u/2)*32 + (i/8)*16 + (u%2)*8 + ((i/4)%2)*4 + i%4,
//    so a lane (query lane % 16, row group lane / 16) ends with exactly the
//    8 keys that the V^T layout stores, for each 32-key step, in its 8 P^T
//    operand slots (perm16 columns g*8 .. g*8+7); P feeds the second MFMA
//    straight from the S registers, as in the 32x32 kernels;
//  * O^T = V^T P^T: 8 MFMAs of 16 head dimensions per query block, the V^T
//    rows of MFMA pair (w, v) ordered so that a lane holds 8 consecutive
//    dimensions w*32 + g*8 .. +7 (one 16-byte output store);
//  * a query's 64 scores of a tile sit in the 4 lanes lane % 16 + 16 r: the
//    row max / sum take an xor-16 and an xor-32 lane exchange;
//  * K rows are swizzled by key bits 0-2 and 4, V^T rows by dimension bits
//    1, 3 and 4, so every 16-lane fragment read hits 16 distinct banks.
__device__ __forceinline__ int fa16_kswz(int row) { return (row & 7) | (((row >> 4) & 1) << 3); }
__device__ __forceinline__ int fa16_vswz(int row) { return ((row >> 1) & 1) | (((row >> 3) & 3) << 1); }
__device__ __forceinline__ int fa16_key(int u, int i) {
    return (u >> 1) * 32 + (i >> 3) * 16 + (u & 1) * 8 + ((i >> 2) & 1) * 4 + (i & 3);
}
// max / sum over the 4 lanes lane % 16 + 16 r (v_permlane16_swap exchanges
// rows 0 <-> 1 and 2 <-> 3 of 16 lanes, v_permlane32_swap the two halves)
__device__ __forceinline__ float xor16_32_max(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return xor32_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
__device__ __forceinline__ float xor16_32_sum(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return xor32_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

// MODE FA_PLAIN: S % 64 == 0, every row sees every key, tiles of every head by
// themselves (the row bookkeeping of the other modes costs it 1-7 %, more than
// sharing left-over rows gives). FA_CAUSAL: any S, and
// the units past the chunks are causal rows. FA_DENSE: any S, an additive mask
// (and the causal test per element when ar_len > 0 comes with it).
enum { FA_PLAIN = 0, FA_CAUSAL = 1, FA_DENSE = 2 };
template <int MODE>
__global__ __launch_bounds__(512, 1) void flash_pp16_kernel(FaArgs a) {
    constexpr int PF16 = FA_PF;   // 4 and 12 measured equal or slower
    constexpr int BQ = 256, LPW = 2, NB = 4;
    __shared__ __attribute__((aligned(1024))) uint16_t smem[NB * (FA_BK * FA_D + FA_D * FA_BK)];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave >> 2;
    const int l16 = lane & 15, g = lane >> 4;

    // every kernel argument is in its register from here on: one wait for
    // all of them, and no scalar load that may still be in flight in the loop,
    // which would make the compiler drain all LDS reads (lgkmcnt(0)) at the
    // first fragment of every tile (1.5 % of the kernel)
    asm volatile("" ::"s"(a.part), "s"(a.out), "s"(a.n_chunks), "s"(a.q_row_end), "s"(a.out_rows),
                 "s"(a.out_seq_major), "s"(a.Hq), "s"(a.Hkv), "s"(a.scale_log2), "s"(a.q), "s"(a.k), "s"(a.vt), "s"(a.S),
                 "s"(a.S_pad), "s"(a.n_whole), "s"(a.split), "s"(a.q_row_begin));
    if constexpr (MODE != FA_PLAIN) asm volatile("" ::"s"(a.ar_len), "s"(a.inv_scale), "s"(a.mask));
    int lin = blockIdx.x, chunk = -1, item = 0;
    bool causal_unit = false;
    if (MODE == FA_CAUSAL && lin >= a.n_whole + a.n_chunks) {
        lin -= a.n_whole + a.n_chunks;
        causal_unit = true;
    } else if (lin >= a.n_whole) {
        // neighbouring units of one chunk on an XCD: they share its K / V^T in
        // L2 (2371 tokens, all units split: 103.7 -> 100.2 us; others equal)
        const int c = fa_xcd_remap(lin - a.n_whole, a.n_chunks), n_tail = a.n_chunks / a.split;
        chunk = c / n_tail;
        const int t = c - chunk * n_tail;
        item = t * a.split + chunk;
        lin = a.n_whole + t;
    } else {
        lin = fa_xcd_remap(lin, a.n_whole);
    }
    int b, hk, qbase, q0, kv_end = a.S;
    int my_q[2], my_h[2];   // this lane's two query rows and their heads
    if constexpr (MODE == FA_PLAIN) {
        const int nqt = (a.q_row_end - a.q_row_begin + BQ - 1) / BQ, group = a.Hq / a.Hkv;
        const int gq = lin % group; lin /= group;
        const int qt = lin % nqt; lin /= nqt;
        hk = lin % a.Hkv;
        b = lin / a.Hkv;
        qbase = a.q_row_begin + qt * BQ;
        q0 = qbase + wave * 32;
        my_q[0] = q0 + l16;
        my_q[1] = q0 + 16 + l16;
        my_h[0] = my_h[1] = hk * group + gq;
    } else {
        // (by value: a selected pointer into the arguments would be read with
        // vector loads and make everything below per-lane)
        FaRows rows = a.full;
        const int group = a.Hq / a.Hkv;
        if (MODE == FA_CAUSAL && causal_unit) {
            rows = a.causal;
            lin = fa_longest_first(rows, a.batch, a.Hkv, group, lin);
        }
        FaUnit un = fa_unit(rows, a.batch, a.Hkv, group, lin);
        un.b = __builtin_amdgcn_readfirstlane(un.b);
        un.hk = __builtin_amdgcn_readfirstlane(un.hk);
        un.qbase = __builtin_amdgcn_readfirstlane(un.qbase);
        un.g0 = __builtin_amdgcn_readfirstlane(un.g0);
        un.left = __builtin_amdgcn_readfirstlane(un.left);
        un.hp = __builtin_amdgcn_readfirstlane(un.hp);
        b = un.b;
        hk = un.hk;
        qbase = un.qbase;
        q0 = qbase + (un.left ? 0 : wave * 32);   // lowest row of this wave
#pragma unroll
        for (int qq = 0; qq < 2; qq++) {
            const FaRowHead rh = fa_unit_row(un, group, wave * 32 + qq * 16 + l16);
            my_q[qq] = rh.row;
            my_h[qq] = rh.head;
        }
        if (qbase < a.ar_len) {
            const int last_row = qbase + (un.left ? un.left : BQ) - 1;
            if (last_row < a.ar_len) kv_end = last_row + 1;
        }
    }
    int t_begin = 0, t_end = (kv_end + FA_BK - 1) / FA_BK;
    if (chunk >= 0) {
        const int nt = t_end;
        t_begin = chunk * nt / a.split;
        t_end = (chunk + 1) * nt / a.split;
    }

    // Q^T operand: query block qq, head dimensions ks*32 + g*8 .. +7
    bf16x8_t qf[2][4];
#pragma unroll
    for (int qq = 0; qq < 2; qq++) {
        const uint16_t *qrow = a.q + (((size_t)b * a.Hq + my_h[qq]) * a.S + min(my_q[qq], a.S - 1)) * FA_D;
#pragma unroll
        for (int ks = 0; ks < 4; ks++) qf[qq][ks] = *(const bf16x8_t *)(qrow + ks * 32 + g * 8);
    }

    const uint16_t *kbase = a.k + ((size_t)b * a.Hkv + hk) * (size_t)a.S * FA_D;
    const uint16_t *vbase = a.vt + ((size_t)b * a.Hkv + hk) * (size_t)FA_D * a.S_pad;
    uint16_t *Ks0 = smem, *Vs0 = smem + NB * FA_BK * FA_D;
    const int kbytes = a.S * FA_D * 2, vbytes = FA_D * a.S_pad * 2;
    uint32_t k_vo[LPW], v_vo[LPW];
#pragma unroll
    for (int i = 0; i < LPW; i++) {
        const int krow = (wave * LPW + i) * 4 + (lane >> 4);
        k_vo[i] = (uint32_t)(krow * FA_D + (((lane & 15) ^ fa16_kswz(krow)) * 8)) * 2;
        const int vrow = (wave * LPW + i) * 8 + (lane >> 3);
        v_vo[i] = (uint32_t)(vrow * a.S_pad + (((lane & 7) ^ fa16_vswz(vrow)) * 8)) * 2;
    }
    auto issue = [&](int t) {
        const int buf = t & (NB - 1);
        uint16_t *Ks = Ks0 + buf * FA_BK * FA_D, *Vs = Vs0 + buf * FA_D * FA_BK;
#pragma unroll
        for (int i = 0; i < LPW; i++)
            fa_buf_load16(kbase, kbytes, k_vo[i], (uint32_t)t * FA_BK * FA_D * 2,
                          (HD_LDS void *)(Ks + (wave * LPW + i) * 512));
#pragma unroll
        for (int i = 0; i < LPW; i++)
            fa_buf_load16(vbase, vbytes, v_vo[i], (uint32_t)t * FA_BK * 2,
                          (HD_LDS void *)(Vs + (wave * LPW + i) * 512));
    };

    // this lane's fragment rows: K row of S-MFMA u, V^T row of O-MFMA (w, v)
    int krow_u[4];
#pragma unroll
    for (int u = 0; u < 4; u++) krow_u[u] = fa16_key(u, l16);
    const int vrow0 = (l16 >> 2) * 8 + (l16 & 3);   // + w*32 + v*4

    f32x4_t o[2][8];
#pragma unroll
    for (int qq = 0; qq < 2; qq++)
#pragma unroll
        for (int i = 0; i < 8; i++) o[qq][i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    float m_run[2] = {-1e30f, -1e30f}, l_run[2] = {0.f, 0.f};
    f32x4_t s[2][4];
    bf16x8_t pf[2][2];

    auto kfrag = [&](const uint16_t *Ks, int u, int ks) {
        const int row = krow_u[u];
        const int c = ((ks * 4 + g) ^ fa16_kswz(row)) * 8;
        return *(const bf16x8_t *)(Ks + row * FA_D + c);
    };
    auto vfrag = [&](const uint16_t *Vs, int w, int v, int st) {
        const int row = w * 32 + v * 4 + vrow0;
        const int c = ((st * 4 + g) ^ fa16_vswz(row)) * 8;
        return *(const bf16x8_t *)(Vs + row * FA_BK + c);
    };
    // S(t) = K(t) Q^T
    auto qk = [&](int t) {
        const uint16_t *Ks = Ks0 + (t & (NB - 1)) * FA_BK * FA_D;
#pragma unroll
        for (int qq = 0; qq < 2; qq++)
#pragma unroll
            for (int u = 0; u < 4; u++) s[qq][u] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const bf16x8_t kf = kfrag(Ks, u, ks);
#pragma unroll
                for (int qq = 0; qq < 2; qq++)
                    s[qq][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[qq][ks], s[qq][u], 0, 0, 0);
            }
    };
    // O += V^T(t) P(t)^T
    auto pv = [&](int t) {
        const uint16_t *Vs = Vs0 + (t & (NB - 1)) * FA_D * FA_BK;
#pragma unroll
        for (int st = 0; st < 2; st++)
#pragma unroll
            for (int x = 0; x < 8; x++) {
                const bf16x8_t vf = vfrag(Vs, x >> 1, x & 1, st);
#pragma unroll
                for (int qq = 0; qq < 2; qq++)
                    o[qq][x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[qq][st], o[qq][x], 0, 0, 0);
            }
    };
    // both products of one MFMA phase, interleaved (independent chains)
    auto pv_qk = [&](int t) {
        const uint16_t *Vs = Vs0 + ((t - 1) & (NB - 1)) * FA_D * FA_BK;
        const uint16_t *Ks = Ks0 + (t & (NB - 1)) * FA_BK * FA_D;
#pragma unroll
        for (int qq = 0; qq < 2; qq++)
#pragma unroll
            for (int u = 0; u < 4; u++) s[qq][u] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int y = 0; y < 16; y++) {
            const int st = y >> 3, x = y & 7;
            const bf16x8_t vf = vfrag(Vs, x >> 1, x & 1, st);
#pragma unroll
            for (int qq = 0; qq < 2; qq++)
                o[qq][x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[qq][st], o[qq][x], 0, 0, 0);
            const int ks = y >> 2, u = y & 3;
            const bf16x8_t kf = kfrag(Ks, u, ks);
#pragma unroll
            for (int qq = 0; qq < 2; qq++)
                s[qq][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[qq][ks], s[qq][u], 0, 0, 0);
        }
        // fragment reads run PF16 reads ahead of the MFMAs (two MFMAs per read)
        __builtin_amdgcn_sched_group_barrier(0x100, PF16, 0);
#pragma unroll
        for (int i = 0; i < 32 - PF16; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * PF16, 0);
    };
    // dense mask of tile t in the order of the scores: lanes of row groups 2r
    // and 2r + 1 need keys {0-3, 8-11} and {4-7, 12-15} of a 16-key run, so
    // each loads 8 consecutive keys and one 16-lane row swap exchanges the
    // inner halves. Requested at the start of tile t's MFMA phase, before the
    // K / V^T loads of a later tile, so the values land under the MFMAs and
    // the phase's vmcnt wait covers them. Rows start at any even address (S
    // may be odd): unaligned 16-byte loads; the tile that holds key S - 1
    // reads element by element, clamped to the row.
    // Tiles that fa_mask_bits_kernel found to be all zero or all dead are not
    // read: bit t of this wave's 32-row strip, 32 tiles per lane.
    u32x4_t mk[2][2];
    uint32_t mbits = ~0u, dbits = 0u;
    if constexpr (MODE == FA_DENSE) {
        const int strip = (qbase >> 5) + wave, strips = (a.S + 31) / 32, nw = (a.S + FA_BK * 32 - 1) / (FA_BK * 32);
        if (a.mask_bits) {
            mbits = 0u;
            if (lane < nw && strip < strips) {
                mbits = a.mask_bits[(size_t)strip * nw + lane];
                dbits = a.mask_bits[(size_t)(strips + strip) * nw + lane];
            }
        }
    }
    auto is_dead = [&](int t) {
        return MODE == FA_DENSE && (__builtin_amdgcn_readlane(dbits, t >> 5) >> (t & 31) & 1);
    };
    auto has_mask = [&](int t) {
        return MODE == FA_DENSE && (__builtin_amdgcn_readlane(mbits, t >> 5) >> (t & 31) & 1);
    };
    auto load_mask = [&](int t) {
        if (has_mask(t)) {
            const int kv0 = t * FA_BK + (g >> 1) * 16 + (g & 1) * 8;
#pragma unroll
            for (int qq = 0; qq < 2; qq++) {
                const uint16_t *row = a.mask + (size_t)min(my_q[qq], a.S - 1) * a.S;
#pragma unroll
                for (int w = 0; w < 2; w++) {
                    const int k0 = kv0 + w * 32;
                    if ((t + 1) * FA_BK <= a.S) {
                        __builtin_memcpy(&mk[qq][w], row + k0, 16);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            mk[qq][w][e] = (uint32_t)row[min(k0 + 2 * e, a.S - 1)] |
                                           ((uint32_t)row[min(k0 + 2 * e + 1, a.S - 1)] << 16);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto swap_mask = [&]() {
        if constexpr (MODE == FA_DENSE) {
#pragma unroll
            for (int qq = 0; qq < 2; qq++)
#pragma unroll
                for (int w = 0; w < 2; w++)
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const auto r = __builtin_amdgcn_permlane16_swap(mk[qq][w][e], mk[qq][w][e + 2], false, false);
                        mk[qq][w][e] = r[0];
                        mk[qq][w][e + 2] = r[1];
                    }
        }
    };
    // softmax of S(t) into P(t), with the lazy O rescale
    auto softmax = [&](int t) {
        const int kv0 = t * FA_BK;
        // the wave-uniform test is taken once per tile: tiles without dead
        // keys run exactly the plain kernel's max loop
        const bool dead_keys = MODE != FA_PLAIN &&
                               (kv0 + FA_BK > a.S || (q0 < a.ar_len && kv0 + FA_BK - 1 > q0));
        if (has_mask(t)) swap_mask();
#pragma unroll
        for (int qq = 0; qq < 2; qq++) {
            float mt = -INFINITY;
            if (has_mask(t)) {
                asm volatile("");
#pragma unroll
                for (int u = 0; u < 4; u++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint32_t m2 = mk[qq][u >> 1][(u & 1) * 2 + (e >> 1)];
                        s[qq][u][e] = fmaf(e & 1 ? hi_bf(m2) : lo_bf(m2), a.inv_scale, s[qq][u][e]);
                    }
            }
            if (is_dead(t)) {
                asm volatile("");
#pragma unroll
                for (int u = 0; u < 4; u++)
#pragma unroll
                    for (int e = 0; e < 4; e++) s[qq][u][e] -= INFINITY;
            }
            if (dead_keys) {
                // a branch, not 32 selects in every tile, and its key
                // indexes are formed inside it
                int kvb = kv0;
                asm volatile("" : "+s"(kvb));
                const int mq = my_q[qq];
#pragma unroll
                for (int u = 0; u < 4; u++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int kv = kvb + fa16_key(u, g * 4 + e);
                        const bool dead = kv >= a.S || (mq < a.ar_len && kv > mq);
                        const float v = dead ? -INFINITY : s[qq][u][e];
                        s[qq][u][e] = v;
                        mt = fmaxf(mt, v);
                    }
            } else {
#pragma unroll
                for (int u = 0; u < 4; u++)
#pragma unroll
                    for (int e = 0; e < 4; e++) mt = fmaxf(mt, s[qq][u][e]);
            }
            mt = xor16_32_max(mt);
            if (__builtin_amdgcn_ballot_w64((mt - m_run[qq]) * a.scale_log2 > FA_TAU)) {
                const float m_new = fmaxf(m_run[qq], mt);
                const float alpha = __builtin_amdgcn_exp2f((m_run[qq] - m_new) * a.scale_log2);
                m_run[qq] = m_new;
                l_run[qq] *= alpha;
#pragma unroll
                for (int i = 0; i < 8; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) o[qq][i][e] *= alpha;
            }
            const float mc = -m_run[qq] * a.scale_log2;
#pragma unroll
            for (int st = 0; st < 2; st++) {
                bf16x8_t p8;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float p = __builtin_amdgcn_exp2f(fmaf(s[qq][st * 2 + (e >> 2)][e & 3], a.scale_log2, mc));
                    l_run[qq] += p;
                    p8[e] = (__bf16)p;
                }
                pf[qq][st] = p8;
            }
        }
    };
    auto pin_softmax = [&]() {
        asm volatile("" ::"v"(pf[0][0]), "v"(pf[0][1]), "v"(pf[1][0]), "v"(pf[1][1]), "v"(l_run[0]),
                     "v"(l_run[1]));
    };
    auto wait_next = [&](bool issued) {
        if (issued) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        else fa_wait_vm0();
    };
    // the barrier sequence of the phases above (2T + 3 barriers per wave)
    issue(t_begin);
    if (t_begin + 1 < t_end) {
        issue(t_begin + 1);
        wait_next(true);
    } else {
        fa_wait_vm0();
    }
    fa_barrier();
    if (grp) fa_barrier();
    {
        const bool ld = t_begin + 2 < t_end;
        load_mask(t_begin);
        if (ld) issue(t_begin + 2);
        qk(t_begin);
        wait_next(ld);
        fa_barrier();
    }
    // The loop's speed depends on where it starts in the 32-byte instruction
    // fetch windows: 12 or 16 bytes past one is 1-2 % faster than most other
    // places (all 16 places of a word tried: 12 and 16 at 3490 us for 16640 keys,
    // the rest 3520-3580; at 28, where it stood by chance, 3624 against 3588 in
    // turn, 4352 keys x 2 520.2 against 515.6, 1152 keys 32.0 against 31.4). The
    // code from here to the loop's first instruction ends 20 bytes past such a
    // window, so 6 words more put it at 12 (a test reads it from the built code).
    if constexpr (MODE == FA_PLAIN) asm volatile(".p2align 5\n\t.rept 6\n\ts_nop 0\n\t.endr");
    for (int t = t_begin + 1; t < t_end; t++) {
        softmax(t - 1);
        pin_softmax();
        fa_barrier();
        const bool ld = t + 2 < t_end;
        load_mask(t);
        if (ld) issue(t + 2);
        pv_qk(t);
        wait_next(ld);
        fa_barrier();
    }
    softmax(t_end - 1);
    pin_softmax();
    fa_barrier();
    pv(t_end - 1);
    fa_barrier();

    // ---- normalise and store: a lane holds dimensions w*32 + g*8 .. +7 -----
#pragma unroll
    for (int qq = 0; qq < 2; qq++) {
        const float l_tot = xor16_32_sum(l_run[qq]);
        const int row = wave * 32 + qq * 16 + l16;
        if (chunk >= 0) {
            float *po = a.part + ((size_t)item * BQ + row) * FA_D;
#pragma unroll
            for (int w = 0; w < 4; w++) {
                *(f32x4_t *)(po + w * 32 + g * 8) = o[qq][w * 2];
                *(f32x4_t *)(po + w * 32 + g * 8 + 4) = o[qq][w * 2 + 1];
            }
            if (g == 0) {
                float2 *pml = (float2 *)(a.part + (size_t)a.n_chunks * BQ * FA_D);
                pml[(size_t)item * BQ + row] = make_float2(m_run[qq], l_tot);
            }
        } else if (my_q[qq] < a.q_row_end) {
            const float inv = 1.0f / l_tot;
            uint16_t *dst;
            if (a.out_seq_major)
                dst = a.out + (((size_t)b * a.out_rows + my_q[qq]) * a.Hq + my_h[qq]) * FA_D;
            else
                dst = a.out + (((size_t)b * a.Hq + my_h[qq]) * a.out_rows + my_q[qq]) * FA_D;
#pragma unroll
            for (int w = 0; w < 4; w++) {
                const f32x4_t x0 = o[qq][w * 2], x1 = o[qq][w * 2 + 1];
                const u32x4_t v = {pack_bf2(x0[0] * inv, x0[1] * inv), pack_bf2(x0[2] * inv, x0[3] * inv),
                                   pack_bf2(x1[0] * inv, x1[1] * inv), pack_bf2(x1[2] * inv, x1[3] * inv)};
                *(u32x4_t *)(dst + w * 32 + g * 8) = v;
            }
        }
    }
    if (!grp) fa_barrier();
}

// ---------------------------------------------------------------------------
// Full attention at head_dim 72 (the vision tower), operands unpadded: q, k
// [BH, S, 72], vt [BH, 72, S_pad] (perm16 columns, zero past S), out seq-major
// [B, S, heads * 72]. The 4-wave kernel's scheme (32 queries per wave, 32x32x16
// MFMAs, S^T then O^T) with 5 k-steps of 16 for 72 + 8 zero dimensions and 3
// row tiles of 32 for 72 + 24 zero rows: 22 MFMAs per 64 keys, where heads
// padded to 128 take 32, and half their memory. K rows stand 176 bytes apart in
// LDS (11 16-byte chunks, the last two zero: 16 rows of one chunk hit 16 bank
// groups); chunks and rows past 72 are loads past the records, which read zero.
// KS waves share each 32 queries, every KS-th key tile each, and merge at the
// end: the tower's 576 rows are 80 blocks of 128 queries, so with KS = 2 its
// 144 blocks of 64 take half the key tiles each on otherwise idle CUs.
// Bound by latency at 576 rows (9 key tiles): 14.8 us with heads padded to 128,
// and 4.5 more to take the padding out again -> 10.9 us; three images, KS = 1:
// 13.0 us.
// ---------------------------------------------------------------------------
struct FaV72Args {
    const uint16_t *q, *k, *vt;
    uint16_t *out;
    int S, S_pad, heads;
    float scale_log2;
};
template <int KS>
__global__ __launch_bounds__(256, KS == 1 ? 3 : 2) void flash_v72_kernel(FaV72Args a) {
    constexpr int D = 72, KP = 88, VR = 96, BK = 64, QG = 4 / KS, KT = BK * KP, VT = VR * BK;
    constexpr int KI = BK * KP / 8 / 64, VI = VR * BK / 8 / 64;   // load instructions of a tile: 11 and 12
    __shared__ __attribute__((aligned(1024))) uint16_t smem[2 * KS * (KT + VT)];
    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wave / QG, qw = wave % QG;
    const int bh = blockIdx.y, q0 = blockIdx.x * QG * 32 + qw * 32, my_q = q0 + l32;
    const int nt = (a.S + BK - 1) / BK, nit = (nt + KS - 1) / KS;

    const uint16_t *qrow = a.q + ((size_t)bh * a.S + min(my_q, a.S - 1)) * D;
    bf16x8_t qf[5];
#pragma unroll
    for (int ks = 0; ks < 5; ks++) {
        const int d = ks * 16 + h * 8;
        qf[ks] = __builtin_bit_cast(bf16x8_t, (u32x4_t){0, 0, 0, 0});
        if (d < D) qf[ks] = *(const bf16x8_t *)(qrow + d);
    }
    const uint16_t *kbase = a.k + (size_t)bh * a.S * D, *vbase = a.vt + (size_t)bh * D * a.S_pad;
    const int kbytes = a.S * D * 2, vbytes = D * a.S_pad * 2;
    // a tile's loads are spread over the QG waves of its key group
    constexpr int KPW = (KI + QG - 1) / QG, VPW = (VI + QG - 1) / QG;
    uint32_t k_vo[KPW], v_vo[VPW];
#pragma unroll
    for (int i = 0; i < KPW; i++) {
        const int c = (qw * KPW + i) * 64 + lane, row = c / (KP / 8), ch = c % (KP / 8);
        k_vo[i] = ch < D / 8 ? (uint32_t)(row * D + ch * 8) * 2 : 0x80000000u;
    }
#pragma unroll
    for (int i = 0; i < VPW; i++) {
        const int row = (qw * VPW + i) * 8 + (lane >> 3);
        v_vo[i] = row < D ? (uint32_t)(row * a.S_pad + ((lane & 7) ^ ((row >> 1) & 7)) * 8) * 2 : 0x80000000u;
    }
    auto issue = [&](int it, int buf) {
        const int t = it * KS + kg;
        // a key group without a tile in the last round reads zeros; the scalar
        // offset stays inside the records
        const bool live = t < nt;
        uint16_t *Ks = smem + (buf * KS + kg) * (KT + VT), *Vs = Ks + KT;
#pragma unroll
        for (int i = 0; i < KPW; i++)
            if (qw * KPW + i < KI)
                fa_buf_load16(kbase, kbytes, live ? k_vo[i] : 0x80000000u, live ? (uint32_t)t * BK * D * 2 : 0u,
                              (HD_LDS void *)(Ks + (qw * KPW + i) * 512));
#pragma unroll
        for (int i = 0; i < VPW; i++)
            if (qw * VPW + i < VI)
                fa_buf_load16(vbase, vbytes, live ? v_vo[i] : 0x80000000u, live ? (uint32_t)t * BK * 2 : 0u,
                              (HD_LDS void *)(Vs + (qw * VPW + i) * 512));
    };
    f32x16_t o[3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[i][r] = 0.f;
    float m_run = -1e30f, l_run = 0.f;

    issue(0, 0);
    fa_wait_vm0();
    __syncthreads();
    for (int it = 0; it < nit; it++) {
        const int buf = it & 1, t = it * KS + kg, kv0 = t * BK;
        if (it + 1 < nit) issue(it + 1, buf ^ 1);
        if (t < nt) {
            const uint16_t *Ks = smem + (buf * KS + kg) * (KT + VT), *Vs = Ks + KT;
            f32x16_t s[2];
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) s[j][r] = 0.f;
#pragma unroll
            for (int ks = 0; ks < 5; ks++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const bf16x8_t kf = *(const bf16x8_t *)(Ks + (j * 32 + l32) * KP + (ks * 2 + h) * 8);
                    s[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], s[j], 0, 0, 0);
                }
            float mt = -INFINITY;
            if (kv0 + BK > a.S) {
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int kv = kv0 + j * 32 + (r >> 2) * 8 + h * 4 + (r & 3);
                        s[j][r] = kv < a.S ? s[j][r] : -INFINITY;
                        mt = fmaxf(mt, s[j][r]);
                    }
            } else {
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) mt = fmaxf(mt, s[j][r]);
            }
            mt = xor32_max(mt);
            if (__builtin_amdgcn_ballot_w64((mt - m_run) * a.scale_log2 > FA_TAU)) {
                const float m_new = fmaxf(m_run, mt);
                const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * a.scale_log2);
                m_run = m_new;
                l_run *= alpha;
#pragma unroll
                for (int i = 0; i < 3; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) o[i][r] *= alpha;
            }
            const float mc = -m_run * a.scale_log2;
            bf16x8_t pf[4];
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int hh = 0; hh < 2; hh++) {
                    bf16x8_t pv;
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const float p = __builtin_amdgcn_exp2f(fmaf(s[j][hh * 8 + e], a.scale_log2, mc));
                        l_run += p;
                        pv[e] = (__bf16)p;
                    }
                    pf[j * 2 + hh] = pv;
                }
#pragma unroll
            for (int st = 0; st < 4; st++)
#pragma unroll
                for (int dt = 0; dt < 3; dt++) {
                    const int row = dt * 32 + l32;
                    const bf16x8_t vf = *(const bf16x8_t *)(Vs + row * BK + ((st * 2 + h) ^ ((row >> 1) & 7)) * 8);
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[st], o[dt], 0, 0, 0);
                }
        }
        fa_wait_vm0();
        __syncthreads();
    }
    float l_tot = xor32_sum(l_run);
    if constexpr (KS == 2) {
        // key group 1 hands its sums over (the tile buffers are free), group 0
        // merges them relative to the larger of the two running maxima
        float *x = (float *)smem + qw * 50 * 64 + lane;   // [50][64] per 32 queries
        if (kg == 1) {
#pragma unroll
            for (int i = 0; i < 3; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) x[(i * 16 + r) * 64] = o[i][r];
            x[48 * 64] = m_run;
            x[49 * 64] = l_tot;
        }
        __syncthreads();
        if (kg == 1) return;
        const float m1 = x[48 * 64], m = fmaxf(m_run, m1);
        const float w0 = __builtin_amdgcn_exp2f((m_run - m) * a.scale_log2);
        const float w1 = __builtin_amdgcn_exp2f((m1 - m) * a.scale_log2);
        l_tot = l_tot * w0 + x[49 * 64] * w1;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[i][r] = o[i][r] * w0 + x[(i * 16 + r) * 64] * w1;
    }
    if (my_q >= a.S) return;
    const float inv = 1.0f / l_tot;
    // lane (query, h) holds dimensions dt*32 + g*8 + h*4 .. +3: 8-byte stores,
    // two lanes fill 16 bytes; dimensions past 72 are dropped
    uint16_t *dst = a.out + (((size_t)(bh / a.heads) * a.S + my_q) * a.heads + bh % a.heads) * D;
#pragma unroll
    for (int dt = 0; dt < 3; dt++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int d = dt * 32 + g * 8 + h * 4;
            if (dt * 32 + g * 8 < D)
                *(u32x2_t *)(dst + d) = (u32x2_t){pack_bf2(o[dt][g * 4] * inv, o[dt][g * 4 + 1] * inv),
                                                  pack_bf2(o[dt][g * 4 + 2] * inv, o[dt][g * 4 + 3] * inv)};
        }
}

int hd_flash_v72(const void *q, const void *k, const void *vt, void *out, int batch, int heads, int seq,
                 float scale) {
    FaV72Args a = {(const uint16_t *)q, (const uint16_t *)k, (const uint16_t *)vt, (uint16_t *)out, seq,
                   (int)fa_spad(seq), heads, scale * 1.44269504088896341f};
    if (batch * heads * ((seq + 63) / 64) <= 256)
        flash_v72_kernel<2><<<dim3((seq + 63) / 64, batch * heads), 256, 0, hd_stream()>>>(a);
    else
        flash_v72_kernel<1><<<dim3((seq + 127) / 128, batch * heads), 256, 0, hd_stream()>>>(a);
    hd_check_launch("flash_v72");
    return 0;
}

// V [BH, S, D] -> vt [BH, D, S_pad] with perm16 columns and zero padding.
// One block per 64-key tile: rows in through LDS (16-byte loads when V is
// 16-byte aligned), 16-byte stores of 8 storage columns per dimension. HBM
// bound in principle (4 B per element); at S = 2371, 8 heads it is one short
// launch: 8.4 us with 2-byte accesses, 4.0 us in this form, 5.2 in a trace (S = 16640: 26.9 ->
// 11.5 us).
template <bool V16>
__global__ __launch_bounds__(256) void fa_vt_kernel(const uint16_t *v, uint16_t *vt, int S,
                                                    int S_pad) {
    constexpr int LD = FA_D + 8;
    __shared__ __attribute__((aligned(16))) uint16_t tile[64][LD];
    const int bh = blockIdx.y, s0 = blockIdx.x * 64;
    const uint16_t *src = v + (size_t)bh * S * FA_D;
    if constexpr (V16) {
        for (int i = threadIdx.x; i < 64 * FA_D / 8; i += 256) {
            const int t = i / (FA_D / 8), c = (i % (FA_D / 8)) * 8;
            u32x4_t x = {0, 0, 0, 0};
            if (s0 + t < S) x = *(const u32x4_t *)(src + (size_t)(s0 + t) * FA_D + c);
            *(u32x4_t *)&tile[t][c] = x;
        }
    } else {
        for (int i = threadIdx.x; i < 64 * FA_D; i += 256) {
            int t = i / FA_D, d = i % FA_D;
            tile[t][d] = (s0 + t < S) ? src[(size_t)(s0 + t) * FA_D + d] : (uint16_t)0;
        }
    }
    __syncthreads();
    uint16_t *dst = vt + (size_t)bh * FA_D * S_pad + s0;
    for (int i = threadIdx.x; i < FA_D * 8; i += 256) {
        const int d = i / 8, p0 = (i % 8) * 8;   // 8 storage columns p0 .. p0+7 of the tile
        u32x4_t o;
#pragma unroll
        for (int e = 0; e < 4; e++)
            o[e] = (uint32_t)tile[perm16(p0 + 2 * e)][d] | ((uint32_t)tile[perm16(p0 + 2 * e + 1)][d] << 16);
        *(u32x4_t *)(dst + (size_t)d * S_pad + p0) = o;
    }
}
static void fa_vt_launch(const void *v, void *vt, int bh, int S, hipStream_t st) {
    const dim3 g(hd_cdiv(fa_spad(S), 64), bh);
    if ((uintptr_t)v % 16 == 0)
        fa_vt_kernel<true><<<g, 256, 0, st>>>((const uint16_t *)v, (uint16_t *)vt, S, (int)fa_spad(S));
    else
        fa_vt_kernel<false><<<g, 256, 0, st>>>((const uint16_t *)v, (uint16_t *)vt, S, (int)fa_spad(S));
}

// Merges the tail units' key-chunk partials: O = sum_i w_i O_i / sum_i w_i l_i
// with w_i = 2^((m_i - max_j m_j) * scale_log2). One thread per (row, 8
// consecutive d): two 16-byte partial loads per chunk, one 16-byte store.
// SHARED: units of fa_unit's numbering (left-over rows share units).
template <int BQ, bool SHARED>
__global__ __launch_bounds__(256) void fa_merge_kernel(FaArgs a, int n_tail) {
    const int idx = blockIdx.x * 256 + threadIdx.x;
    const int d0 = (idx % (FA_D / 8)) * 8, row = (idx / (FA_D / 8)) % BQ, tu = idx / (FA_D / 8 * BQ);
    if (tu >= n_tail) return;
    const int P = a.split, n_items = n_tail * P;
    const float2 *pml = (const float2 *)(a.part + (size_t)n_items * BQ * FA_D);
    float m = -INFINITY;
    for (int i = 0; i < P; i++) m = fmaxf(m, pml[(size_t)(tu * P + i) * BQ + row].x);
    float L = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < P; i++) {
        const float2 ml = pml[(size_t)(tu * P + i) * BQ + row];
        const float w = __builtin_amdgcn_exp2f((ml.x - m) * a.scale_log2);
        L = fmaf(w, ml.y, L);
        const float4 *src = (const float4 *)(a.part + ((size_t)(tu * P + i) * BQ + row) * FA_D + d0);
        const float4 p0 = src[0], p1 = src[1];
        const float pv[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
#pragma unroll
        for (int e = 0; e < 8; e++) acc[e] = fmaf(w, pv[e], acc[e]);
    }
    int b, hq, my_q;
    if constexpr (SHARED) {
        const int group = a.Hq / a.Hkv;
        const FaUnit un = fa_unit(a.full, a.batch, a.Hkv, group, a.n_whole + tu);
        const FaRowHead rh = fa_unit_row(un, group, row);
        b = un.b;
        hq = rh.head;
        my_q = rh.row;
    } else {
        const int nqt = (a.q_row_end - a.q_row_begin + BQ - 1) / BQ, group = a.Hq / a.Hkv;
        int lin = a.n_whole + tu;
        const int g = lin % group; lin /= group;
        const int qt = lin % nqt; lin /= nqt;
        b = lin / a.Hkv;
        hq = (lin % a.Hkv) * group + g;
        my_q = a.q_row_begin + qt * BQ + row;
    }
    if (my_q >= a.q_row_end) return;
    const size_t o = a.out_seq_major ? (((size_t)b * a.out_rows + my_q) * a.Hq + hq) * FA_D + d0
                                     : (((size_t)b * a.Hq + hq) * a.out_rows + my_q) * FA_D + d0;
    const float inv = 1.0f / L;
    u32x4_t v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = pack_bf2(acc[2 * e] * inv, acc[2 * e + 1] * inv);
    *(u32x4_t *)(a.out + o) = v;
}

// Resident flash blocks on the current device (occupancy x CUs), cached.
static int fa_slots(int nwv = 4) {
    static int dev_cached = -1, slots4 = 0, slots8 = 0;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (dev != dev_cached) {
        int per4 = 0, per8 = 0, cus = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per4, flash_fwd_kernel<false, 4>, 256, 0) !=
                hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per8, flash_pp16_kernel<FA_PLAIN>, 512, 0) !=
                hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        slots4 = per4 * cus;
        slots8 = per8 * cus;
        dev_cached = dev;
    }
    return nwv == 8 ? slots8 : slots4;
}

// Workspace for the tail split: at most one round of partial blocks.
extern "C" int64_t hd_flash_ws_bytes(void) {
    // one round of partial blocks of either family (slots x rows per block)
    const int64_t r4 = (int64_t)fa_slots(4) * 128, r8 = (int64_t)fa_slots(8) * 256;
    const int64_t rows = r4 > r8 ? r4 : r8;
    return (rows > 0 ? rows : 1024 * 128) * (FA_D + 2) * 4;
}

extern "C" int64_t hd_flash_vt_bytes(int batch, int kv_heads, int seq) {
    return (int64_t)batch * kv_heads * FA_D * fa_spad(seq) * 2;
}

// Writes the flash V^T layout from a head-major V (used by the plan API; the
// decoder block's QKV epilogue writes it directly).
extern "C" void hd_flash_make_vt(const void *v, void *vt, int bh, int seq) {
    if (!v || !vt || bh <= 0 || seq <= 0) {
        snprintf(hd_cuda_errbuf(), 512, "flash_make_vt: bad args");
        return;
    }
    fa_vt_launch(v, vt, bh, seq, hd_stream());
    hd_check_launch("flash_make_vt");
}

// Bytes of the tile bits of a dense mask (0: too long for one lane per word).
static int64_t fa_mask_bits_bytes(int seq) {
    const int64_t words = (seq + FA_BK * 32 - 1) / (FA_BK * 32);
    return words <= 64 ? (seq + 31) / 32 * words * 8 : 0;
}

// Key tiles that the causal rows [0, ar_len) of one head read, in blocks of n rows.
static int64_t fa_causal_tiles(int ar_len, int n) {
    const int64_t full = ar_len / n;
    return full * (full + 1) / 2 * (n / FA_BK) + (ar_len % n ? (ar_len + FA_BK - 1) / FA_BK : 0);
}

// Key chunks of the units in the last, partly filled round (rem of them, nt key
// tiles each; 1: no split) beside n_causal causal units of w key tiles in all.
static int fa_split(int rem, int nt, int n_causal, int64_t w, int slots) {
    if (rem == 0) return 1;
    int P = (slots - n_causal) / rem;
    // causal units that need the free slots themselves: chunks short enough to
    // end with them
    if (P < 2) P = n_causal ? (int)hd_cdiv((int64_t)nt * slots, (int64_t)rem * nt + w) : slots / rem;
    if (P > FA_MAX_SPLIT) P = FA_MAX_SPLIT;
    return P < nt ? P : nt;
}

// Ways to run a causal text prefix (rows < ar_len see keys <= row, the others all):
//  FA_ONE    one masked launch of 4-wave blocks. The block that holds row ar_len
//            runs every key, masked ones too unless ar_len % 128 == 0
//  FA_TWO    the prefix rows as FA_ONE, whose blocks all end at their diagonal,
//            then the other rows as full attention (8-wave with a workspace)
//  FA_UNITS  one launch of 8-wave blocks, causal rows as units of their own behind
//            the full ones, longest first; FA_UNITS_WHOLE the same without key
//            chunks
// A call without a workspace takes the kernel for the causal rows that it would
// take with one, so that these rows do not depend on it.
// From FA_PP_MIN keys on the lowest predicted time is taken: us per 64-key tile of a
// full round's and of a lone block, the launches' fixed costs, and the work of all
// blocks over the CUs, fitted to all four at 1650 calls with a workspace (1-3 x 8-32
// heads, S = 1024-8704, ar_len = 1 .. S - 1): the choice is 0.9 % off the fastest on
// average. FA_UNITS in all cases would be 6 % off and up to 1.46 times as long where
// causal rows are many or the grid is less than a round; us, fastest second:
//   32 heads, S = 2371, ar_len 114: ONE 114, UNITS 102; S = 4239, 142: ONE 311, UNITS 269
//   32 heads, S = 1024, ar_len 1023: UNITS 36.4, ONE 25.5; 8 heads, 1101, 256: 34.4, 25.4
//   32 heads, S = 4352, ar_len 256: UNITS 256, TWO 247; 2 x 1152, 142: 50.9, 46.5
enum { FA_ONE, FA_TWO, FA_UNITS, FA_UNITS_WHOLE };
static int fa_prefix_route(int batch, int hq, int hkv, int seq, int ar_len, int q_row_end, bool ws) {
    const int slots = fa_slots(8), nt = (seq + FA_BK - 1) / FA_BK, group = hq / hkv, bh = batch * hq;
    if (slots <= 0) return FA_ONE;
    const double per_cu = 1.0 / slots;
    double best = 1e30;
    int route = FA_ONE;
    auto offer = [&](int r, double us) {
        if (us < best) {
            best = us;
            route = r;
        }
    };
    // 4-wave blocks, two per CU: the longest one, or the work of all and the free
    // slots of the last round (each hides most of the other)
    auto blocks4_us = [&](int64_t blocks, double tiles, double longest) {
        const int64_t last = blocks % (2 * slots);
        double work = 0.96 * tiles * per_cu;
        if (blocks > 2 * slots && last) work += 0.36 * nt * (1.0 - 0.5 * last * per_cu);
        const double lo = fmin(longest, work), hi = fmax(longest, work);
        return 7.4 + hi + 0.3 * lo * lo / hi;
    };
    const int mixed = ar_len % 128 ? nt - ar_len / FA_BK : 0;   // masked tiles of the block with row ar_len
    const int64_t pre = ar_len / 128, per_head = (q_row_end + 127) / 128;
    const double one = blocks4_us(bh * per_head, (double)bh * (pre * (pre + 1) + (per_head - pre) * nt + mixed),
                                  1.02 * nt + 1.06 * mixed);
    offer(FA_ONE, one);
    // 8-wave blocks: whole rounds, then what is left over beside w causal tiles
    auto units_us = [&](int units, int n_causal, int64_t w, double tile, bool split) {
        const int rem = units % slots, P = split && units >= slots ? fa_split(rem, nt, n_causal, w, slots) : 1;
        const double left = tile * ((double)rem * nt + w) * per_cu, us = 9.7 + tile * nt * (units / slots);
        if (P > 1)
            return us + 15.3 + 10.5 * fmax(0.0, (rem * P + n_causal) * per_cu - 1.0) +
                   fmax(1.37 * ((nt + P - 1) / P) + 7.3, left);
        return us + fmax(rem ? 1.37 * nt : 0.0, left) + (units + n_causal > slots ? 7.3 : 0.0);
    };
    const FaRows full = fa_rows_of(ar_len, q_row_end - ar_len, group, true), causal = fa_rows_of(0, ar_len, group, false);
    const int units = fa_rows_units(full, batch, hkv, group), n_causal = fa_rows_units(causal, batch, hkv, group);
    const int64_t w = bh * fa_causal_tiles(ar_len, FA_ROWS);
    offer(FA_UNITS, units_us(units, n_causal, w, 1.80, true));
    offer(FA_UNITS_WHOLE, 1.01 * units_us(units, n_causal, w, 1.80, false));
    const double first = 3.4 + fmax(2.04 * ((ar_len + 127) / 128), 0.85 * bh * fa_causal_tiles(ar_len, 128) * per_cu);
    if (seq % FA_BK == 0)
        offer(FA_TWO, 1.02 * (first + units_us(bh * ((q_row_end - ar_len + FA_ROWS - 1) / FA_ROWS), 0, 0, 1.74, true)));
    if (ws) return route;
    if (route >= FA_UNITS) return FA_UNITS_WHOLE;
    const int64_t rest = bh * ((q_row_end - ar_len + 127) / 128);   // 4-wave blocks here
    return first + blocks4_us(rest, (double)rest * nt, 1.02 * nt) < one ? FA_TWO : FA_ONE;
}

static int fa_launch(const void *q, const void *k, const void *vt, const void *mask, void *out,
                     int batch, int hq, int hkv, int seq, int ar_len, int q_row_end, float scale,
                     int out_seq_major, hipStream_t st, void *ws = nullptr, int64_t ws_bytes = 0,
                     int out_rows = 0, int q_row_begin = 0) {
    const bool with_prefix = ar_len > 0 && !mask && q_row_begin == 0 && ar_len < q_row_end;
    int route = FA_ONE;
    if (with_prefix) {
        if (seq >= FA_PP_MIN) route = fa_prefix_route(batch, hq, hkv, seq, ar_len, q_row_end, ws != nullptr);
        else if (ws && seq % FA_BK == 0) route = FA_TWO;
    }
    if (route == FA_TWO) {
        const int rc = fa_launch(q, k, vt, nullptr, out, batch, hq, hkv, seq, ar_len, ar_len, scale,
                                 out_seq_major, st, nullptr, 0, out_rows, 0);
        if (rc) return rc;
        return fa_launch(q, k, vt, nullptr, out, batch, hq, hkv, seq, 0, q_row_end, scale, out_seq_major, st,
                         ws, ws_bytes, out_rows, ar_len);
    }
    const bool prefix = route >= FA_UNITS;   // causal rows on units of their own
    FaArgs a;
    a.q = (const uint16_t *)q;
    a.k = (const uint16_t *)k;
    a.vt = (const uint16_t *)vt;
    a.mask = (const uint16_t *)mask;
    a.out = (uint16_t *)out;
    a.batch = batch;
    a.S = seq;
    a.S_pad = (int)fa_spad(seq);
    a.Hq = hq;
    a.Hkv = hkv;
    a.ar_len = ar_len;
    a.q_row_begin = q_row_begin;
    a.q_row_end = q_row_end;
    a.scale_log2 = scale * 1.44269504088896341f;
    a.inv_scale = 1.0f / scale;
    a.out_seq_major = out_seq_major;
    a.out_rows = out_rows > 0 ? out_rows : seq;
    // 8-wave blocks (one copy of each K / V^T tile for 256 queries) when the
    // sequence is long enough to amortise the larger block and
    //  * the tail split can fill the last round (+3 % at S = 16640 / 16896,
    //    equal at 4352; without the split the finer grain of 4 waves wins), or
    //  * there is a causal prefix that the route above gives to units of
    //    their own, or
    //  * there is a dense mask: its values are prefetched as 16-byte pieces
    //    under the MFMA phase, where a tile needs them (4-wave blocks
    //    with 2-byte loads, causal text rows above zeros: S = 300 26.6 ->
    //    25.6 us, 1209 199 -> 57, 4239 1937 -> 318; equal
    //    at 200, where one 256-row block per head is as long as two of 128).
    const bool pp = mask ? seq >= FA_PP_MIN_DENSE : seq >= FA_PP_MIN && (prefix || (ws && ar_len == 0));
    const int nwv = pp ? 8 : 4;
    const int BQ = nwv * 32;
    const int group = hq / hkv;
    int units, n_causal = 0;
    const bool plain = !mask && ar_len == 0 && seq % FA_BK == 0;
    a.full = a.causal = {};
    if (pp && !plain) {
        if (prefix) a.q_row_begin = ar_len;   // the causal rows are units of their own
        a.full = fa_rows_of(a.q_row_begin, q_row_end - a.q_row_begin, group, !mask);
        units = fa_rows_units(a.full, batch, hkv, group);
        if (prefix) {
            a.causal = fa_rows_of(0, ar_len, group, false);
            n_causal = fa_rows_units(a.causal, batch, hkv, group);
        }
    } else {
        units = batch * hq * ((q_row_end - a.q_row_begin + BQ - 1) / BQ);
    }
    // Tail split (units that see every key only): the units of the last
    // partial round of resident blocks run as P key chunks each, launched
    // last, so that round is filled (together with the causal units) instead
    // of running a few blocks for a whole round.
    a.n_whole = units;
    a.split = 1;
    a.part = (float *)ws;
    int n_tail = 0;
    // dense mask: the tile bits lie behind the partials in the workspace
    const int64_t bits_bytes = pp && mask && q_row_begin == 0 ? fa_mask_bits_bytes(seq) : 0;
    const bool bits = bits_bytes > 0 && ws && bits_bytes <= ws_bytes;
    if (bits) ws_bytes -= bits_bytes;
    const int slots = ws ? fa_slots(nwv) : 0;
    if (slots > 0 && (ar_len == 0 || route == FA_UNITS) && units >= slots) {
        const int rem = units % slots, ntile = (seq + FA_BK - 1) / FA_BK;
        int P = fa_split(rem, ntile, n_causal, n_causal ? batch * hq * fa_causal_tiles(ar_len, BQ) : 0, slots);
        const int64_t chunk_bytes = (int64_t)BQ * (FA_D + 2) * 4;
        if (bits && rem * P * chunk_bytes > ws_bytes) P = (int)(ws_bytes / (rem * chunk_bytes));
        if (rem && P >= 2 && rem * P * chunk_bytes <= ws_bytes) {
            n_tail = rem;
            a.n_whole = units - rem;
            a.split = P;
        }
    }
    a.n_chunks = n_tail * a.split;
    a.mask_bits = nullptr;
    if (bits) {
        uint8_t *at = (uint8_t *)ws + (int64_t)a.n_chunks * BQ * (FA_D + 2) * 4;
        fa_mask_bits_kernel<<<dim3((seq + FA_BK * 32 - 1) / (FA_BK * 32) * 4, (seq + 31) / 32), 64, 0, st>>>(
            (const uint16_t *)mask, at, at + bits_bytes / 2, seq, a.inv_scale);
        a.mask_bits = (const uint32_t *)at;
    }
    dim3 grid((unsigned)(a.n_whole + a.n_chunks + n_causal));
    if (pp) {
        // the ping-pong form: +2.5-4.7 % at S = 4352-16640 over 8-wave
        // blocks in lockstep
        if (mask) flash_pp16_kernel<FA_DENSE><<<grid, 512, 0, st>>>(a);
        else if (!plain) flash_pp16_kernel<FA_CAUSAL><<<grid, 512, 0, st>>>(a);
        else flash_pp16_kernel<FA_PLAIN><<<grid, 512, 0, st>>>(a);
    } else {
        if (mask || ar_len > 0 || seq % FA_BK) flash_fwd_kernel<true, 4><<<grid, 256, 0, st>>>(a);
        else flash_fwd_kernel<false, 4><<<grid, 256, 0, st>>>(a);
    }
    if (n_tail) {
        dim3 gm((unsigned)hd_cdiv((int64_t)n_tail * BQ * (FA_D / 8), 256));
        if (!pp) fa_merge_kernel<128, false><<<gm, 256, 0, st>>>(a, n_tail);
        else if (plain) fa_merge_kernel<256, false><<<gm, 256, 0, st>>>(a, n_tail);
        else fa_merge_kernel<256, true><<<gm, 256, 0, st>>>(a, n_tail);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        snprintf(hd_cuda_errbuf(), 512, "hd_sdpa: flash launch failed: %s", hipGetErrorString(e));
        return 1;
    }
    return 0;
}

extern "C" int hd_flash_attention(const void *q, const void *k, const void *vt, const void *mask,
                                  void *out, int batch, int q_heads, int kv_heads, int seq,
                                  int head_dim, int ar_len, float scale, int out_seq_major) {
    if (!q || !k || !vt || !out || batch <= 0 || q_heads <= 0 || kv_heads <= 0 ||
        q_heads % kv_heads || seq <= 0 || head_dim != FA_D || ar_len < 0 || ar_len > seq) {
        snprintf(hd_cuda_errbuf(), 512, "hd_sdpa: flash bad args");
        return 1;
    }
    return fa_launch(q, k, vt, mask, out, batch, q_heads, kv_heads, seq, ar_len, seq, scale,
                     out_seq_major, hd_stream());
}

extern "C" int hd_flash_attention_ws(const void *q, const void *k, const void *vt, const void *mask,
                                     void *out, int batch, int q_heads, int kv_heads, int seq,
                                     int head_dim, int ar_len, float scale, int out_seq_major,
                                     void *ws, int64_t ws_bytes) {
    if (!q || !k || !vt || !out || batch <= 0 || q_heads <= 0 || kv_heads <= 0 ||
        q_heads % kv_heads || seq <= 0 || head_dim != FA_D || ar_len < 0 || ar_len > seq) {
        snprintf(hd_cuda_errbuf(), 512, "hd_sdpa: flash bad args");
        return 1;
    }
    return fa_launch(q, k, vt, mask, out, batch, q_heads, kv_heads, seq, ar_len, seq, scale,
                     out_seq_major, hd_stream(), ws, ws_bytes);
}

// ---------------------------------------------------------------------------
// Plan API (hd_cudnn_sdpa.h). A plan is shape + split point + a V^T staging
// buffer allocated once at create time (the reference allocates its cuDNN
// workspace and causal staging there too, hd_cudnn_sdpa.cu:233-247, :354-368).
// ---------------------------------------------------------------------------
struct hd_sdpa_plan {
    int B, Hq, Hkv, Sq, Skv, D;
    int ar_len;
    float scale;
    void *vt;
    size_t vt_bytes;
    void *ws = nullptr;      // tail-split partials (hd_flash_ws_bytes)
    int64_t ws_bytes = 0;
    void *o_stage = nullptr; // split plans: causal-prefix rows of pass 0, [B, ar_len, Hq, D]
};

static int sdpa_err(const char *m) {
    snprintf(hd_cuda_errbuf(), 512, "hd_sdpa: %s", m);
    return 1;
}

static int plan_new(hd_sdpa_plan **out, int batch, int hq, int hkv, int sq, int skv, int d,
                    int ar_len, float scale) {
    if (!out) return sdpa_err("null out");
    *out = nullptr;
    if (batch < 1) return sdpa_err("invalid batch");
    if (hq < 1 || hkv < 1 || hq % hkv) return sdpa_err("invalid head counts (q_heads % kv_heads != 0)");
    if (sq < 1 || skv < 1 || d < 1) return sdpa_err("invalid dims");
    if (d != FA_D) return sdpa_err("head_dim must be 128");
    if (sq != skv) return sdpa_err("seq_q must equal seq_kv");
    hd_sdpa_plan *p = new hd_sdpa_plan();
    p->B = batch; p->Hq = hq; p->Hkv = hkv; p->Sq = sq; p->Skv = skv; p->D = d;
    p->ar_len = ar_len;
    p->scale = scale;
    p->vt_bytes = (size_t)hd_flash_vt_bytes(batch, hkv, skv);
    if (hipMalloc(&p->vt, p->vt_bytes) != hipSuccess) {
        delete p;
        return sdpa_err("hipMalloc V^T staging failed");
    }
    p->ws_bytes = hd_flash_ws_bytes() + fa_mask_bits_bytes(sq);
    if (hipMalloc(&p->ws, (size_t)p->ws_bytes) != hipSuccess) {
        (void)hipFree(p->vt);
        delete p;
        return sdpa_err("hipMalloc flash workspace failed");
    }
    if (ar_len > 0 &&
        hipMalloc(&p->o_stage, (size_t)batch * ar_len * hq * d * 2) != hipSuccess) {
        (void)hipFree(p->vt);
        (void)hipFree(p->ws);
        delete p;
        return sdpa_err("hipMalloc causal-prefix staging failed");
    }
    *out = p;
    return 0;
}

extern "C" int hd_sdpa_create(hd_sdpa_plan **out, int batch, int q_heads, int kv_heads, int seq_q,
                              int seq_kv, int head_dim, float scale) {
    return plan_new(out, batch, q_heads, kv_heads, seq_q, seq_kv, head_dim, 0, scale);
}

extern "C" int hd_sdpa_create_split(hd_sdpa_plan **out, int batch, int q_heads, int kv_heads,
                                    int seq, int ar_len, int head_dim, float scale) {
    if (out) *out = nullptr;
    if (ar_len < 0 || ar_len >= seq) return sdpa_err("invalid ar_len (must be 0 < ar_len < seq)");
    return plan_new(out, batch, q_heads, kv_heads, seq, seq, head_dim, ar_len, scale);
}

extern "C" int hd_sdpa_create_prod(hd_sdpa_plan **out, int batch, int q_heads, int kv_heads,
                                   int seq, int ar_len, int head_dim, float scale) {
    if (!out) return sdpa_err("null out");
    *out = nullptr;
    if (ar_len > 0 && ar_len < seq)
        return hd_sdpa_create_split(out, batch, q_heads, kv_heads, seq, ar_len, head_dim, scale);
    return hd_sdpa_create(out, batch, q_heads, kv_heads, seq, seq, head_dim, scale);
}

extern "C" void hd_sdpa_destroy(hd_sdpa_plan *p) {
    if (!p) return;
    if (p->vt) (void)hipFree(p->vt);
    if (p->ws) (void)hipFree(p->ws);
    if (p->o_stage) (void)hipFree(p->o_stage);
    delete p;
}

static int plan_run(hd_sdpa_plan *p, const void *q, const void *k, const void *v, const void *mask,
                    void *out, void *stream, int ar_len, int q_row_end, bool to_stage = false) {
    hipStream_t st = stream ? (hipStream_t)stream : hd_stream();
    fa_vt_launch(v, p->vt, p->B * p->Hkv, p->Skv, st);
    if (hipGetLastError() != hipSuccess) return sdpa_err("V^T staging launch failed");
    if (to_stage)   // pass 0: the causal rows into the plan's staging, seq-major
        return fa_launch(q, k, p->vt, mask, p->o_stage, p->B, p->Hq, p->Hkv, p->Sq, ar_len, q_row_end,
                         p->scale, 1, st, p->ws, p->ws_bytes, p->ar_len);
    return fa_launch(q, k, p->vt, mask, out, p->B, p->Hq, p->Hkv, p->Sq, ar_len, q_row_end,
                     p->scale, 0, st, p->ws, p->ws_bytes);
}

extern "C" int hd_sdpa_execute(hd_sdpa_plan *p, const void *q, const void *k, const void *v,
                               const void *mask, void *out, void *stream) {
    if (!p || !q || !k || !v || !out) return sdpa_err("null arg in execute");
    if (p->ar_len > 0) return hd_sdpa_execute_split(p, q, k, v, out, stream);
    return plan_run(p, q, k, v, mask, out, stream, 0, p->Sq);
}

extern "C" int hd_sdpa_execute_split(hd_sdpa_plan *p, const void *q, const void *k, const void *v,
                                     void *out, void *stream) {
    if (!p || !q || !k || !v || !out) return sdpa_err("null arg in execute");
    if (p->ar_len <= 0) return sdpa_err("execute_split on a non-split plan");
    return plan_run(p, q, k, v, nullptr, out, stream, p->ar_len, p->Sq);
}

extern "C" const void *hd_sdpa_plan_stage(const hd_sdpa_plan *p) { return p ? p->o_stage : nullptr; }

extern "C" int hd_sdpa_execute_split_pass(hd_sdpa_plan *p, int which, const void *q, const void *k,
                                          const void *v, void *out, void *stream) {
    if (!p || !q || !k || !v || !out) return sdpa_err("null arg in execute");
    if (p->ar_len <= 0) return sdpa_err("execute_split_pass on a non-split plan");
    // pass 0 leaves `out` untouched: its rows go to the plan's staging, as
    // the reference's causal pass writes only its staged head
    // (hd_cudnn_sdpa.cu:455-468)
    if (which == 0) return plan_run(p, q, k, v, nullptr, out, stream, p->ar_len, p->ar_len, true);
    return plan_run(p, q, k, v, nullptr, out, stream, 0, p->Sq);
}

// ---------------------------------------------------------------------------
// Eager attention (attn.cu:22-173 semantics) for small validation shapes:
// fp32 scores, fp32 softmax, bf16 probs, fp32 P.V over bf16 probs,
// seq-major output. Scores are recomputed instead of kept in an fp32
// scratch, so nothing is allocated.
// ---------------------------------------------------------------------------
__global__ void eager_probs_kernel(const uint16_t *q, const uint16_t *k, const uint16_t *mask,
                                   uint16_t *scores, uint16_t *probs, int H, int KV, int S, int D,
                                   float scaling) {
    int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= H * S) return;
    int s = idx % S, hh = idx / S, kh = hh / (H / KV);
    const uint16_t *qr = q + ((size_t)hh * S + s) * D;
    auto score = [&](int t) {
        const uint16_t *kr = k + ((size_t)kh * S + t) * D;
        float acc = 0.f;
        for (int d = 0; d < D; d++) acc += bf2f(qr[d]) * bf2f(kr[d]);
        acc *= scaling;
        return acc + bf2f(mask[(size_t)s * S + t]);
    };
    float mx = -INFINITY;
    for (int t = 0; t < S; t++) mx = fmaxf(mx, score(t));
    float sum = 0.f;
    for (int t = 0; t < S; t++) sum += expf(score(t) - mx);
    float inv = 1.0f / sum;
    for (int t = 0; t < S; t++) {
        float sc = score(t);
        scores[((size_t)hh * S + s) * S + t] = f2bf(sc);
        probs[((size_t)hh * S + s) * S + t] = f2bf(expf(sc - mx) * inv);
    }
}
__global__ void eager_out_kernel(const uint16_t *probs, const uint16_t *v, uint16_t *out, int H,
                                 int KV, int S, int D) {
    size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)H * S * D) return;
    int d = idx % D;
    size_t r = idx / D;
    int hh = r % H, s = r / H, kh = hh / (H / KV);   // idx enumerates [S,H,D]
    const uint16_t *pr = probs + ((size_t)hh * S + s) * S;
    float acc = 0.f;
    for (int t = 0; t < S; t++) acc += bf2f(pr[t]) * bf2f(v[((size_t)kh * S + t) * D + d]);
    out[idx] = f2bf(acc);
}
extern "C" void hd_attention_eager(const void *q, const void *k, const void *v, const void *mask,
                                   void *scores, void *probs, void *out, int heads, int kv_heads,
                                   int seq, int dim, float scaling) {
    if (!q || !k || !v || !mask || !scores || !probs || !out || heads <= 0 || kv_heads <= 0 ||
        seq <= 0 || dim <= 0 || heads % kv_heads) {
        snprintf(hd_cuda_errbuf(), 512, "attention_eager: bad args");
        return;
    }
    eager_probs_kernel<<<hd_cdiv((size_t)heads * seq, 128), 128, 0, hd_stream()>>>(
        (const uint16_t *)q, (const uint16_t *)k, (const uint16_t *)mask, (uint16_t *)scores,
        (uint16_t *)probs, heads, kv_heads, seq, dim, scaling);
    eager_out_kernel<<<hd_cdiv((size_t)heads * seq * dim, 256), 256, 0, hd_stream()>>>(
        (const uint16_t *)probs, (const uint16_t *)v, (uint16_t *)out, heads, kv_heads, seq, dim);
    hd_check_launch("attention_eager");
}

extern "C" int hd_sdpa_plan_ar_len(const hd_sdpa_plan *p) { return p ? p->ar_len : 0; }

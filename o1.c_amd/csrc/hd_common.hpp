// Shared device/host helpers of the MI355X engine (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

// ---- library-wide launch stream and error buffer (support.hip) ----------
extern "C" char *hd_cuda_errbuf(void);
hipStream_t hd_stream(void);
// Records a launch failure (if any) of the previous kernel under `what`.
void hd_check_launch(const char *what);

// hd_linear_qkv_rope_ws for any sequence length (gemm.hip).
int hd_qkv_rope_gemm(const void *x, const void *wq, const void *wk, const void *wv, const void *qn_w,
                     const void *kn_w, const float *cs, void *q, void *k, void *vt, int batch, int seq,
                     int heads, int kv_heads, int hidden, float eps, void *ws, int64_t ws_bytes);

// y = bf16(gelu(bf16(bf16(x . w^T) + bias))), tanh or erf form, rows of ldc (gemm.hip).
void hd_linear_gelu(const void *x, const void *w, const void *bias, void *y, int M, int N, int K, bool erf,
                    void *ws, int64_t ws_bytes, int ldc);
// hd_linear_ws over operand rows of lda and ldb elements (gemm.hip): the K-group kernels where K % 8 == 0 but
// not K % 64, in pieces of rows past 2 GiB of x; the reference kernel otherwise.
void hd_linear_strided(const void *x, int lda, const void *w, int ldb, const void *bias, void *y, int M, int N,
                       int K, void *ws, int64_t ws_bytes);
// Attention of the vision tower: q, k [batch * heads, seq, 72], vt [batch * heads, 72, round_up(seq, 64)]
// in the flash key order, out [batch, seq, heads * 72] (attention.hip).
int hd_flash_v72(const void *q, const void *k, const void *vt, void *out, int batch, int heads, int seq,
                 float scale);

// ---- bf16 <-> fp32 ------------------------------------------------------
// bf16 payloads are uint16_t. fp32 -> bf16 uses gfx950's v_cvt_pk_bf16_f32,
// IEEE round-to-nearest-even: for finite values the same bits as the
// reference's integer rule (support.cu:21-28); NaN payloads are not produced
// on this path.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float bf2f(uint16_t b) {
    return __uint_as_float(((uint32_t)b) << 16);
}
// Two floats -> packed bf16x2 (low half = a), one instruction.
__device__ __forceinline__ uint32_t pack_bf2(float a, float b) {
    bf16x2_t v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float bfround(float f) { return bf2f(f2bf(f)); }
__device__ __forceinline__ float lo_bf(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_bf(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

// ---- GELU, tanh and erf forms (vision_kernels.cu) -----------------------
// 0.5 (1 + tanh(u)) = 1 / (1 + e^-2u): no cancellation where tanh nears -1, and
// the hardware exp and reciprocal (about 1 ulp each) instead of tanhf's ~50
// instructions, which were half of a small fc1 GEMM's time as its epilogue.
__device__ __forceinline__ float gelu_tanh_f(float v) {
    const float u2 = 1.5957691216057308f * (v + 0.044715f * v * v * v);
    return v * __builtin_amdgcn_rcpf(1.0f + __expf(-u2));
}
__device__ __forceinline__ float gelu_erf_f(float v) {
    return 0.5f * v * (1.0f + erff(v * 0.7071067811865476f));
}

// ---- MFMA operand types -------------------------------------------------
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

#define HD_LDS __attribute__((address_space(3)))

static inline unsigned hd_cdiv(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

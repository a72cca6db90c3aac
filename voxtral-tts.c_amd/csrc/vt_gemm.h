/*
 * vt_gemm.h - launchers of the bf16 MFMA matrix product on (hi, lo) activation
 * planes and of the row kernels that produce those planes.
 */
#ifndef VT_GEMM_H
#define VT_GEMM_H

#include <stddef.h>
#include <stdint.h>

#include "vt_gemm_plans.h"

/* N a multiple of 128, K/splits a multiple of 64 */
int vt_gemm_shape_ok(int M, int N, int K, int splits);
/* d_C: `splits` planes of [M, N] fp32, plane s holds the sum over K range s */
void vt_launch_gemm(float *d_C, const uint16_t *d_Ahi, const uint16_t *d_Alo, const uint16_t *d_W,
                    int M, int N, int K, int splits);
/* the same with the row pitch of C and the distance between planes given */
void vt_launch_gemm_ex(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                       const uint16_t *d_W, int M, int N, int K, int splits);
/* K % 64 == 0; N % 256 == 0, up to 64 rows N % 96 == 0 (swiglu: % 288); swiglu: for vt_launch_gemm_frag_swiglu */
vt_gemm_plan vt_gemm_frag_plan(int M, int N, int K, int swiglu);
/* The same on row-major weights W[N, K], N % 128 == 0, K % 64 == 0, in at most `most` cuts: d_y [M, N]; d_part: pl.cuts planes of
 * [M, N - pl.col0] (pl.cuts 1: not used) */
vt_gemm_plan vt_gemm_row_major_plan(int M, int N, int K, int most, float *us);      /* us: what it is expected to take; infinite where no strip or tile takes so many columns or such a K */
float vt_gemm_equal_us(int M, int N, int K, int cuts);      /* the same of vt_launch_gemm and, with cuts, the sum of its planes */
int vt_gemm_row_major_prepare(void);      /* once per context; 0 / -1 */
void vt_launch_gemm_row_major(float *d_y, float *d_part, const uint16_t *d_Ahi, const uint16_t *d_Alo, const uint16_t *d_W, int M, int N, int K,
                              const vt_gemm_plan &pl);
void vt_launch_gemm_frag(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                         const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl);
/* gate|up product on paired weights with SiLU(gate) * up as its epilogue -> planes d_hhi / d_hlo [M, ldh]; the
 * columns from pl.col0 on pass through d_tail [pl.cuts][M, N - pl.col0] and a second launch */
void vt_launch_gemm_frag_swiglu(uint16_t *d_hhi, uint16_t *d_hlo, int ldh, float *d_tail, const uint16_t *d_Ahi,
                                const uint16_t *d_Alo, const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl);
/* The same for M <= 64 rows on strips of 96 columns, or 288 for the gate|up product (vt_gemm_rows.hip), weights in the same
 * fragment order: N a multiple of those; the cuts need not divide K. */
void vt_launch_gemm_few_rows(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                             const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl);
/* The codec's products (vt_codec_gemm.hip): activations as two fp16 planes [M, K] with an exponent per row, weights in
 * fragment order with an exponent per column, from fp32 W[N, K] by vt_codec_weight_layout (d_Wf: 2 N K elements; 0 / -1).
 * N % 64 == 0 (more than 64 rows: % 256), K % 64 == 0.  d_C: [M, pl.col0] and, behind it, pl.cuts planes of
 * [M, N - pl.col0]. */
vt_gemm_plan vt_codec_gemm_plan(int M, int N, int K);
int vt_codec_weight_layout(uint16_t *d_Wf, int *d_col_exp, const float *d_W, int N, int K);
void vt_launch_codec_gemm(float *d_C, const uint16_t *d_hi, const uint16_t *d_lo, const int *d_row_exp,
                          const uint16_t *d_Wf, const int *d_col_exp, int M, int N, int K, const vt_gemm_plan &pl);
/* row-major bf16 W[N, K] -> the fragment-order copy (same size); N % 32 == 0, K % 64 == 0.  pair: W holds
 * (gate, up) rows interleaved and every 32 fragment columns become 16 gates followed by their 16 ups, the order
 * vt_launch_gemm_frag_swiglu expects. */
void vt_launch_frag_layout(uint16_t *d_Wf, const uint16_t *d_W, int N, int K, int pair);
void vt_launch_swiglu_pair_tail(uint16_t *d_hi, uint16_t *d_lo, int ldh, int h_col0, const float *d_tail, int planes,
                                size_t stride, int rows, int tw);
/* n even */
void vt_launch_split(uint16_t *d_hi, uint16_t *d_lo, const float *d_x, size_t n);
/* rows of 3072: x = x_in (d_x itself, or rows in memory that the device reads) + the product (cuts > 0; one plane below col0, the
 * sum of `cuts` from there on), then planes of rmsnorm(x)*w (d_w != NULL) */
void vt_launch_residual_norm_split(float *d_x, const float *x_in, const float *d_part, int col0, int cuts, size_t part_stride,
                                   const float *d_w, uint16_t *d_hi, uint16_t *d_lo, int rows);
/* n_out a multiple of 4, tail_col0 of 8: planes of silu(gate)*up from interleaved (gate, up) pairs */
void vt_launch_swiglu_split(uint16_t *d_hi, uint16_t *d_lo, const float *d_gu, size_t n_out, int tail_col0,
                            const float *d_tail, int tail_planes, size_t tail_stride);
void vt_launch_sum_planes(float *d_out, const float *d_part, int splits, size_t stride, size_t n);

#ifdef __HIPCC__
/* SiLU(gate) * up (voxtral_tts_kernels.c's tts_silu and tts_mul_inplace), four at a time.  The quotient
 * g / (1 + exp(-g)) with exp2 of the product with log2(e), the product's rounding error carried on to first order, a
 * denominator in two floats, and the reciprocal estimate with one correction of the quotient.  Largest error against 64
 * bits, and of g / (1 + expf(-g)) with an IEEE division: 1.36e-7 / 1.84e-7 for g in -83 .. 0, 0.91e-7 / 1.50e-7 above.
 * A third of the instructions of that formula: as the epilogue of a 128 x 256 gate|up tile it took 5 of its 7.5 us. */
__device__ __forceinline__ float vt_silu_mul_small(float g, float u) {       /* |g| < VT_SILU_SMALL, or NaN */
    const float log2e = 1.44269504f, log2e_lo = 1.92596303e-8f;              /* log2(e) = their sum */
    const float t = __fmul_rn(-g, log2e);
    const float r = fmaf(-g, log2e_lo, fmaf(-g, log2e, -t));                 /* what the product's rounding left out */
    const float e = __builtin_amdgcn_exp2f(t);
    const float d = __fadd_rn(1.0f, e);                                      /* the denominator is d + dl */
    const float dl = fmaf(e, r * 0.693147181f, fminf(e, 1.0f) - (d - fmaxf(e, 1.0f)));
    const float y = __builtin_amdgcn_rcpf(d);
    float q = g * y;
    q = fmaf(fmaf(-q, dl, fmaf(-q, d, g)), y, q);
    return q * u;
}
#define VT_SILU_SMALL 83.0f       /* exp(-g) and its reciprocal stay normal, with room for the quotient */
/* h = silu(g) * u for N of them */
template <int N>
__device__ __forceinline__ void vt_silu_mul(float (&h)[N], const float (&g)[N], const float (&u)[N]) {
    float m = 0.f;
#pragma unroll
    for (int v = 0; v < N; v++) {
        h[v] = vt_silu_mul_small(g[v], u[v]);
        m = fmaxf(m, fabsf(g[v]));
    }
    /* beyond, infinities included, the formula itself (rare: skipped by waves that have no such gate) */
    if (__builtin_expect(m >= VT_SILU_SMALL, 0)) {
#pragma unroll
        for (int v = 0; v < N; v++)
            if (fabsf(g[v]) >= VT_SILU_SMALL) h[v] = __fmul_rn(__fdiv_rn(g[v], __fadd_rn(1.0f, expf(-g[v]))), u[v]);
    }
}
__device__ __forceinline__ f32x4 vt_silu_mul4(const f32x4 &g, const f32x4 &u) {
    const float gs[4] = {g.x, g.y, g.z, g.w}, us[4] = {u.x, u.y, u.z, u.w};
    float h[4];
    vt_silu_mul<4>(h, gs, us);
    return f32x4{h[0], h[1], h[2], h[3]};
}

/* Four rows v = 0..3 of a paired column block (16 gates in lanes 0..15 of 32, the ups of the same h columns in lanes 16..31): the
 * rows 0 and 1 for the lanes below 16, 2 and 3 for those above, gate and up side by side. */
__device__ __forceinline__ void vt_pair_rows(const f32x4 &q, float (&g)[2], float (&u)[2]) {
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(q[r]), __float_as_uint(q[2 + r]), false, false);
        g[r] = __uint_as_float(x[0]);
        u[r] = __uint_as_float(x[1]);
    }
}
/* Those two rows of h -> plane words of two columns, so that a plane takes one store of 4 bytes per lane: an even lane's row 0, an odd
 * one's row 1, columns c & ~1 and c | 1. */
__device__ __forceinline__ void vt_pair_words(float h0, float h1, unsigned &hi, unsigned &lo) {
    const bool odd = threadIdx.x & 1;
    const float got = vt_dpp<0xB1>(odd ? h0 : h1);               /* the other lane's value of my row */
    vt_split_planes2(odd ? got : h0, odd ? h1 : got, hi, lo);
}
#endif

#endif /* VT_GEMM_H */

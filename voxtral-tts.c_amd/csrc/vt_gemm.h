/*
 * vt_gemm.h - launchers of the bf16 MFMA matrix product on (hi, lo) activation
 * planes and of the row kernels that produce those planes.
 */
#ifndef VT_GEMM_H
#define VT_GEMM_H

#include <stddef.h>
#include <stdint.h>

/* N a multiple of 128, K/splits a multiple of 64 */
int vt_gemm_shape_ok(int M, int N, int K, int splits);
/* d_C: `splits` planes of [M, N] fp32, plane s holds the sum over K range s */
void vt_launch_gemm(float *d_C, const uint16_t *d_Ahi, const uint16_t *d_Alo, const uint16_t *d_W,
                    int M, int N, int K, int splits);
/* the same with the row pitch of C and the distance between planes given */
void vt_launch_gemm_ex(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                       const uint16_t *d_W, int M, int N, int K, int splits);
/* How a product of the backbone is done on fragment-order weights (vt_launch_frag_layout): the columns below
 * col0 as whole tiles (one plane), the others with K in `cuts` cuts (that many partial planes, to be added in
 * order by whoever reads the result).  mb, cw: the tile (vt_gemm_wide.hip; mb 0: vt_gemm_rows.hip). */
#define VT_MAX_CUTS 8
struct vt_gemm_plan { int mb, cw, col0, cuts; };
/* N % 256 == 0, K % 64 == 0; swiglu: for vt_launch_gemm_frag_swiglu */
vt_gemm_plan vt_gemm_frag_plan(int M, int N, int K, int swiglu);
void vt_launch_gemm_frag(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                         const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl);
/* gate|up product on paired weights with SiLU(gate) * up as its epilogue -> planes d_hhi / d_hlo [M, ldh]; the
 * columns from pl.col0 on pass through d_tail [pl.cuts][M, N - pl.col0] and a second launch */
void vt_launch_gemm_frag_swiglu(uint16_t *d_hhi, uint16_t *d_hlo, int ldh, float *d_tail, const uint16_t *d_Ahi,
                                const uint16_t *d_Alo, const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl);
/* The same product for M <= 64 rows on 64-column tiles (vt_gemm_rows.hip), weights in the same fragment order:
 * N % 64 == 0, K % 64 == 0; the cuts need not divide K. */
int vt_gemm_rows_ok(int M, int N, int K);
int vt_gemm_rows_cuts(int M, int N, int K, int most);
void vt_launch_gemm_rows(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                         const uint16_t *d_Wf, int M, int N, int K, int splits);
void vt_launch_gemm_rows_swiglu(uint16_t *d_hhi, uint16_t *d_hlo, int ldh, float *d_tail, const uint16_t *d_Ahi,
                                const uint16_t *d_Alo, const uint16_t *d_Wf, int M, int n_main, int n_tail, int K,
                                int tail_splits);
/* row-major bf16 W[N, K] -> the fragment-order copy (same size); N % 32 == 0, K % 64 == 0.  pair: W holds
 * (gate, up) rows interleaved and every 64 fragment columns become 32 gates followed by their 32 ups
 * (N % 64 == 0), the order vt_launch_gemm_frag_swiglu expects. */
void vt_launch_frag_layout(uint16_t *d_Wf, const uint16_t *d_W, int N, int K, int pair);
void vt_launch_swiglu_pair_tail(uint16_t *d_hi, uint16_t *d_lo, int ldh, int h_col0, const float *d_tail, int planes,
                                size_t stride, int rows, int tw);
/* n even */
void vt_launch_split(uint16_t *d_hi, uint16_t *d_lo, const float *d_x, size_t n);
/* rows of 3072: x += the product (cuts > 0; one plane below col0, the sum of `cuts` from there on), then planes
 * of rmsnorm(x)*w (d_w != NULL) */
void vt_launch_residual_norm_split(float *d_x, const float *d_part, int col0, int cuts, size_t part_stride,
                                   const float *d_w, uint16_t *d_hi, uint16_t *d_lo, int rows);
/* n_out a multiple of 4, tail_col0 of 8: planes of silu(gate)*up from interleaved (gate, up) pairs */
void vt_launch_swiglu_split(uint16_t *d_hi, uint16_t *d_lo, const float *d_gu, size_t n_out, int tail_col0,
                            const float *d_tail, int tail_planes, size_t tail_stride);
void vt_launch_sum_planes(float *d_out, const float *d_part, int splits, size_t stride, size_t n);

#endif /* VT_GEMM_H */

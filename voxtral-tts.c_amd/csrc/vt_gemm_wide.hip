/*
 * vt_gemm_wide.hip - the backbone's prefill products on the tile kernels of vt_gemm_tiles.h, more than 64 rows; the
 * plans (vt_gemm_plans.h) on this card.
 */
#include "vt_gemm_tiles.h"

/* ---- plans and launches ---------------------------------------------------------------------------- */

vt_gemm_plan vt_gemm_frag_plan(int M, int N, int K, int swiglu) { return gp_frag(g_vt.n_cu, M, N, K, swiglu); }
vt_gemm_plan vt_codec_gemm_plan(int M, int N, int K) { return gp_codec(g_vt.n_cu, M, N, K); }
vt_gemm_plan vt_gemm_row_major_plan(int M, int N, int K, int most, float *us) { return gp_row_major(g_vt.n_cu, M, N, K, most, us); }
float vt_gemm_equal_us(int M, int N, int K, int cuts) { return gp_equal_us(g_vt.n_cu, M, N, K, cuts); }

template <int MB, int CW, int NB, bool FRAG = true, bool PAIR = false>
static int gw_prepare(void) {
    static int attr_device = -1;
    if (attr_device == g_vt.device) return 0;
    if (vt_check(hipFuncSetAttribute((const void *)vt_gemm_wide_kernel<gm_bf16, MB, CW, NB, FRAG, PAIR>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     2 * gw_shape<MB, CW, PAIR>::STAGE), "product LDS size"))
        return -1;
    attr_device = g_vt.device;
    return 0;
}

/* With the context: a product on a caller's weights may be the first call inside a stream capture */
int vt_gemm_row_major_prepare(void) {
    return gw_prepare<3, 2, 2, false>() || gw_prepare<3, 2, 3, false>() || gw_prepare<3, 4, 2, false>() || gw_prepare<4, 2, 3, false>() || gw_prepare<4, 4, 2, false>() ? -1 : 0;
}

template <int MB, int CW, int NB, bool FRAG = true, bool PAIR = false>
static void gw_launch(const gw_list &list, const uint16_t *d_Ahi, const uint16_t *d_Alo, int M, int K) {
    constexpr int LDS = 2 * gw_shape<MB, CW, PAIR>::STAGE;
    if (gw_prepare<MB, CW, NB, FRAG, PAIR>()) return;
    const int items = list.part[0].items;      /* every workgroup takes an item of the first part */
    hipLaunchKernelGGL((vt_gemm_wide_kernel<gm_bf16, MB, CW, NB, FRAG, PAIR>), dim3(items < g_vt.n_cu ? items : g_vt.n_cu), dim3(256), LDS, g_vt.stream,
                       list, d_Ahi, d_Alo, M, K);
}

static void gw_run(const vt_gemm_plan &pl, gw_part whole, gw_part cut, const uint16_t *d_Ahi, const uint16_t *d_Alo, int M, int N, int K) {
    gw_list list = {};
    whole.n_tiles = pl.col0 / pl.tn;
    whole.splits = 1;
    cut.n_tiles = (N - pl.col0) / pl.tn;
    cut.splits = pl.cuts;
    gw_add(list, whole, M, pl.tm, K);
    gw_add(list, cut, M, pl.tm, K);
    typedef void (*fn)(const gw_list &, const uint16_t *, const uint16_t *, int, int);
    static const fn launch[4][4] = {{NULL, gw_launch<5, 2, 3, true, true>, gw_launch<5, 4, 2, true, true>, gw_launch<5, 4, 3, true, true>},
                                    {gw_launch<3, 2, 2>, gw_launch<3, 2, 3>, gw_launch<3, 4, 2>, gw_launch<3, 4, 3>},
                                    {NULL, NULL, gw_launch<7, 4, 2, true, true>, NULL},
                                    {NULL, gw_launch<4, 2, 3>, gw_launch<4, 4, 2>, gw_launch<4, 4, 3>}};
    static const fn row_major[2][3] = {{gw_launch<3, 2, 2, false>, gw_launch<3, 2, 3, false>, gw_launch<3, 4, 2, false>}, {NULL, gw_launch<4, 2, 3, false>, gw_launch<4, 4, 2, false>}};
    (pl.row_major ? row_major[pl.tm == 128][gw_width(pl.tn)] : launch[gw_height(pl.tm)][gw_width(pl.tn)])(list, d_Ahi, d_Alo, M, K);
}

/* y[:, col0 ..] = the planes' sum, in order, all of them requested in front of the first addition: a chain of memory latencies */
__global__ void __launch_bounds__(256) vt_sum_cut_columns_kernel(float *y, const float *part, int cuts, int M, int N, int col0) {
    const int w = (N - col0) / 4;
    const size_t n = (size_t)M * w;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        f32x4 q[VT_MAX_CUTS];
#pragma unroll
        for (int p = 0; p < VT_MAX_CUTS; p++) q[p] = reinterpret_cast<const f32x4 *>(part)[(p < cuts ? p : 0) * n + i];
        f32x4 v = q[0];
#pragma unroll
        for (int p = 1; p < VT_MAX_CUTS; p++)
            if (p < cuts) { v.x = __fadd_rn(v.x, q[p].x); v.y = __fadd_rn(v.y, q[p].y); v.z = __fadd_rn(v.z, q[p].z); v.w = __fadd_rn(v.w, q[p].w); }
        *reinterpret_cast<f32x4 *>(y + i / w * N + col0 + i % w * 4) = v;
    }
}

void vt_launch_gemm_row_major(float *d_y, float *d_part, const uint16_t *d_Ahi, const uint16_t *d_Alo, const uint16_t *d_W, int M, int N, int K,
                              const vt_gemm_plan &pl) {
    const int cut = N - pl.col0;
    const size_t plane = (size_t)M * cut;
    if (pl.tm == 0) vt_launch_gemm_few_rows(pl.cuts > 1 ? d_part : d_y, N, plane, d_Ahi, d_Alo, d_W, M, N, K, pl);
    else gw_run(pl, gw_part{d_y, d_W, 0, N, 0, 0, NULL, NULL, 0, NULL, NULL},
                gw_part{d_part, d_W + (size_t)pl.col0 * K, plane, cut, 0, 0, NULL, NULL, 0, NULL, NULL}, d_Ahi, d_Alo, M, N, K);
    if (pl.cuts > 1) {
        const size_t n = plane / 4;
        hipLaunchKernelGGL(vt_sum_cut_columns_kernel, dim3((unsigned)((n + 255) / 256 > 4096 ? 4096 : (n + 255) / 256)), dim3(256), 0, g_vt.stream, d_y, d_part, pl.cuts, M, N, pl.col0);
    }
}

void vt_launch_gemm_frag(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                         const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl) {
    if (pl.tm == 0) { vt_launch_gemm_few_rows(d_C, ldc, plane_stride, d_Ahi, d_Alo, d_Wf, M, N, K, pl); return; }
    gw_run(pl, gw_part{d_C, d_Wf, plane_stride, ldc, 0, 0, NULL, NULL, 0, NULL, NULL},
           gw_part{d_C + pl.col0, d_Wf + (size_t)pl.col0 * K, plane_stride, ldc, 0, 0, NULL, NULL, 0, NULL, NULL}, d_Ahi, d_Alo, M, N, K);
}

void vt_launch_gemm_frag_swiglu(uint16_t *d_hhi, uint16_t *d_hlo, int ldh, float *d_tail, const uint16_t *d_Ahi,
                                const uint16_t *d_Alo, const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl) {
    const int tail = N - pl.col0;
    if (pl.tm == 0)
        vt_launch_gemm_few_rows(d_tail, N, (size_t)M * N, d_Ahi, d_Alo, d_Wf, M, N, K, pl);
    else
        gw_run(pl, gw_part{NULL, d_Wf, 0, 0, 0, 0, d_hhi, d_hlo, ldh, NULL, NULL},
               gw_part{d_tail, d_Wf + (size_t)pl.col0 * K, (size_t)M * tail, tail, 0, 0, NULL, NULL, 0, NULL, NULL}, d_Ahi, d_Alo, M, N, K);
    if (tail) vt_launch_swiglu_pair_tail(d_hhi, d_hlo, ldh, pl.col0 / 2, d_tail, pl.cuts, (size_t)M * tail, M, tail);
}

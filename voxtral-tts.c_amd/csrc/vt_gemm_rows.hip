/*
 * vt_gemm_rows.hip - the backbone's prefill products of up to 64 rows, on vt_gemm_rows_kernel (vt_gemm_tiles.h).
 */
#include "vt_gemm_tiles.h"

int vt_gemm_rows_ok(int M, int N, int K) { return M >= 1 && M <= 64 && N % GR_TN == 0 && K % 64 == 0; }

/* Waves of a workgroup: 8 while the registers of a wave (sums, two sets of weights, staged rows) fit two waves
 * per SIMD; beyond 40 rows they spill (64 rows, gate|up: 63 us against 34 with 4 waves). */
#define GR_ROWS_8_WAVES 40
int vt_gemm_rows_waves(int M) { return M <= GR_ROWS_8_WAVES ? 8 : 4; }

template <int NP>
static int gr_launch_np(const gr_plan &plan, int grid, const uint16_t *d_Ahi, const uint16_t *d_Alo, int M, int K) {
    constexpr int NW = 8 * NP <= GR_ROWS_8_WAVES ? 8 : 4;
    static int attr_set = 0;
    const int lds = NW * 2 * 32 * ((NP + 3) / 4) * GM_STAGE_ROW;
    if (!attr_set) {
        if (vt_check(hipFuncSetAttribute((const void *)vt_gemm_rows_kernel<gm_bf16, NP, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, lds), "product LDS size"))
            return -1;
        attr_set = 1;
    }
    hipLaunchKernelGGL((vt_gemm_rows_kernel<gm_bf16, NP, NW>), dim3(grid), dim3(64 * NW), lds, g_vt.stream, plan, d_Ahi, d_Alo, M, K);
    return 0;
}

static void gr_launch(const gr_plan &plan, const uint16_t *d_Ahi, const uint16_t *d_Alo, int M, int K) {
    static int (*const launch[8])(const gr_plan &, int, const uint16_t *, const uint16_t *, int, int) = {
        gr_launch_np<1>, gr_launch_np<2>, gr_launch_np<3>, gr_launch_np<4>, gr_launch_np<5>, gr_launch_np<6>, gr_launch_np<7>, gr_launch_np<8>};
    const int items = plan.part[0].n_tiles * plan.part[0].splits;     /* every workgroup takes an item of the first part */
    launch[(M + 7) / 8 - 1](plan, items < g_vt.n_cu ? items : g_vt.n_cu, d_Ahi, d_Alo, M, K);
}

int vt_gemm_rows_cuts(int nw, int N, int K, int most) {
    /* of the cut counts that leave every CU at most one item, the fewest planes among those with the fewest
     * K steps on the busiest wave */
    const int tiles = N / GR_TN, steps = K / 64;
    int best = 1, best_cost = steps;
    for (int c = 1; c <= most && tiles * c <= g_vt.n_cu; c++) {
        const int cost = ((steps + c - 1) / c + nw - 1) / nw;
        if (c == 1 || cost < best_cost) { best = c; best_cost = cost; }
    }
    return best;
}

void vt_launch_gemm_rows(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                         const uint16_t *d_Wf, int M, int N, int K, int splits) {
    gr_plan plan = {};
    plan.n_parts = 1;
    plan.part[0] = gr_part{d_C, d_Wf, plane_stride, ldc, N / GR_TN, splits, NULL, NULL, 0, NULL, NULL};
    gr_launch(plan, d_Ahi, d_Alo, M, K);
}

void vt_launch_gemm_rows_swiglu(uint16_t *d_hhi, uint16_t *d_hlo, int ldh, float *d_tail, const uint16_t *d_Ahi,
                                const uint16_t *d_Alo, const uint16_t *d_Wf, int M, int n_main, int n_tail, int K, int tail_splits) {
    gr_plan plan = {};
    if (n_main > 0) plan.part[plan.n_parts++] = gr_part{NULL, d_Wf, 0, 0, n_main / GR_TN, 1, d_hhi, d_hlo, ldh, NULL, NULL};
    if (n_tail > 0)
        plan.part[plan.n_parts++] = gr_part{d_tail, d_Wf + (size_t)n_main * K, (size_t)M * n_tail, n_tail, n_tail / GR_TN, tail_splits, NULL, NULL, 0, NULL, NULL};
    gr_launch(plan, d_Ahi, d_Alo, M, K);
}

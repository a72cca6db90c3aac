/*
 * vt_prefill.hip - backbone prefill over a row block of the sequence (replaces
 * tts_cuda_llm_prefill, voxtral_tts_cuda.cu:806-893; the layer follows
 * voxtral_tts_llm.c:299-366).
 *
 * Per layer: RMSNorm into (hi, lo) bf16 planes -> q|k|v product on the matrix
 * cores -> RoPE + cache append -> causal attention on the matrix cores ->
 * output projection -> residual + RMSNorm -> gate/up product with SiLU*up ->
 * down projection -> residual fused with the next layer's RMSNorm.  Tiles and
 * K cuts of the products follow the row count (vt_gemm_frag_plan); the kernels
 * between them are told which columns are cut.
 */
#include "vt_state.h"
#include "vt_gemm.h"
#include "vt_requests.h"

#include <math.h>
#include <string.h>


/* ---- causal attention, 32 query rows x 32 keys per matrix-core tile ----------------
 * (tts_causal_attention, voxtral_tts_kernels.c:403-465, for head_dim 128 and four
 * query heads per KV head.)
 *
 * Workgroup = (KV head, block of QB queries of its four query heads), eight waves.  A wave holds 32 query rows: QB = 32
 * queries of one head, or QB = 16 queries of two heads; the NS = 2 or 4 waves with the same rows take the key
 * tiles in turn (tile modulo NS) and merge at the end.  The waves of a residue share a tile of 32 keys in LDS.  Both
 * products run on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16) with every fp32 operand split in (hi, lo) bf16
 * planes as in the projections: a b = hi_a hi_b + hi_a lo_b + lo_a hi_b, 16 mantissa bits per operand, fp32 accumulation.
 * Scores are computed transposed, S^T = K Q^T, so that a lane owns one query row: lane l holds row l%32 and the keys
 * 8*(v/4) + 4*(l/32) + v%4 in accumulator element v.  The softmax state is then per lane (one exchange between the
 * two lane groups per tile), and the sixteen probabilities a lane holds are exactly its share of the reduction index
 * of the second product O^T = V^T P^T (the k order inside a matrix instruction is free as long as both operands
 * agree: slot j of lane group g in the instruction of key half t stands for key 16 t + 8*(j/4) + 4 g + j%4).
 *
 * A tile of K and V is 32 KB of operands in the order in which the instructions take them (1 KB per instruction and
 * plane, lane l at byte 16 l), made once per layer by vt_kv_image_kernel; a workgroup copies tiles from
 * memory straight into LDS (buffer loads to LDS, no registers).  Two arrays, not two halves of one: the compiler then
 * knows that reading one does not have to wait for what arrives in the other.
 *
 * What bounds it: 48 matrix instructions of 32 cycles per wave and tile beside 32 KB of LDS reads and about 250 vector
 * instructions, two waves per SIMD: 2.0 to 2.3 us per NS tiles, 1.28 of them matrix instructions at 2.4 GHz; and
 * 7 to 9 us in front and behind (queries 2.1, their planes 1.5, merge and stores 2.5: each of them code that is run once and
 * comes from memory).  us per launch inside a prefill of 37 / 226 / 512 / 1531 rows: 7.7 / 12.2 / 17.8 /
 * 65.6, where 16 queries per wave on 16 x 16 x 32 instructions, four waves and tiles copied through registers took 9.0 / 15.8 /
 * 24.5 / 125.5; at 37 rows 10.9 now with the tiles made here (PA_HERE_ROWS), which took a launch of 6.1. */
/* Queries per workgroup: 16 as long as that gives the CUs more to do at once (twice the workgroups, each half as many
 * rounds of tiles), 32 from where every CU is busy either way and the tiles are copied half as often.  us per launch
 * at 37 / 226 / 512 / 1000 / 1531 / 3000 rows, 16: 7.5 / 10.5 / 16.4 / 34.4 / 70.1 / 236.7, 32: 9.0 / 14.3 / 22.4 / 39.5 /
 * 65.4 / 213.8. */
#define PA_SHORT_QT 16
#define PA_LONG_QT 32
#define PA_SHORT_ROWS 1200
/* Up to this many rows in all, the cached ones included, the attention's workgroups make the (at most two) tiles themselves instead of
 * reading what a launch of its own has made: with the strips' shorter code (vt_gemm_rows.hip) prefills of 6 / 20 / 37 / 64 rows 1780 / 2010 / 2356 / 2840 ->
 * 1701 / 1861 / 2244 / 2599 us.  With three and four tiles a workgroup makes them two at a time, and every one of six or eight workgroups per
 * head makes its own: 3177 us instead of 3130 at 96 rows, the same at 128.  (Asking for the rows in front of the queries' work needs 160 registers, and
 * its code twice: 2387 us at 37 rows.) */
#define PA_HERE_ROWS 64
#define PA_PLANE 8192             /* bytes of a plane of a tile: 8 slices of K, 4 dim blocks x 2 key halves of V, 1 KB each */
#define PA_TILE_BYTES (4 * PA_PLANE)                  /* K hi, K lo, V hi, V lo */

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

/* eight consecutive k of a matrix-core operand from two fp32 quads: (hi, lo) planes */
__device__ __forceinline__ void pa_planes8(const f32x4 &a, const f32x4 &b, bf16x8 &hi, bf16x8 &lo) {
    unsigned h0, h1, h2, h3, l0, l1, l2, l3;
    vt_split_planes2(a.x, a.y, h0, l0);
    vt_split_planes2(a.z, a.w, h1, l1);
    vt_split_planes2(b.x, b.y, h2, l2);
    vt_split_planes2(b.z, b.w, h3, l3);
    hi = __builtin_bit_cast(bf16x8, u32x4{h0, h1, h2, h3});
    lo = __builtin_bit_cast(bf16x8, u32x4{l0, l1, l2, l3});
}

/* K and V of one layer as the attention wants them in its LDS: per (kv head, tile of 32 keys) the operands described
 * above, img[kvh][tile].  K: slice ks of lane l = key l%32, dims 16 ks + 8 (l/32) .. + 8; V: dim block b and key half t of
 * lane l = dim 32 b + l%32, keys 16 t + 4 (l/32) + 0..3 and the four 8 further on.  Workgroup = (tile, kv head), 128
 * threads for K and 128 for V; thread (sg, cg) owns the dims 4*cg .. + 4 of the 8 keys that lane group sg % 2 meets in
 * key half sg / 2, so that the transposed V write is one 16-byte store per dim and plane.
 * The rows from `start` on come from the q|k|v product: the sum of `planes` split-K planes (`plane_stride` floats apart, fixed order; only
 * the columns from col0 on are cut, a multiple of 128), k rotated (adjacent pairs, voxtral_tts_kernels.c:616-634; the table holds
 * (cos, sin) per pair), and are appended to the cache on the way (voxtral_tts_llm.c:317-324).  Earlier rows come from the cache; rows
 * from kv_rows on are zeros (their keys are masked).
 *
 * Every request goes through a descriptor that covers the rows which this source has, and brings zeros for the others, so that a row is the sum
 * of what its sources brought: no address of 64 bits and no branch per row.  Up to three planes are in flight beside the first:
 * with one after the other a launch at 37 rows in four cuts took 7.3 us.  (What runs once comes from memory, instructions included:
 * with addresses and branches per row the kernel had 7.4 KB of code instead of 4.1, and at 96 rows a launch took 7.0 us instead of 6.3.) */
__device__ __forceinline__ int pa_key(int sg, int i) { return 16 * (sg >> 1) + 4 * (sg & 1) + 8 * (i >> 2) + (i & 3); }

struct pa_rows {
    const float *qkv;             /* [kv_rows - start, 6144] planes */
    int col0, planes;
    size_t plane_stride;
    float *kc, *vc;               /* [kv_rows, 1024] */
    const float *rope;
    int start, kv_rows;
};

/* 256 threads make the K planes of tile `tile` of kv head kvh at Kt (threads 0..127) and its V planes at Vt (threads 128..255); of the
 * rows from `start` on, first .. first + n - 1 are appended to the cache. */
template <class PTR>
__device__ __forceinline__ void pa_make_tile(PTR Kt, PTR Vt, const pa_rows &in, int kvh, int tile, int thread, int first, int n) {
    const bool is_v = __builtin_amdgcn_readfirstlane(thread >> 7);           /* a wave is all K or all V */
    const int tl = thread & 127, sg = tl >> 5, cg = tl & 31;
    const int wide = VT_Q_DIM + (is_v ? VT_KV_DIM : 0) + kvh * VT_HEAD_DIM, col = kvh * VT_HEAD_DIM + 4 * cg;
    const int planes = wide < in.col0 ? 1 : in.planes;                       /* a head whose columns are not cut has one */
    /* descriptors begin at the tile's first row, or the source's where that lies within (rows in front of it: beyond any size) */
    const int t0 = tile * 32, row0 = t0 + pa_key(sg, 0), f0 = max(t0, in.start), fresh_bytes = max(min(in.kv_rows - f0, 32), 0) * VT_QKV_DIM * 4;
    const float *fresh = in.qkv + (size_t)(f0 - in.start) * VT_QKV_DIM;
    float *const kc = in.kc, *const vc = in.vc, *const cache = is_v ? vc : kc;
    const int at = (row0 - f0) * (VT_QKV_DIM * 4) + (wide + 4 * cg) * 4;
    auto off = [](int i, int pitch) { return (8 * (i >> 2) + (i & 3)) * pitch; };
    f32x4 r8[8], cs[8], w[3][8];
    const __amdgpu_buffer_rsrc_t d0 = vt_buffer(fresh, fresh_bytes);
    /* (a caller's own K and V may have more rows than the table: nothing of it is read for rows that are not rotated) */
    const __amdgpu_buffer_rsrc_t dc = vt_buffer(in.rope + (size_t)t0 * VT_HEAD_DIM, is_v || fresh_bytes == 0 ? 0 : min(in.kv_rows - t0, 32) * VT_HEAD_DIM * 4);
#pragma unroll
    for (int i = 0; i < 8; i++) r8[i] = vt_buffer_ld4(d0, at + off(i, VT_QKV_DIM * 4));
#pragma unroll
    for (int i = 0; i < 8; i++) cs[i] = vt_buffer_ld4(dc, (row0 - t0) * (VT_HEAD_DIM * 4) + 16 * cg + off(i, VT_HEAD_DIM * 4));
    for (int p = 1; p < planes; p += 3) {
#pragma unroll
        for (int z = 0; z < 3; z++) {
            const __amdgpu_buffer_rsrc_t d = vt_buffer(fresh + (size_t)min(p + z, planes - 1) * in.plane_stride, p + z < planes ? fresh_bytes : 0);
#pragma unroll
            for (int i = 0; i < 8; i++) w[z][i] = vt_buffer_ld4(d, at + off(i, VT_QKV_DIM * 4));
        }
#pragma unroll
        for (int z = 0; z < 3; z++)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                r8[i].x = __fadd_rn(r8[i].x, w[z][i].x); r8[i].y = __fadd_rn(r8[i].y, w[z][i].y);
                r8[i].z = __fadd_rn(r8[i].z, w[z][i].z); r8[i].w = __fadd_rn(r8[i].w, w[z][i].w);
            }
    }
    if (!is_v) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const f32x4 k = r8[i], c = cs[i];
            r8[i] = f32x4{__fsub_rn(__fmul_rn(k.x, c.x), __fmul_rn(k.y, c.y)), __fadd_rn(__fmul_rn(k.x, c.y), __fmul_rn(k.y, c.x)),
                          __fsub_rn(__fmul_rn(k.z, c.z), __fmul_rn(k.w, c.w)), __fadd_rn(__fmul_rn(k.z, c.w), __fmul_rn(k.w, c.z))};
        }
    }
    const int s0 = max(t0, first);
    const __amdgpu_buffer_rsrc_t ds = vt_buffer(cache + (size_t)s0 * VT_KV_DIM, max(min(min(first + n, in.kv_rows), t0 + 32) - s0, 0) * VT_KV_DIM * 4);
#pragma unroll
    for (int i = 0; i < 8; i++)
        vt_buffer_st4(ds, (row0 - s0) * (VT_KV_DIM * 4) + col * 4 + off(i, VT_KV_DIM * 4), r8[i]);
    if (t0 < in.start) {                                 /* earlier rows */
        const __amdgpu_buffer_rsrc_t d = vt_buffer(cache + (size_t)t0 * VT_KV_DIM, min(in.start - t0, 32) * VT_KV_DIM * 4);
#pragma unroll
        for (int i = 0; i < 8; i++) w[0][i] = vt_buffer_ld4(d, (row0 - t0) * (VT_KV_DIM * 4) + col * 4 + off(i, VT_KV_DIM * 4));
#pragma unroll
        for (int i = 0; i < 8; i++) r8[i] += w[0][i];
    }
    if (!is_v) {
        PTR to = Kt + (cg >> 2) * 1024 + ((cg >> 1) & 1) * 512 + pa_key(sg, 0) * 16 + (cg & 1) * 8;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            u32x2 h, l;
            vt_split_planes4(r8[i].x, r8[i].y, r8[i].z, r8[i].w, h, l);
            *reinterpret_cast<u32x2 *>(to + off(i, 16)) = h;
            *reinterpret_cast<u32x2 *>(to + off(i, 16) + PA_PLANE) = l;
        }
    } else {
        PTR to = Vt + ((cg >> 3) * 2 + (sg >> 1)) * 1024 + ((sg & 1) * 32 + (4 * cg) % 32) * 16;
#pragma unroll
        for (int d = 0; d < 4; d++) {
            bf16x8 h, l;
            pa_planes8(f32x4{r8[0][d], r8[1][d], r8[2][d], r8[3][d]}, f32x4{r8[4][d], r8[5][d], r8[6][d], r8[7][d]}, h, l);
            *reinterpret_cast<bf16x8 *>(to + 16 * d) = h;
            *reinterpret_cast<bf16x8 *>(to + 16 * d + PA_PLANE) = l;
        }
    }
}

__global__ void __launch_bounds__(256) vt_kv_image_kernel(unsigned char *img, int img_tiles, pa_rows in) {
    unsigned char *Kt = img + ((size_t)blockIdx.y * img_tiles + blockIdx.x) * PA_TILE_BYTES;
    pa_make_tile(Kt, Kt + 2 * PA_PLANE, in, (int)blockIdx.y, (int)blockIdx.x, (int)threadIdx.x, in.start, in.kv_rows - in.start);
}

typedef float pa_f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ pa_f32x16 pa_mfma(const bf16x8 &a, const bf16x8 &b, const pa_f32x16 &c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
/* the larger of this lane's value and that of the lane 32 away */
__device__ __forceinline__ float pa_max_halves(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

/* HERE (QB 16, at most two tiles in all): no images; a workgroup makes the tiles that its queries see in its own LDS, from the rows
 * `in`, and appends its queries' rows to the cache. */
template <int QB, bool HERE>
__global__ void __launch_bounds__(512)
vt_prefill_attention_kernel(float *out, uint16_t *out_hi, uint16_t *out_lo, const float *Q,
                            int q_stride, int q_col0, int q_planes, size_t q_plane_stride, const float *rope,
                            const unsigned char *img, int img_tiles, int S, int start_pos, float scale, pa_rows in) {
    static_assert(!HERE || QB == 16, "a residue each for two tiles");
    constexpr int HW = QB / 8, NS = 8 / HW;              /* waves of a residue, residues */
    /* QB 32: a tile of each residue of the even and of the odd steps; QB 16: K and V of a tile of each residue */
    __shared__ __attribute__((aligned(16))) unsigned char pa_a[65536], pa_b[65536];
    __shared__ f32x2 pa_ml[8][64];
    const int kvh = (int)blockIdx.x;
    const int qt = (int)gridDim.y - 1 - (int)blockIdx.y;         /* the blocks with the most keys first */
    const int t = (int)threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int hq = wave % HW, pz = wave / HW;
    const int g = lane >> 5, li = lane & 31;
    const int q0 = qt * QB;
    const int my_q = q0 + li % QB;
    const int last_q = (q0 + QB - 1 < S ? q0 + QB - 1 : S - 1) + start_pos;
    const int ntiles = last_q / 32 + 1;                  /* key tiles 0 .. ntiles-1 are visible */
    const int nsteps = (ntiles + NS - 1) / NS;

    /* the waves of a residue copy KB kilobytes of its tile, from `from` of the tile on, 1 KB per wave and request; for a tile
     * past the last visible one: zeros, which nobody reads */
    constexpr int KB = QB == 32 ? 32 : 16;
    auto fetch = [&](unsigned char *buf, int step, int from) {
        const vt_request rq = vt_tile_request(step * NS + pz, ntiles, PA_TILE_BYTES, from);
        const __amdgpu_buffer_rsrc_t t_rs = __builtin_amdgcn_make_buffer_rsrc((void *)(img + (size_t)kvh * img_tiles * PA_TILE_BYTES), 0, rq.bytes, 0x00020000);
#pragma unroll
        for (int i = 0; i < KB / HW; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(t_rs, (__attribute__((address_space(3))) void *)(buf + pz * KB * 1024 + (i * HW + hq) * 1024), 16,
                                                     (i * HW + hq) * 1024 + lane * 16, rq.soff, 0, 0);
    };
    if constexpr (!HERE) fetch(pa_a, 0, 0);

    /* The queries of the four heads, QB rows x 512 columns: Q as it is, or (rope != NULL) the raw product: the sum of
     * q_planes split-K planes, rotated here (adjacent pairs, voxtral_tts_kernels.c:616-634; the table holds (cos, sin)
     * per pair).  Fetched once per workgroup, whole 128-byte lines per eight lanes, and handed to the waves through LDS as
     * the B operands of K Q^T: lane l holds row l%32, dims 16*ks + 8*(l/32) .. + 8 in slice ks.  (A wave fetching its
     * own operands touches 64 pieces of 16 bytes per request: 10 us of a launch.) */
    bf16x8 qhi[8], qlo[8];
    {
        constexpr int NR = QB / 8, N = 2 * NR;                               /* row groups of 8, quads per thread */
        const int qh = wave >> 1, r = lane >> 3, qd = lane & 7;              /* wave w: columns 64 w .. + 64 */
        const int planes = rope && (kvh * 4 + qh) * VT_HEAD_DIM >= q_col0 ? q_planes : 1;       /* a head whose columns are not cut has one */
        const float *qp = Q + (kvh * 4 + qh) * VT_HEAD_DIM + (wave & 1) * 64 + 4 * qd;
        size_t row[NR];
        f32x4 a[N], c[N];
#pragma unroll
        for (int i = 0; i < NR; i++) row[i] = (size_t)min(q0 + 8 * i + r, S - 1);
#pragma unroll
        for (int i = 0; i < N; i++) a[i] = *reinterpret_cast<const f32x4 *>(qp + row[i % NR] * q_stride + 32 * (i / NR));
        if (rope) {
#pragma unroll
            for (int i = 0; i < N; i++)
                c[i] = *reinterpret_cast<const f32x4 *>(rope + (start_pos + row[i % NR]) * VT_HEAD_DIM + (wave & 1) * 64 + 32 * (i / NR) + 4 * qd);
            for (int p = 1; p < planes; p++) {
                f32x4 b[N];
#pragma unroll
                for (int i = 0; i < N; i++) b[i] = *reinterpret_cast<const f32x4 *>(qp + p * q_plane_stride + row[i % NR] * q_stride + 32 * (i / NR));
#pragma unroll
                for (int i = 0; i < N; i++) {
                    a[i].x = __fadd_rn(a[i].x, b[i].x); a[i].y = __fadd_rn(a[i].y, b[i].y);
                    a[i].z = __fadd_rn(a[i].z, b[i].z); a[i].w = __fadd_rn(a[i].w, b[i].w);
                }
            }
#pragma unroll
            for (int i = 0; i < N; i++) {
                const f32x4 q = a[i], k = c[i];
                a[i] = f32x4{__fsub_rn(__fmul_rn(q.x, k.x), __fmul_rn(q.y, k.y)), __fadd_rn(__fmul_rn(q.x, k.y), __fmul_rn(q.y, k.x)),
                             __fsub_rn(__fmul_rn(q.z, k.z), __fmul_rn(q.w, k.w)), __fadd_rn(__fmul_rn(q.z, k.w), __fmul_rn(q.w, k.z))};
            }
        }
#pragma unroll
        for (int i = 0; i < N; i++) {
            u32x2 h, l;
            vt_split_planes4(a[i].x, a[i].y, a[i].z, a[i].w, h, l);
            /* dims 64 (w%2) + 32 (i/NR) + 4 qd: slice 4 (w%2) + 2 (i/NR) + qd/4, lane group (qd/2)%2, half qd%2 of its 16 bytes */
            const int col = 8 * (i % NR) + r + (QB == 16 ? 16 * (qh & 1) : 0), grp = QB == 16 ? qh >> 1 : qh;
            unsigned char *at = pa_b + grp * 16384 + (4 * (wave & 1) + 2 * (i / NR) + (qd >> 2)) * 1024 + ((qd >> 1 & 1) * 32 + col) * 16 + (qd & 1) * 8;
            *reinterpret_cast<u32x2 *>(at) = h;
            *reinterpret_cast<u32x2 *>(at + PA_PLANE) = l;
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            qhi[ks] = *reinterpret_cast<const bf16x8 *>(pa_b + hq * 16384 + ks * 1024 + lane * 16);
            qlo[ks] = *reinterpret_cast<const bf16x8 *>(pa_b + hq * 16384 + PA_PLANE + ks * 1024 + lane * 16);
        }
    }
    pa_f32x16 o[4];
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
        for (int v = 0; v < 16; v++) o[b][v] = 0.f;
    /* scores in units of log2: exp2 of a difference is the exponential */
    const float to_log2 = __fmul_rn(scale, 1.44269504f);
    float m = -1e30f, lsum = 0.f;
    const int qpos = start_pos + my_q;

    pa_f32x16 s;
    auto scores = [&](const unsigned char *Kt) {         /* S^T = K Q^T */
#pragma unroll
        for (int v = 0; v < 16; v++) s[v] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            const bf16x8 khi = *reinterpret_cast<const bf16x8 *>(Kt + lane * 16 + 1024 * ks);
            const bf16x8 klo = *reinterpret_cast<const bf16x8 *>(Kt + lane * 16 + PA_PLANE + 1024 * ks);
            s = pa_mfma(klo, qhi[ks], s);
            s = pa_mfma(khi, qlo[ks], s);
            s = pa_mfma(khi, qhi[ks], s);
        }
    };
    auto weigh = [&](const unsigned char *Vt, int tile) {
        /* online softmax for this lane's query row; element v is key 8*(v/4) + 4*g + v%4.  A score that is no number counts
         * as masked. */
        float mx = -1e30f;
#pragma unroll
        for (int v = 0; v < 16; v++) s[v] = fmaxf(__fmul_rn(s[v], to_log2), -3e38f);
        if (tile * 32 + 31 > start_pos + q0) {           /* the tile reaches beyond the first query */
#pragma unroll
            for (int v = 0; v < 16; v++) s[v] = tile * 32 + 8 * (v >> 2) + 4 * g + (v & 3) <= qpos ? s[v] : -3e38f;
        }
#pragma unroll
        for (int v = 0; v < 16; v++) mx = fmaxf(mx, s[v]);
        mx = pa_max_halves(mx);
        /* (Letting the maximum lag by up to 2^8, so that fewer tiles rescale the sums, makes the results' error against 64 bits
         * 2.5 % larger: a probability of exactly 1 has no rounding error, and a row's largest one no longer is.) */
        if (__any(mx > m)) {
            const float mn = fmaxf(m, mx), corr = __builtin_amdgcn_exp2f(m - mn);
            m = mn;
            lsum *= corr;
#pragma unroll
            for (int b = 0; b < 4; b++) o[b] = o[b] * corr;
        }
#pragma unroll
        for (int v = 0; v < 16; v++) s[v] = __builtin_amdgcn_exp2f(s[v] - m);
        lsum += (((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]))) +
                (((s[8] + s[9]) + (s[10] + s[11])) + ((s[12] + s[13]) + (s[14] + s[15])));
        /* O^T += V^T P^T */
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
            bf16x8 phi, plo;
            pa_planes8(f32x4{s[8 * kt], s[8 * kt + 1], s[8 * kt + 2], s[8 * kt + 3]}, f32x4{s[8 * kt + 4], s[8 * kt + 5], s[8 * kt + 6], s[8 * kt + 7]}, phi, plo);
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const bf16x8 vhi = *reinterpret_cast<const bf16x8 *>(Vt + lane * 16 + (b * 2 + kt) * 1024);
                const bf16x8 vlo = *reinterpret_cast<const bf16x8 *>(Vt + lane * 16 + PA_PLANE + (b * 2 + kt) * 1024);
                o[b] = pa_mfma(vlo, phi, o[b]);
                o[b] = pa_mfma(vhi, plo, o[b]);
                o[b] = pa_mfma(vhi, phi, o[b]);
            }
        }
    };
    /* every wave waits for what it asked for, then for all the others: they have then also read what is written next */
#define PA_LANDED() do { __builtin_amdgcn_s_waitcnt(0x0f70); __syncthreads(); } while (0)     /* vmcnt(0) */
    PA_LANDED();
    if constexpr (HERE) {
        const int tile = wave >> 2;                      /* half of the waves for each */
        if (tile < ntiles) pa_make_tile(pa_a + tile * 2 * PA_PLANE, pa_b + tile * 2 * PA_PLANE, in, kvh, tile, t & 255, start_pos + q0, QB);
        __syncthreads();
        if (pz < ntiles) { scores(pa_a + pz * 2 * PA_PLANE); weigh(pa_b + pz * 2 * PA_PLANE, pz); }
        __syncthreads();
    } else if constexpr (QB == 32) {
        /* the next tile arrives while this one is worked on: one barrier per tile */
        const unsigned char *even = pa_a + pz * PA_TILE_BYTES, *odd = pa_b + pz * PA_TILE_BYTES;
        for (int step = 0; step < nsteps; step += 2) {
            fetch(pa_b, step + 1, 0);
            if (step * NS + pz < ntiles) { scores(even); weigh(even + 2 * PA_PLANE, step * NS + pz); }
            PA_LANDED();
            fetch(pa_a, step + 2, 0);
            if ((step + 1) * NS + pz < ntiles) { scores(odd); weigh(odd + 2 * PA_PLANE, (step + 1) * NS + pz); }
            PA_LANDED();
        }
    } else {
        /* V of a tile arrives under its scores, K of the next one under the rest */
        for (int step = 0; step < nsteps; step++) {
            const int tile = step * NS + pz;
            fetch(pa_b, step, 2 * PA_PLANE);
            if (tile < ntiles) scores(pa_a + pz * 2 * PA_PLANE);
            PA_LANDED();
            fetch(pa_a, step + 1, 0);
            if (tile < ntiles) weigh(pa_b + pz * 2 * PA_PLANE, tile);
            PA_LANDED();
        }
    }
#undef PA_LANDED

    /* Merge: of the NS waves with the same rows, wave pz finishes 128 / NS dims.  Each parks its sums, 16 quads of
     * dims (behind the last barrier nobody reads tiles); they are added in the order of the residues. */
    constexpr int NB = 4 / NS;                           /* dim blocks that a wave finishes */
    auto park = [&](int w, int b, int v) {
        return reinterpret_cast<f32x4 *>((w < 4 ? pa_a : pa_b) + (w & 3) * 16384 + (4 * b + v) * 1024 + lane * 16);
    };
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) *park(wave, b, v) = f32x4{o[b][4 * v], o[b][4 * v + 1], o[b][4 * v + 2], o[b][4 * v + 3]};
    pa_ml[wave][lane] = f32x2{m, lsum};
    __syncthreads();
    float c[NS], inv;
    {
        f32x2 ml[NS];
#pragma unroll
        for (int r = 0; r < NS; r++) ml[r] = pa_ml[r * HW + hq][lane];
        float mn = ml[0].x, L = 0.f;
#pragma unroll
        for (int r = 1; r < NS; r++) mn = fmaxf(mn, ml[r].x);
#pragma unroll
        for (int r = 0; r < NS; r++) {
            c[r] = __builtin_amdgcn_exp2f(ml[r].x - mn);
            L = fmaf(ml[r].y, c[r], L);
        }
        L += __shfl_xor(L, 32);
        inv = L > 0.f ? __fdiv_rn(1.0f, L) : 0.f;
    }
    f32x4 res[NB][4];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            f32x4 x = *park(hq, NB * pz + b, v) * c[0];
#pragma unroll
            for (int r = 1; r < NS; r++) {
                const f32x4 y = *park(r * HW + hq, NB * pz + b, v);
                x = f32x4{fmaf(y.x, c[r], x.x), fmaf(y.y, c[r], x.y), fmaf(y.z, c[r], x.z), fmaf(y.w, c[r], x.w)};
            }
            res[b][v] = x * inv;
        }
    const int hd = QB == 16 ? 2 * hq + (li >> 4) : hq;   /* this lane's head of the four */
    if (out && my_q < S) {
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                *reinterpret_cast<f32x4 *>(out + (size_t)my_q * VT_Q_DIM + (kvh * 4 + hd) * VT_HEAD_DIM + 32 * (NB * pz + b) + 8 * v + 4 * g) = res[b][v];
    }
    if (!out_hi) return;
    __syncthreads();
    /* the planes leave through LDS, as whole lines: rows of 256 bytes, [query][head], 16-byte piece i at place i ^ query % 16 */
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            u32x2 h, l;
            vt_split_planes4(res[b][v].x, res[b][v].y, res[b][v].z, res[b][v].w, h, l);
            const int at = ((li % QB) * 4 + hd) * 256 + (((4 * (NB * pz + b) + v) ^ (li & 15)) * 16) + 8 * g;
            *reinterpret_cast<u32x2 *>(pa_a + at) = h;
            *reinterpret_cast<u32x2 *>(pa_b + at) = l;
        }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < QB / 8; i++) {                   /* a wave stores one query's four heads */
        const int r = 8 * i + wave;
        if (q0 + r < S) {
            const size_t at = (size_t)(q0 + r) * VT_Q_DIM + kvh * 4 * VT_HEAD_DIM + 8 * lane;
            const int from = (r * 4 + (lane >> 4)) * 256 + (((lane & 15) ^ (r & 15)) * 16);
            *reinterpret_cast<u32x4 *>(out_hi + at) = *reinterpret_cast<const u32x4 *>(pa_a + from);
            *reinterpret_cast<u32x4 *>(out_lo + at) = *reinterpret_cast<const u32x4 *>(pa_b + from);
        }
    }
}

/* Tiles of 32 keys that cover `rows` cache rows, and the tile images of one layer's K and V (a buffer of the
 * library's own that grows with the longest cache seen) */
static int pa_tiles(int rows) { return (rows + 31) / 32; }
unsigned char *vt_pa_image(int rows) {
    const size_t bytes = (size_t)VT_KV_HEADS * pa_tiles(rows) * PA_TILE_BYTES;
    if (bytes > g_vt.kv_img_bytes) {
        if (g_vt.d_kv_img) {
            (void)hipStreamSynchronize(g_vt.stream);
            (void)hipFree(g_vt.d_kv_img);
        }
        g_vt.d_kv_img = vt_dev_alloc(bytes);
        g_vt.kv_img_bytes = g_vt.d_kv_img ? bytes : 0;
    }
    return (unsigned char *)g_vt.d_kv_img;
}

/* d_qkv != NULL: rows start_pos .. start_pos + S - 1 are taken from the q|k|v product (summed, k rotated)
 * and appended to the cache d_K / d_V; otherwise all start_pos + S rows are in the cache already */
void vt_pa_launch_image(unsigned char *d_img, const float *d_qkv, int col0, int planes, size_t plane_stride, float *d_K,
                        float *d_V, int S, int start_pos) {
    const int rows = start_pos + S;
    hipLaunchKernelGGL(vt_kv_image_kernel, dim3(pa_tiles(rows), VT_KV_HEADS), dim3(256), 0, g_vt.stream, d_img, pa_tiles(rows),
                       pa_rows{d_qkv, col0, planes, plane_stride, d_K, d_V, g_vt.d_rope, d_qkv ? start_pos : rows, rows});
}

/* Q rows are q_stride floats apart; out / (out_hi, out_lo) are [S,4096], each optional.  d_rope != NULL: d_Q
 * holds q_planes split-K planes (q_plane_stride floats apart; heads below column q_col0 have one) of the raw q product, to be summed and
 * rotated with the table rows start_pos .. by the kernel.  d_img: the tile images of the start_pos + S
 * cache rows (vt_kv_image_kernel). */
void vt_launch_prefill_attention_raw(float *d_out, uint16_t *d_hi, uint16_t *d_lo, const float *d_Q,
                                     int q_stride, int q_col0, int q_planes, size_t q_plane_stride, const float *d_rope,
                                     const unsigned char *d_img, int S, int start_pos, float scale) {
    const bool lng = S > PA_SHORT_ROWS;
    const int qb = lng ? PA_LONG_QT : PA_SHORT_QT;
    const dim3 grid(VT_KV_HEADS, (S + qb - 1) / qb);
#define CALL(QB) hipLaunchKernelGGL((vt_prefill_attention_kernel<QB, false>), grid, dim3(512), 0, g_vt.stream, d_out, d_hi, d_lo, d_Q, q_stride, q_col0, \
                                    q_planes, q_plane_stride, d_rope, d_img, pa_tiles(start_pos + S), S, start_pos, scale, pa_rows{})
    if (lng) CALL(PA_LONG_QT);
    else CALL(PA_SHORT_QT);
#undef CALL
}

/* A layer's attention on the raw q|k|v product and the cache rows in front of it, rows start_pos .. + S - 1 appended; with up to
 * PA_HERE_ROWS rows in all as one launch */
static void pa_launch_layer(uint16_t *d_hi, uint16_t *d_lo, const float *d_qkv, int col0, int planes, size_t plane_stride, float *d_K, float *d_V,
                            unsigned char *d_img, int S, int start_pos) {
    if (start_pos + S <= PA_HERE_ROWS) {
        hipLaunchKernelGGL((vt_prefill_attention_kernel<16, true>), dim3(VT_KV_HEADS, (S + 15) / 16), dim3(512), 0, g_vt.stream, (float *)NULL, d_hi, d_lo, d_qkv, VT_QKV_DIM,
                           col0, planes, plane_stride, g_vt.d_rope, (const unsigned char *)NULL, 0, S, start_pos, VT_ATT_SCALE,
                           pa_rows{d_qkv, col0, planes, plane_stride, d_K, d_V, g_vt.d_rope, start_pos, start_pos + S});
        return;
    }
    vt_pa_launch_image(d_img, d_qkv, col0, planes, plane_stride, d_K, d_V, S, start_pos);
    vt_launch_prefill_attention_raw(NULL, d_hi, d_lo, d_qkv, VT_QKV_DIM, col0, planes, plane_stride, g_vt.d_rope, d_img, S, start_pos, VT_ATT_SCALE);
}

void vt_launch_prefill_attention(float *d_out, uint16_t *d_hi, uint16_t *d_lo, const float *d_Q,
                                 int q_stride, const float *d_K, const float *d_V, int S, int start_pos,
                                 float scale) {
    unsigned char *img = vt_pa_image(start_pos + S);
    if (!img) return;
    /* (the image kernel only reads a cache that is complete) */
    vt_pa_launch_image(img, NULL, 0, 0, 0, const_cast<float *>(d_K), const_cast<float *>(d_V), S, start_pos);
    vt_launch_prefill_attention_raw(d_out, d_hi, d_lo, d_Q, q_stride, 0, 1, 0, NULL, img, S, start_pos, scale);
}

/* ---- backbone prefill ------------------------------------------------------------ */

/* The input rows -> x and the planes of their RMSNorm.  Pageable rows of a longer prompt go piece by piece through pinned memory that the
 * kernel reads itself, a launch per piece, while the next piece is copied: a prefill of 226 / 512 / 1531 rows takes 80 / 210 / 930 us
 * longer than one of rows on the device; 140 / 290 / 1000 with the runtime's own staging in front of the first kernel, which up to PF_STAGED_ROWS
 * rows is as fast (30 us at 37).  What is left is the copy, 20 GB/s from memory that is in no cache; three more threads copying
 * made it 410 us at 800 rows and 440 at 1000, as long, and 570 to 690 at 1531: not kept. */
#define PF_STAGED_ROWS 96
#define PF_PIECE_ROWS 64
static int pf_take_rows(float *x, const float *rows, int n, uint16_t *hi, uint16_t *lo) {
    const float *norm = g_vt.h_layers[0].attn_norm;
    if (n <= PF_STAGED_ROWS || n > VT_PIN_ROWS || !g_vt.h_rows || !vt_pageable(rows)) {
        VT_TRY(hipMemcpyAsync(x, rows, sizeof(float) * VT_DIM * n, hipMemcpyDefault, g_vt.stream));
        vt_launch_residual_norm_split(x, x, NULL, 0, 0, 0, norm, hi, lo, n);
        return 0;
    }
    for (int i = 0; i < n; i += PF_PIECE_ROWS) {
        const int m = n - i < PF_PIECE_ROWS ? n - i : PF_PIECE_ROWS;
        const size_t at = (size_t)i * VT_DIM;
        memcpy(g_vt.h_rows + at, rows + at, sizeof(float) * VT_DIM * m);
        vt_launch_residual_norm_split(x + at, g_vt.h_rows + at, NULL, 0, 0, 0, norm, hi + at, lo + at, m);
    }
    return 0;
}

extern "C" void tts_hip_llm_prefill_out(const float *embeds, int seq_len, int start_pos, float *out_x) {
    if (!g_vt.initialized || g_vt.n_dec_layers < 1) { vt_set_error("tts_hip_llm_prefill: no weights uploaded"); return; }
    if (seq_len < 1 || start_pos < 0 || start_pos + seq_len > g_vt.kv_max) {
        vt_set_error("tts_hip_llm_prefill: rows [%d, %d) outside the KV cache (max %d)", start_pos,
                     start_pos + seq_len, g_vt.kv_max);
        return;
    }
    const size_t S = (size_t)seq_len;
    hipStream_t st = g_vt.stream;
    bool frag = true;                 /* every layer has its fragment-order copy (otherwise: the 128 x 128 kernel on row-major weights) */
    for (int l = 0; l < g_vt.n_dec_layers; l++) {
        const vt_layer_frag *F = &g_vt.h_frag[l];
        frag = frag && F->wqkv && F->wo && F->w13 && F->w2;
    }
    const int m_tiles = (seq_len + 127) / 128;
    vt_gemm_plan pq, po, pg, pd;      /* q|k|v, output, gate|up, down */
    vt_gemm_plan pkv = {};            /* k|v alone: its columns, with the last 64 of q where strips of 96 take them */
    const int kv0 = vt_gemm_rows_ok(seq_len, VT_QKV_DIM, VT_DIM) ? VT_Q_DIM - 64 : VT_Q_DIM;
    if (frag) {
        pkv = vt_gemm_frag_plan(seq_len, VT_QKV_DIM - kv0, VT_DIM, 0);
        pq = vt_gemm_frag_plan(seq_len, VT_QKV_DIM, VT_DIM, 0);
        po = vt_gemm_frag_plan(seq_len, VT_DIM, VT_Q_DIM, 0);
        pg = vt_gemm_frag_plan(seq_len, 2 * VT_FFN, VT_DIM, 1);
        pd = vt_gemm_frag_plan(seq_len, VT_DIM, VT_FFN, 0);
    } else {                          /* cuts that divide K */
        pq = vt_gemm_plan{0, 0, 0, m_tiles >= 3 ? 2 : 4};
        po = pd = vt_gemm_plan{0, 0, 0, m_tiles >= 3 ? 4 : 8};
        /* 4 M tiles x 144 N tiles are 576 workgroups for 512 slots: the last 16 N tiles get their K cut in 4 */
        pg = vt_gemm_plan{0, 0, 2 * VT_FFN - (m_tiles == 4 ? 16 * 128 : 0), 4};
    }
    /* work area: x | q|k|v planes (without fragment copies also the gate|up product) | planes of the output and
     * down products | planes of the cut gate|up columns | bf16 planes: products' input, SiLU(gate) * up */
    const int gu_tail = 2 * VT_FFN - pg.col0;
    const size_t w_qkv = (size_t)(pq.cuts > pkv.cuts ? pq.cuts : pkv.cuts) * VT_QKV_DIM, w_gu = frag ? 0 : 2 * VT_FFN;
    const size_t n_x = S * VT_DIM, n_wide = S * (w_qkv > w_gu ? w_qkv : w_gu), n_part = S * VT_DIM * (po.cuts > pd.cuts ? po.cuts : pd.cuts);
    const size_t n_tail = S * gu_tail * pg.cuts, n_plane = S * VT_FFN;      /* bf16 elements per plane */
    const size_t bytes = sizeof(float) * (n_x + n_wide + n_part + n_tail) + 4 * sizeof(uint16_t) * n_plane;
    float *x = (float *)vt_scratch(bytes);
    unsigned char *img = vt_pa_image(start_pos + seq_len);
    if (!x || !img) return;
    float *wide = x + n_x, *part = wide + n_wide, *tail = part + n_part;
    uint16_t *hi = (uint16_t *)(tail + n_tail), *lo = hi + n_plane, *h_hi = lo + n_plane, *h_lo = h_hi + n_plane;
    const size_t ps = S * VT_DIM;

    if (pf_take_rows(x, embeds, seq_len, hi, lo)) return;
    for (int l = 0; l < g_vt.n_dec_layers; l++) {
        const vt_layer_dev *L = &g_vt.h_layers[l];
        float *kc = g_hip.kv_cache_k_gpu + (size_t)l * g_vt.kv_max * VT_KV_DIM;
        float *vc = g_hip.kv_cache_v_gpu + (size_t)l * g_vt.kv_max * VT_KV_DIM;
        const vt_layer_frag *F = &g_vt.h_frag[l];
        if (l + 1 == g_vt.n_dec_layers && !out_x && frag) {
            /* the caller wants the cache only: behind the last layer's k and v nothing of it is read, and q is not
             * either.  25.08 of 26 layers' products remain: prefills of
             * 37, 226, 512, 1531 rows take 0.968, 0.950, 0.974, 0.944 of their time. */
            vt_launch_gemm_frag(wide + kv0, VT_QKV_DIM, S * VT_QKV_DIM, hi, lo, F->wqkv + (size_t)kv0 * VT_DIM,
                                seq_len, VT_QKV_DIM - kv0, VT_DIM, pkv);
            vt_pa_launch_image(img, wide, kv0 + pkv.col0, pkv.cuts, S * VT_QKV_DIM, kc, vc, seq_len, start_pos);
            break;
        }
        if (frag) vt_launch_gemm_frag(wide, VT_QKV_DIM, S * VT_QKV_DIM, hi, lo, F->wqkv, seq_len, VT_QKV_DIM, VT_DIM, pq);
        else vt_launch_gemm(wide, hi, lo, L->wqkv, seq_len, VT_QKV_DIM, VT_DIM, pq.cuts);
        /* k (rotated) and v into the cache and, with the earlier rows, into the attention's tile images; the
         * attention takes q from the product's planes itself */
        pa_launch_layer(hi, lo, wide, pq.col0, pq.cuts, S * VT_QKV_DIM, kc, vc, img, seq_len, start_pos);
        if (frag) vt_launch_gemm_frag(part, VT_DIM, ps, hi, lo, F->wo, seq_len, VT_DIM, VT_Q_DIM, po);
        else vt_launch_gemm(part, hi, lo, L->wo, seq_len, VT_DIM, VT_Q_DIM, po.cuts);
        vt_launch_residual_norm_split(x, x, part, po.col0, po.cuts, ps, L->ffn_norm, hi, lo, seq_len);
        if (frag) {
            vt_launch_gemm_frag_swiglu(h_hi, h_lo, VT_FFN, tail, hi, lo, F->w13, seq_len, 2 * VT_FFN, VT_DIM, pg);
        } else {
            vt_launch_gemm_ex(wide, 2 * VT_FFN, 0, hi, lo, L->w13, seq_len, pg.col0, VT_DIM, 1);
            if (gu_tail)
                vt_launch_gemm_ex(tail, gu_tail, S * gu_tail, hi, lo, L->w13 + (size_t)pg.col0 * VT_DIM, seq_len, gu_tail, VT_DIM, pg.cuts);
            vt_launch_swiglu_split(h_hi, h_lo, wide, S * VT_FFN, pg.col0, tail, gu_tail ? pg.cuts : 0, S * gu_tail);
        }
        if (frag) vt_launch_gemm_frag(part, VT_DIM, ps, h_hi, h_lo, F->w2, seq_len, VT_DIM, VT_FFN, pd);
        else vt_launch_gemm(part, h_hi, h_lo, L->w2, seq_len, VT_DIM, VT_FFN, pd.cuts);
        const float *next_norm = l + 1 < g_vt.n_dec_layers ? g_vt.h_layers[l + 1].attn_norm : NULL;
        vt_launch_residual_norm_split(x, x, part, pd.col0, pd.cuts, ps, next_norm, hi, lo, seq_len);
    }
    const hipError_t launched = hipGetLastError();
    VT_TRYV(hipStreamSynchronize(st));    /* in any case: the pinned rows are free for the next call */
    VT_TRYV(launched);
    if (out_x) VT_TRYV(hipMemcpy(out_x, x, sizeof(float) * n_x, hipMemcpyDefault));
}

extern "C" void tts_hip_llm_prefill(const float *embeds, int seq_len, int start_pos) {
    tts_hip_llm_prefill_out(embeds, seq_len, start_pos, NULL);
}

/*
 * vt_codec.hip - audio codec decoder on the device: frames of 37 codes -> 24 kHz waveform
 * (tts_codec_decode, voxtral_tts_codec.c:389-503; one transformer layer :306-383; the
 * convolutions voxtral_tts_kernels.c:217-327; ALiBi sliding-window attention :527-596).
 *
 * Layout: activations are token-major [T, C] from the first kernel to the last, so the
 * reference's channel-first transposes around every convolution disappear and the last
 * product writes the waveform ([T, 240] row-major is the sample order).  Weights are re-laid
 * once at upload:
 *   - q|k|v and gate|up are stacked into one [3072, 1024] and one [8192, 1024] matrix;
 *   - the input convolution (taps 3, 292 channels) becomes a product over the shifted copies of
 *     the embedding: W'[oc][k * 292 + ic] = w[oc][ic][k], K padded with zeros;
 *   - the others multiply every row with all taps, and the kernel that reads the result adds the
 *     taps' columns of neighbouring rows.  Transposed (taps 4, stride 2): out[2j+p][oc] =
 *     sum_ic x[j][ic] w[ic][oc][p] + x[j-1][ic] w[ic][oc][p+2], so W'[q * 2048 + p * 1024 + oc][ic]
 *     = w[ic][oc][p + 2q].  Output (taps 7): W'[k * 256 + oc][ic] = w[oc][ic][k].  The sums are those
 *     of a product over shifted copies of the rows, in two and seven pieces, without four launches that
 *     write the copies (100 us of a 1003-frame decode); us per decode of 21 / 212 / 1003 frames:
 *     731 / 1595 / 4983 -> 712 / 1558 / 4890 (584 / 1359 / 4212 now, with the products and row kernels as they are).
 * Every product runs on the fp16 matrix cores with both operands as two fp16 planes
 * (vt_codec_gemm.hip); whoever produces a product's input leaves it as planes with one exponent
 * per row.  Where a launch would not fill the chip K is cut, and the kernel that reads the
 * result adds the partial planes in a fixed order, next to bias / layer scale / residual and
 * the next RMSNorm.
 */
#include "vt_state.h"
#include "vt_gemm.h"

#include <stdlib.h>
#include <string.h>

#define CD_DIM 1024
#define CD_HID 4096
#define CD_HEADS 8
#define CD_HEAD_DIM 128
#define CD_EPS 1e-2f
#define CD_QK_EPS 1e-6f
#define CD_EMBED 292
#define CD_SEM_DIM 256
#define CD_SEM_SIZE 8192
#define CD_PATCH 240
#define CD_LAYERS 8
#define CD_IN_TAPS 3
#define CD_OUT_TAPS 7
#define CD_IN_K 896           /* 3 * 292 = 876 padded to a multiple of 64 */
#define CD_OUT_PITCH 256      /* a tap's 240 columns */
#define CD_OUT_N (CD_OUT_TAPS * CD_OUT_PITCH)
#define CD_UP_N (4 * CD_DIM)  /* (tap pair q, phase p, channel) */

/* ---- row kernels ------------------------------------------------------------------------- */

/* block-wide sum and maximum over 256 threads (4 waves), the same value in every thread; red: 4 floats for this one reduction */
__device__ __forceinline__ float cd_block_sum(float v, float *red) {
    v = vt_wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}
__device__ __forceinline__ float cd_block_max(float v, float *red) {
    v = vt_wave_max(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}
__device__ __forceinline__ float cd_max4(const f32x4 &v) { return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))); }

/* A product's input: two fp16 planes [rows, K] of the rows times 2^exp, an exponent per row */
struct cd_planes { uint16_t *hi, *lo; int *exp; };

__device__ __forceinline__ void cd_put4(const cd_planes &p, size_t at, const f32x4 &v, int e) {
    u32x2 h, l;
    vt_split_f16x4(vt_ldexp4(v, e), h, l);
    *(u32x2 *)(p.hi + at) = h;
    *(u32x2 *)(p.lo + at) = l;
}

/* A product's result as vt_launch_codec_gemm leaves it: the columns below col0, [rows, col0], and behind them `cuts`
 * partial planes of the others, [rows, n - col0] */
struct cd_product { const float *p; int rows, n, col0, cuts; };

/* Four columns of a row: the whole column and each plane of a cut one, which bring zeros for the columns that they do not have (and
 * planes that do not exist, for all).  The kernels ask for all that they need and put cd_asked() behind it (one after the other the
 * planes cost a memory latency each); total() adds the planes in order. */
template <int C>
struct cd_quads {
    f32x4 whole, q[C];
    __device__ __forceinline__ void ask(const cd_product &r, int row, int col) {
        const int cut = r.n - r.col0;
        whole = vt_buffer_ld4(vt_buffer(r.p + (size_t)row * r.col0, r.col0 * 4), 4 * col);
        const float *pc = r.p + (size_t)r.rows * r.col0 + (size_t)row * cut;
#pragma unroll
        for (int s = 0; s < C; s++) q[s] = vt_buffer_ld4(vt_buffer(pc + (size_t)(s < r.cuts ? s : 0) * ((size_t)r.rows * cut), s < r.cuts ? cut * 4 : 0), 4 * (col - r.col0));
    }
    __device__ __forceinline__ f32x4 total() const {
        f32x4 v = whole;
#pragma unroll
        for (int s = 0; s < C; s++) v += q[s];
        return v;
    }
};
__device__ __forceinline__ void cd_asked() { __builtin_amdgcn_sched_barrier(0); }

/* One row of 1024: val = the product's result (+ bias) (* scale) (+ residual).  With a norm weight val -> x_out and
 * val * rsqrt(mean(val^2) + eps) * norm_w (tts_rms_norm, voxtral_tts_kernels.c:333-349) as planes; without one the
 * rows go into a convolution next, val itself as planes.  UP: rows of the upsampling product, row 2 j + p is the sum of
 * phase p's columns of row j and, for the other tap, of row j - 1. */
template <int C, bool UP>
__global__ void __launch_bounds__(256)
vt_codec_row_kernel(float *x_out, cd_planes xn, const float *x_in, cd_product in, const float *__restrict__ bias,
                    const float *__restrict__ scale, const float *__restrict__ norm_w, float eps) {
    __shared__ float red[2][4];
    const int row = blockIdx.x, c = threadIdx.x * 4;
    const size_t at = (size_t)row * CD_DIM + c;
    f32x4 r = {0.f, 0.f, 0.f, 0.f};
    if (x_in) r = *(const f32x4 *)(x_in + at);
    f32x4 v;
    if (UP) {
        const int j = row >> 1, col = (row & 1) * CD_DIM + c;
        cd_quads<C> q, before;
        q.ask(in, j, col);
        before.ask(in, max(j - 1, 0), 2 * CD_DIM + col);
        cd_asked();
        v = q.total();
        if (j > 0) v += before.total();
    } else {
        cd_quads<C> q;
        q.ask(in, row, c);
        cd_asked();
        v = q.total();
    }
    if (bias) v += *(const f32x4 *)(bias + c);
    if (scale) v *= *(const f32x4 *)(scale + c);
    v += r;
    if (norm_w) {
        *(f32x4 *)(x_out + at) = v;
        const float ss = cd_block_sum(v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w, red[0]);
        const float inv = 1.0f / sqrtf(ss / (float)CD_DIM + eps);
        v = v * inv * *(const f32x4 *)(norm_w + c);
    }
    const int e = vt_f16_exp(cd_block_max(cd_max4(v), red[1]));
    cd_put4(xn, at, v, e);
    if (threadIdx.x == 0) xn.exp[row] = e;
}

/* q|k|v [T, 3072] summed, with the RMSNorm over the whole 1024-wide q row and k row (tts_qk_norm,
 * voxtral_tts_kernels.c:351-355, eps 1e-6) when the layer has those weights.  PARTS 2: q and k only, where v has nothing to be added and
 * the attention reads it where the product left it (cd_v_rows): the kernel is bound by memory, and a decode of 1003 frames takes 4345 us
 * instead of 4377.  Below CD_ATT_SPLIT_BELOW rows it gained nothing (21 frames 596 us, 594 without). */
template <int C, int PARTS>
__global__ void __launch_bounds__(256)
vt_codec_qkv_kernel(float *__restrict__ qkv, cd_product in, const float *__restrict__ q_norm, const float *__restrict__ k_norm) {
    __shared__ float red[2][4];
    const int row = blockIdx.x, c = threadIdx.x * 4;
    const size_t at = (size_t)row * (3 * CD_DIM) + c;
    f32x4 v[PARTS];
    cd_quads<C> q[PARTS];
#pragma unroll
    for (int part = 0; part < PARTS; part++) q[part].ask(in, row, part * CD_DIM + c);
    cd_asked();
#pragma unroll
    for (int part = 0; part < PARTS; part++) v[part] = q[part].total();
#pragma unroll
    for (int part = 0; part < PARTS; part++) {
        const float *nw = part == 0 ? q_norm : part == 1 ? k_norm : nullptr;
        if (nw) {
            const float ss = cd_block_sum(v[part].x * v[part].x + v[part].y * v[part].y + v[part].z * v[part].z + v[part].w * v[part].w, red[part]);
            const float inv = 1.0f / sqrtf(ss / (float)CD_DIM + CD_QK_EPS);
            v[part] = v[part] * inv * *(const f32x4 *)(nw + c);
        }
        *(f32x4 *)(qkv + at + part * CD_DIM) = v[part];
    }
}

/* The v rows of the attention for many tokens, `stride` floats apart */
struct cd_v_rows { const float *p; int stride; };
/* p NULL: some of the v columns of this q|k|v product are in several planes, or whole and cut ones meet among them */
static cd_v_rows cd_v_in_place(const cd_product &in) {
    if (in.col0 == in.n) return cd_v_rows{in.p + 2 * CD_DIM, in.n};
    if (in.cuts > 1 || in.col0 > 2 * CD_DIM) return cd_v_rows{NULL, 0};
    return cd_v_rows{in.p + (size_t)in.rows * in.col0 + (2 * CD_DIM - in.col0), in.n - in.col0};
}

/* gate|up [T, 8192] -> h = silu(gate) * up [T, 4096] (tts_silu, tts_mul_inplace) as planes; one workgroup per row */
template <int C>
__global__ void __launch_bounds__(256)
vt_codec_swiglu_kernel(cd_planes h, cd_product gu) {
    __shared__ float red[4];
    const int row = blockIdx.x;
    f32x4 v[CD_HID / 1024];
    float m = 0.f;
    constexpr int AT_ONCE = C > 4 ? 2 : CD_HID / 1024;        /* registers */
#pragma unroll
    for (int j0 = 0; j0 < CD_HID / 1024; j0 += AT_ONCE) {
        cd_quads<C> g[AT_ONCE], u[AT_ONCE];
#pragma unroll
        for (int j = 0; j < AT_ONCE; j++) {
            g[j].ask(gu, row, 4 * ((int)threadIdx.x + 256 * (j0 + j)));
            u[j].ask(gu, row, CD_HID + 4 * ((int)threadIdx.x + 256 * (j0 + j)));
        }
        cd_asked();
#pragma unroll
        for (int j = 0; j < AT_ONCE; j++) {
            v[j0 + j] = vt_silu_mul4(g[j].total(), u[j].total());
            m = fmaxf(m, cd_max4(v[j0 + j]));
        }
    }
    const int e = vt_f16_exp(cd_block_max(m, red));
#pragma unroll
    for (int j = 0; j < CD_HID / 1024; j++) cd_put4(h, (size_t)row * CD_HID + 4 * ((int)threadIdx.x + 256 * j), v[j], e);
    if (threadIdx.x == 0) h.exp[row] = e;
}

/* ALiBi causal sliding-window attention, the online softmax of a query over the at most `window` keys in ascending
 * order (voxtral_tts_kernels.c:527-596); the result as planes.  A wave works for one head, eight lanes hold a row's 128
 * dims (dims 32 e + 4 sub + 0..3 of lane sub), so that a score is 16 products per lane and three lane steps.  With a
 * wave per (token, head), two dims per lane, it took six shuffles per key and waited for each key's rows in turn. */
struct cd_head_row { f32x4 v[4]; };

__device__ __forceinline__ cd_head_row cd_load_row(const float *p) {
    cd_head_row r;
#pragma unroll
    for (int e = 0; e < 4; e++) r.v[e] = *(const f32x4 *)(p + 32 * e);
    return r;
}

/* q . k over the eight lanes */
__device__ __forceinline__ float cd_row_dot(const cd_head_row &q, const cd_head_row &k) {
    float p = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int i = 0; i < 4; i++) p = fmaf(q.v[e][i], k.v[e][i], p);
    p += vt_dpp<0xB1>(p);                         /* lanes ^1 */
    p += vt_dpp<0x4E>(p);                         /* lanes ^2 */
    return p + vt_dpp<0x141>(p);                  /* the other quad of the eight */
}

struct cd_softmax {
    float mx = -1e30f, se = 0.f;
    cd_head_row o = {};
    __device__ __forceinline__ void add(float sc, const cd_head_row &v) {
        const float d = sc - mx, ex = expf(-fabsf(d)), c = d > 0.f ? ex : 1.0f, w = d > 0.f ? 1.0f : ex;
        mx = d > 0.f ? sc : mx;
        se = fmaf(se, c, w);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < 4; i++) o.v[e][i] = fmaf(v.v[e][i], w, o.v[e][i] * c);
    }
};

/* Many tokens: one workgroup for 8 NT of them, wave h for head h, eight lanes for NT neighbouring tokens, which share
 * all but NT of their keys: a key's rows are read once per NT tokens, and that reading (L2: what a CU's waves have in
 * flight is twice its L1) bounds the kernel.  The rows of the next key are requested in front of the work on this one;
 * with its value rows requested late instead (118 registers at NT = 2, two workgroups to a CU) the eight launches of
 * 1003 frames took 258 us instead of 196.  Tokens past the last one work as the last one and store nothing. */
/* Fewer rows than this: the kernel below.  Measured, NT = 2 / the one below: 848 rows, window 8, 11.3 / 11.3
 * us; 1003 rows, window 2, 8 / 8.5; 1696 rows, window 16, 17.5 / 23.4; 168 rows, window 16, 16 / 5.5. */
#define CD_ATT_SPLIT_BELOW 1024
/* NT = 4 has one workgroup to a CU (233 registers) that takes 1.3 .. 1.8 times as long as two tokens' does, so it pays
 * from where NT = 2 has more than one to a CU on (4097 rows).  Measured, us, NT = 2 / 4: window 8: 2800 rows 14.8 / 18.8, 4000 20 / 23,
 * 4120 27.0 / 23.0, 4800 28.2 / 24.5, 5600 34.2 / 27.3, 8240 46.6 / 47.2, 11200 56.7 / 55.8; window 16: 4160 41.5 / 31.6, 5600
 * 48.5 / 39.1, 8024 67 / 56, 8240 70.0 / 69.0, 8800 70.0 / 76.3, 9600 73.4 / 78.1, 10400 76.3 / 81.5, 11200 82.5 / 83.3, 16480 140.6 / 132.7,
 * 22400 191.7 / 164.7; window 4: 4120 20.9 / 18.7.  (With two tokens from 8200 to 10900 rows decodes of 1100 to 1300 frames, 5.0 to 5.6 ms, take
 * as long: not kept.) */
template <int NT>
__global__ void __launch_bounds__(64 * CD_HEADS)
vt_codec_attention_kernel(cd_planes out, const float *__restrict__ qkv, cd_v_rows vs, int T, int window,
                          const float *__restrict__ slopes, float scale) {
    __shared__ float red[CD_HEADS][8 * NT];
    const int h = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 3, sub = lane & 7;
    const int i0 = (blockIdx.x * 8 + g) * NT;
    const float slope = slopes[h];
    const float *base = qkv + h * CD_HEAD_DIM + 4 * sub, *v_base = vs.p + h * CD_HEAD_DIM + 4 * sub;
    auto row = [&](int j, int part) { return cd_load_row(base + (size_t)j * (3 * CD_DIM) + part * CD_DIM); };
    auto v_row = [&](int j) { return cd_load_row(v_base + (size_t)j * vs.stride); };
    int tok[NT], from[NT];
    cd_head_row q[NT];
    cd_softmax st[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        tok[t] = min(i0 + t, T - 1);
        from[t] = window > 0 && tok[t] - window + 1 > 0 ? tok[t] - window + 1 : 0;
        q[t] = row(tok[t], 0);
    }
    cd_head_row k = row(from[0], 1), v = v_row(from[0]);
    for (int j = from[0]; j <= tok[NT - 1]; j++) {
        const int nx = min(j + 1, tok[NT - 1]);
        const cd_head_row nk = row(nx, 1), nv = v_row(nx);
#pragma unroll
        for (int t = 0; t < NT; t++)
            if (j >= from[t] && j <= tok[t])
                st[t].add(cd_row_dot(q[t], k) * scale + slope * (float)(j - tok[t]), v);
        k = nk; v = nv;
    }
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const float inv = st[t].se > 0.f ? 1.0f / st[t].se : 1.0f;
        float m = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            st[t].o.v[e] *= inv;
            m = fmaxf(m, cd_max4(st[t].o.v[e]));
        }
        m = fmaxf(m, vt_dpp<0xB1>(m));
        m = fmaxf(m, vt_dpp<0x4E>(m));
        m = fmaxf(m, vt_dpp<0x141>(m));
        if (sub == 0) red[h][NT * g + t] = m;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; t++) {
        float m = 0.f;
#pragma unroll
        for (int w = 0; w < CD_HEADS; w++) m = fmaxf(m, red[w][NT * g + t]);
        const int ex = vt_f16_exp(m);
        if (i0 + t < T) {
#pragma unroll
            for (int e = 0; e < 4; e++) cd_put4(out, (size_t)(i0 + t) * CD_DIM + h * CD_HEAD_DIM + 32 * e + 4 * sub, st[t].o.v[e], ex);
            if (h == 0 && sub == 0) out.exp[i0 + t] = ex;
        }
    }
}

/* Few tokens: one workgroup each, wave h for head h; its eight groups of eight lanes take every eighth key, so that
 * a window of 16 is two keys deep, and merge their sums: each step hands half of what a lane still holds to its
 * partner and keeps the other half, two dims per lane at the end. */
__global__ void __launch_bounds__(64 * CD_HEADS)
vt_codec_attention_split_kernel(cd_planes out, const float *__restrict__ qkv, int T, int window,
                                const float *__restrict__ slopes, float scale) {
    __shared__ float red[CD_HEADS];
    const int i = blockIdx.x, h = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 3, sub = lane & 7;
    const float slope = slopes[h];
    const float *base = qkv + h * CD_HEAD_DIM + 4 * sub;
    const cd_head_row q = cd_load_row(base + (size_t)i * (3 * CD_DIM));
    const int j0 = (window > 0 && i - window + 1 > 0) ? i - window + 1 : 0;
    cd_softmax s;
    for (int j = j0 + g; j <= i; j += 8) {
        const float *kr = base + (size_t)j * (3 * CD_DIM) + CD_DIM;
        const cd_head_row k = cd_load_row(kr), v = cd_load_row(kr + CD_DIM);
        s.add(cd_row_dot(q, k) * scale + slope * (float)(j - i), v);
    }
    auto ror8 = [](float v) { return vt_dpp<0x128>(v); };        /* the lane 8 away in its row of 16 */
    const float mx = vt_rows_max(fmaxf(s.mx, ror8(s.mx)));
    const float f = s.mx == mx ? 1.0f : expf(s.mx - mx);
    const float sf = s.se * f, se = vt_rows_sum(sf + ror8(sf));
    const bool b3 = lane & 8, b4 = lane & 16, b5 = lane & 32;
    f32x4 r2[2], r1;
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const f32x4 keep = (b3 ? s.o.v[2 + e] : s.o.v[e]) * f, give = (b3 ? s.o.v[e] : s.o.v[2 + e]) * f;
#pragma unroll
        for (int n = 0; n < 4; n++) r2[e][n] = keep[n] + ror8(give[n]);
    }
#pragma unroll
    for (int n = 0; n < 4; n++) {
        const f32x2 r = vt_swap16(r2[0][n], r2[1][n]);
        r1[n] = r.x + r.y;
    }
    const float inv = se > 0.f ? 1.0f / se : 1.0f;
    const f32x2 rx = vt_swap32(r1[0], r1[2]), ry = vt_swap32(r1[1], r1[3]);
    const float x = (rx.x + rx.y) * inv, y = (ry.x + ry.y) * inv;
    float m = vt_wave_max(fmaxf(fabsf(x), fabsf(y)));
    if (lane == 0) red[h] = m;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < CD_HEADS; k++) m = fmaxf(m, red[k]);
    const int ex = vt_f16_exp(m);
    unsigned hi, lo;
    vt_split_f16x2(__builtin_amdgcn_ldexpf(x, ex), __builtin_amdgcn_ldexpf(y, ex), hi, lo);
    const size_t at = (size_t)i * CD_DIM + h * CD_HEAD_DIM + 32 * (2 * (int)b3 + (int)b4) + 4 * sub + 2 * (int)b5;
    *(unsigned *)(out.hi + at) = hi;
    *(unsigned *)(out.lo + at) = lo;
    if (threadIdx.x == 0) out.exp[i] = ex;
}

/* codes [T, 37] -> the three shifted copies of the 292-wide embedding that the input
 * convolution multiplies (embed_codes, voxtral_tts_codec.c:276-300; causal padding with
 * left reflection, voxtral_tts_kernels.c:217-272): a[t][k * 292 + c] = e[src(t, k)][c],
 * src = t + k - 2, reflected to -src when negative, zero when that is outside too. */
__global__ void __launch_bounds__(256)
vt_codec_embed_kernel(cd_planes a, const int *__restrict__ codes, const float *__restrict__ sem, int T) {
    __shared__ float red[4];
    __shared__ int code[CD_IN_TAPS][37];
    const int t = blockIdx.x, base = threadIdx.x * 4;
    /* each code once (they may lie in host memory) */
    if (threadIdx.x < CD_IN_TAPS * 37) {
        const int k = threadIdx.x / 37, src = abs(t + k - (CD_IN_TAPS - 1));
        code[k][threadIdx.x % 37] = src < T ? codes[(size_t)src * 37 + threadIdx.x % 37] : 0;
    }
    __syncthreads();
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (base < CD_IN_K)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int idx = base + i;
            if (idx < CD_IN_TAPS * CD_EMBED) {
                const int k = idx / CD_EMBED, c = idx % CD_EMBED;
                if (abs(t + k - (CD_IN_TAPS - 1)) < T) {
                    if (c < CD_SEM_DIM) {
                        int s = code[k][0] - 2;
                        s = s < 0 ? 0 : s >= CD_SEM_SIZE ? CD_SEM_SIZE - 1 : s;
                        v[i] = sem[(size_t)s * CD_SEM_DIM + c];
                    } else {
                        int q = code[k][c - CD_SEM_DIM + 1] - 2;
                        q = q < 0 ? 0 : q > 20 ? 20 : q;
                        v[i] = (float)q * 2.0f / 20.0f - 1.0f;
                    }
                }
            }
        }
    const int e = vt_f16_exp(cd_block_max(cd_max4(v), red));
    if (base < CD_IN_K) cd_put4(a, (size_t)t * CD_IN_K + base, v, e);
    if (threadIdx.x == 0) a.exp[t] = e;
}

/* waveform row t, t0 + 0 .. of a launch: bias + the sum over the output convolution's taps k of tap k's columns of product row src(t, k),
 * stride 1, left reflection as above */
template <int C>
__global__ void __launch_bounds__(64)
vt_codec_wave_kernel(float *__restrict__ out, cd_product in, const float *__restrict__ bias, int t0) {
    const int t = t0 + blockIdx.x, c = threadIdx.x * 4;
    if (c >= CD_PATCH) return;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    auto src = [&](int k) { return abs(t + k - (CD_OUT_TAPS - 1)); };
    cd_quads<C> q[CD_OUT_TAPS];
#pragma unroll
    for (int k = 0; k < CD_OUT_TAPS; k++) q[k].ask(in, src(k) < in.rows ? src(k) : 0, k * CD_OUT_PITCH + c);
    if (C <= 4) cd_asked();                              /* (of eight planes the registers do not hold all) */
#pragma unroll
    for (int k = 0; k < CD_OUT_TAPS; k++)
        if (src(k) < in.rows) v += q[k].total();
    if (bias) v += *(const f32x4 *)(bias + c);
    *(f32x4 *)(out + (size_t)t * CD_PATCH + c) = v;
}

/* ---- device state -------------------------------------------------------------------------- */

/* A product's weights in fragment order and the exponents of its columns */
struct cd_matrix { uint16_t *wf; int *exp; int n, k; };

struct cd_layer_dev {
    cd_matrix wqkv, wo, w13, w2;
    float *q_norm, *k_norm, *attention_norm, *ffn_norm, *attn_scale, *ffn_scale;
    int window;
};

#define CD_WAVE_PARTS 16

static struct {
    int uploaded;
    float *sem;                   /* [8192, 256] */
    float *slopes;                /* [8] */
    cd_matrix w_in;               /* [1024, 896] */
    cd_layer_dev layers[CD_LAYERS];
    cd_matrix w_up[3];            /* [4096, 1024] */
    cd_matrix w_out;              /* [1792, 1024] */
    float *b_in, *b_up[3], *b_out;
    /* work area, grown to the largest decode so far and laid out anew by each (cd_carve) */
    unsigned char *work;
    size_t work_bytes;
    float *x, *qkv, *part;
    cd_planes planes;
    unsigned char *host;          /* pinned: the waveform of the largest decode so far and its codes (7828 bytes a frame) */
    size_t host_bytes;
    hipEvent_t written[CD_WAVE_PARTS];
    float *probe_wave;            /* vt_codec_probe_buffers */
    int *probe_codes;
} g_cd;

static void cd_free_ptr(float **p) { if (*p) (void)hipFree(*p); *p = NULL; }

static void cd_free_matrix(cd_matrix *m) {
    if (m->wf) (void)hipFree(m->wf);
    if (m->exp) (void)hipFree(m->exp);
    m->wf = NULL;
    m->exp = NULL;
}

void vt_codec_free(void) {
    cd_free_ptr(&g_cd.sem); cd_free_ptr(&g_cd.slopes); cd_free_matrix(&g_cd.w_in); cd_free_ptr(&g_cd.b_in);
    for (int i = 0; i < CD_LAYERS; i++) {
        cd_layer_dev *l = &g_cd.layers[i];
        cd_free_matrix(&l->wqkv); cd_free_matrix(&l->wo); cd_free_matrix(&l->w13); cd_free_matrix(&l->w2);
        float **ps[] = {&l->q_norm, &l->k_norm, &l->attention_norm,
                        &l->ffn_norm, &l->attn_scale, &l->ffn_scale};
        for (size_t k = 0; k < sizeof ps / sizeof ps[0]; k++) cd_free_ptr(ps[k]);
    }
    for (int i = 0; i < 3; i++) { cd_free_matrix(&g_cd.w_up[i]); cd_free_ptr(&g_cd.b_up[i]); }
    cd_free_matrix(&g_cd.w_out); cd_free_ptr(&g_cd.b_out);
    if (g_cd.work) (void)hipFree(g_cd.work);
    if (g_cd.host) (void)hipHostFree(g_cd.host);
    cd_free_ptr(&g_cd.probe_wave);
    if (g_cd.probe_codes) (void)hipFree(g_cd.probe_codes);
    for (int i = 0; i < CD_WAVE_PARTS; i++)
        if (g_cd.written[i]) (void)hipEventDestroy(g_cd.written[i]);
    memset(&g_cd, 0, sizeof g_cd);
}

static float *cd_upload(const float *src, size_t n) {
    float *d = (float *)vt_dev_alloc(n * sizeof(float));
    if (d && vt_check(hipMemcpy(d, src, n * sizeof(float), hipMemcpyDefault), "codec weight copy")) {
        (void)hipFree(d);
        return NULL;
    }
    return d;
}

/* host copy of a tensor that may live on the host or the device (caller frees) */
static float *cd_host(const float *src, size_t n) {
    float *h = (float *)malloc(n * sizeof(float));
    if (h && vt_check(hipMemcpy(h, src, n * sizeof(float), hipMemcpyDefault), "codec weight read")) { free(h); return NULL; }
    return h;
}

/* stack of row blocks [rows_i, cols] -> one device matrix */
static float *cd_upload_stack(const float *const *srcs, const int *rows, int n, int cols) {
    size_t total = 0;
    for (int i = 0; i < n; i++) total += (size_t)rows[i] * cols;
    float *d = (float *)vt_dev_alloc(total * sizeof(float));
    size_t off = 0;
    for (int i = 0; d && i < n; i++) {
        if (vt_check(hipMemcpy(d + off, srcs[i], (size_t)rows[i] * cols * sizeof(float), hipMemcpyDefault), "codec weight copy")) {
            (void)hipFree(d);
            return NULL;
        }
        off += (size_t)rows[i] * cols;
    }
    return d;
}

/* fp32 device matrix [n, k] (freed here) -> m */
static int cd_matrix_from(cd_matrix *m, float *d, int n, int k) {
    int ok = d != NULL;
    m->n = n; m->k = k;
    ok = ok && (m->wf = (uint16_t *)vt_dev_alloc((size_t)n * k * 2 * sizeof(uint16_t))) != NULL;
    ok = ok && (m->exp = (int *)vt_dev_alloc((size_t)n * sizeof(int))) != NULL;
    ok = ok && vt_codec_weight_layout(m->wf, m->exp, d, n, k) == 0;
    if (d) (void)hipFree(d);
    return ok;
}

/* conv1d weight [out_ch, in_ch, taps] -> zeros [n, k_dim] but for element (oc, ic, k) at row oc + row_tap * k, column
 * ic + col_tap * k */
static float *cd_upload_conv(const tts_hip_host_conv_t *cv, int n, int k_dim, int row_tap, int col_tap) {
    float *h = cd_host(cv->weight, (size_t)cv->out_ch * cv->in_ch * cv->kernel);
    float *r = (float *)calloc((size_t)n * k_dim, sizeof(float));
    float *d = NULL;
    if (h && r) {
        for (int oc = 0; oc < cv->out_ch; oc++)
            for (int ic = 0; ic < cv->in_ch; ic++)
                for (int k = 0; k < cv->kernel; k++)
                    r[(size_t)(oc + row_tap * k) * k_dim + ic + col_tap * k] = h[((size_t)oc * cv->in_ch + ic) * cv->kernel + k];
        d = cd_upload(r, (size_t)n * k_dim);
    } else {
        vt_set_error("codec upload: out of host memory");
    }
    free(h); free(r);
    return d;
}

/* transposed conv weight [in_ch, out_ch, 4] -> [4 * 1024, 1024]: row q * 2048 + p * 1024 + oc, column ic holds
 * w[ic][oc][p + 2q] */
static float *cd_upload_convt(const tts_hip_host_conv_t *cv) {
    const size_t n = (size_t)CD_DIM * CD_DIM * 4;
    float *h = cd_host(cv->weight, n);
    float *r = (float *)malloc(n * sizeof(float));
    float *d = NULL;
    if (h && r) {
        for (int ic = 0; ic < CD_DIM; ic++)
            for (int oc = 0; oc < CD_DIM; oc++)
                for (int k = 0; k < 4; k++) {
                    const int p = k & 1, q = k >> 1;
                    r[((size_t)(2 * q + p) * CD_DIM + oc) * CD_DIM + ic] = h[((size_t)ic * CD_DIM + oc) * 4 + k];
                }
        d = cd_upload(r, n);
    } else {
        vt_set_error("codec upload: out of host memory");
    }
    free(h); free(r);
    return d;
}

static float *cd_upload_bias(const float *bias, int n, int n_pad) {
    if (!bias) return NULL;
    float *h = cd_host(bias, n);
    float *r = (float *)calloc(n_pad, sizeof(float));
    float *d = NULL;
    if (h && r) {
        memcpy(r, h, n * sizeof(float));
        d = cd_upload(r, n_pad);
    }
    free(h); free(r);
    return d;
}

static int cd_conv_is(const tts_hip_host_conv_t *cv, int in_ch, int out_ch, int kernel, int stride, int tr) {
    return cv->weight && cv->in_ch == in_ch && cv->out_ch == out_ch && cv->kernel == kernel &&
           cv->stride == stride && !cv->is_transpose == !tr;
}

extern "C" int tts_hip_upload_codec_weights(void *codec_ptr) {
    if (!g_vt.initialized) { vt_set_error("tts_hip_upload_codec_weights: backend not initialised"); return -1; }
    const tts_hip_host_codec_t *c = (const tts_hip_host_codec_t *)codec_ptr;
    if (!c || !c->semantic_embedding) { vt_set_error("tts_hip_upload_codec_weights: NULL codec"); return -1; }
    if (!cd_conv_is(&c->input_conv, CD_EMBED, CD_DIM, CD_IN_TAPS, 1, 0) ||
        !cd_conv_is(&c->output_proj, CD_DIM, CD_PATCH, CD_OUT_TAPS, 1, 0)) {
        vt_set_error("tts_hip_upload_codec_weights: input / output convolution is not 292->1024 k3 s1 / 1024->240 k7 s1");
        return -1;
    }
    for (int i = 0; i < 3; i++)
        if (!cd_conv_is(&c->stage_convs[i], CD_DIM, CD_DIM, 4, 2, 1)) {
            vt_set_error("tts_hip_upload_codec_weights: upsampling convolution %d is not transposed 1024->1024 k4 s2", i);
            return -1;
        }
    (void)hipDeviceSynchronize();
    vt_codec_free();
    int ok = 1;
    ok &= (g_cd.sem = cd_upload(c->semantic_embedding, (size_t)CD_SEM_SIZE * CD_SEM_DIM)) != NULL;
    ok &= (g_cd.slopes = cd_upload(c->alibi_slopes, CD_HEADS)) != NULL;
    ok &= cd_matrix_from(&g_cd.w_in, cd_upload_conv(&c->input_conv, CD_DIM, CD_IN_K, 0, CD_EMBED), CD_DIM, CD_IN_K);
    g_cd.b_in = cd_upload_bias(c->input_conv.bias, CD_DIM, CD_DIM);
    ok &= cd_matrix_from(&g_cd.w_out, cd_upload_conv(&c->output_proj, CD_OUT_N, CD_DIM, CD_OUT_PITCH, 0), CD_OUT_N, CD_DIM);
    g_cd.b_out = cd_upload_bias(c->output_proj.bias, CD_PATCH, CD_OUT_PITCH);
    for (int i = 0; ok && i < 3; i++) {
        ok &= cd_matrix_from(&g_cd.w_up[i], cd_upload_convt(&c->stage_convs[i]), CD_UP_N, CD_DIM);
        g_cd.b_up[i] = cd_upload_bias(c->stage_convs[i].bias, CD_DIM, CD_DIM);
    }
    for (int i = 0; ok && i < CD_LAYERS; i++) {
        const tts_hip_host_codec_layer_t *s = &c->transformers[i];
        cd_layer_dev *l = &g_cd.layers[i];
        if (!s->wq || !s->wk || !s->wv || !s->wo || !s->w1 || !s->w2 || !s->w3 || !s->attention_norm || !s->ffn_norm) {
            vt_set_error("tts_hip_upload_codec_weights: layer %d has a NULL tensor", i);
            ok = 0;
            break;
        }
        const float *qkv[3] = {s->wq, s->wk, s->wv};
        const int r3[3] = {CD_DIM, CD_DIM, CD_DIM};
        const float *gu[2] = {s->w1, s->w3};
        const int r2[2] = {CD_HID, CD_HID};
        ok &= cd_matrix_from(&l->wqkv, cd_upload_stack(qkv, r3, 3, CD_DIM), 3 * CD_DIM, CD_DIM);
        ok &= cd_matrix_from(&l->w13, cd_upload_stack(gu, r2, 2, CD_DIM), 2 * CD_HID, CD_DIM);
        ok &= cd_matrix_from(&l->wo, cd_upload(s->wo, (size_t)CD_DIM * CD_DIM), CD_DIM, CD_DIM);
        ok &= cd_matrix_from(&l->w2, cd_upload(s->w2, (size_t)CD_DIM * CD_HID), CD_DIM, CD_HID);
        ok &= (l->attention_norm = cd_upload(s->attention_norm, CD_DIM)) != NULL;
        ok &= (l->ffn_norm = cd_upload(s->ffn_norm, CD_DIM)) != NULL;
        l->q_norm = s->q_norm ? cd_upload(s->q_norm, CD_DIM) : NULL;
        l->k_norm = s->k_norm ? cd_upload(s->k_norm, CD_DIM) : NULL;
        l->attn_scale = s->attn_scale ? cd_upload(s->attn_scale, CD_DIM) : NULL;
        l->ffn_scale = s->ffn_scale ? cd_upload(s->ffn_scale, CD_DIM) : NULL;
        l->window = s->window_size;
    }
    ok = ok && !vt_check(hipStreamSynchronize(NULL), "codec weight copy");      /* sources may have been device memory */
    if (!ok) { vt_codec_free(); return -1; }
    g_cd.uploaded = 1;
    return 0;
}

/* rows and products of one decode, in order: input convolution, per layer q|k|v, output, gate|up, down, three
 * upsampling products, output convolution */
static vt_gemm_plan cd_plan(int M, const cd_matrix &w) { return vt_codec_gemm_plan(M, w.n, w.k); }

/* floats that a product's result takes (cd_product) */
static size_t cd_part_floats(int M, const cd_matrix &w) {
    const vt_gemm_plan pl = cd_plan(M, w);
    return (size_t)M * (pl.col0 + (size_t)(w.n - pl.col0) * pl.cuts);
}

static int cd_reserve(int n_frames) {
    const size_t T = (size_t)n_frames * 8;
    /* the gate|up product of the last stage and what cut planes add to it on 256 CUs, whatever the row count: a
     * decode finds room where a longer one did */
    size_t part = T * (2 * CD_HID + 2 * CD_HID / 4) + ((size_t)4 << 20);
    const size_t n_in = cd_part_floats(n_frames, g_cd.w_in);
    part = n_in > part ? n_in : part;
    for (int st = 0; st < 4; st++) {
        const int M = n_frames << st;
        const cd_layer_dev *l = &g_cd.layers[2 * st];
        const cd_matrix *m[4] = {&l->wqkv, &l->wo, &l->w13, &l->w2};
        for (int i = 0; i < 4; i++) { const size_t n = cd_part_floats(M, *m[i]); part = n > part ? n : part; }
        const size_t n = st < 3 ? cd_part_floats(M, g_cd.w_up[st]) : cd_part_floats(M, g_cd.w_out);
        part = n > part ? n : part;
    }
    /* the pieces start at multiples of 256 bytes */
    const size_t f = sizeof(float), sizes[] = {T * CD_DIM * f, T * 3 * CD_DIM * f, part * f, T * CD_HID * 2, T * CD_HID * 2, (T + 4) * f};
    size_t total = 0, at[6];
    for (int i = 0; i < 6; i++) { at[i] = total; total += (sizes[i] + 255) & ~(size_t)255; }
    if (total > g_cd.work_bytes) {
        (void)hipStreamSynchronize(g_vt.stream);
        if (g_cd.work) (void)hipFree(g_cd.work);
        g_cd.work_bytes = 0;
        if (!(g_cd.work = (unsigned char *)vt_dev_alloc(total))) return -1;
        g_cd.work_bytes = total;
    }
    g_cd.x = (float *)(g_cd.work + at[0]);
    g_cd.qkv = (float *)(g_cd.work + at[1]);
    g_cd.part = (float *)(g_cd.work + at[2]);
    g_cd.planes = cd_planes{(uint16_t *)(g_cd.work + at[3]), (uint16_t *)(g_cd.work + at[4]), (int *)(g_cd.work + at[5])};
    return 0;
}

/* the product of the rows in g_cd.planes with w, in g_cd.part */
static cd_product cd_gemm(int M, const cd_matrix &w) {
    const vt_gemm_plan pl = cd_plan(M, w);
    vt_launch_codec_gemm(g_cd.part, g_cd.planes.hi, g_cd.planes.lo, g_cd.planes.exp, w.wf, w.exp, M, w.n, w.k, pl);
    return cd_product{g_cd.part, M, w.n, pl.col0, pl.cuts};
}

/* CALL(C) with the instance that requests enough planes at once */
#define CD_BY_CUTS(cuts, CALL) do { if ((cuts) <= 1) { CALL(1); } else if ((cuts) <= 2) { CALL(2); } else if ((cuts) <= 4) { CALL(4); } else { CALL(VT_MAX_CUTS); } } while (0)

/* the rows of a product (up: of the upsampling product, two rows of 1024 each) -> x (bias or layer scale and residual) and
 * planes of its RMSNorm; norm_w NULL: its planes only */
static void cd_row(const cd_product &in, bool up, const float *x_in, const float *bias, const float *scale, const float *norm_w) {
#define CALL(C) \
    if (up) hipLaunchKernelGGL((vt_codec_row_kernel<C, true>), dim3(2 * in.rows), dim3(256), 0, g_vt.stream, g_cd.x, g_cd.planes, x_in, in, bias, \
                               scale, norm_w, CD_EPS); \
    else hipLaunchKernelGGL((vt_codec_row_kernel<C, false>), dim3(in.rows), dim3(256), 0, g_vt.stream, g_cd.x, g_cd.planes, x_in, in, bias, \
                            scale, norm_w, CD_EPS)
    CD_BY_CUTS(in.cuts, CALL);
#undef CALL
}

/* the decoder up to the output convolution's product, on the library's stream: codes [n_frames, 37] */
static cd_product cd_enqueue(const int *codes, int n_frames) {
    int T = n_frames;
    const float scale = 1.0f / sqrtf((float)CD_HEAD_DIM);
    hipLaunchKernelGGL(vt_codec_embed_kernel, dim3(T), dim3(256), 0, g_vt.stream, g_cd.planes, codes, g_cd.sem, T);
    cd_product p = cd_gemm(T, g_cd.w_in);
    cd_row(p, false, NULL, g_cd.b_in, NULL, g_cd.layers[0].attention_norm);
    for (int li = 0; li < CD_LAYERS; li++) {
        const cd_layer_dev *l = &g_cd.layers[li];
        p = cd_gemm(T, l->wqkv);
        cd_v_rows v = T < CD_ATT_SPLIT_BELOW ? cd_v_rows{NULL, 0} : cd_v_in_place(p);
#define CALL(C) hipLaunchKernelGGL((vt_codec_qkv_kernel<C, 3>), dim3(T), dim3(256), 0, g_vt.stream, g_cd.qkv, p, l->q_norm, l->k_norm)
        if (v.p) hipLaunchKernelGGL((vt_codec_qkv_kernel<1, 2>), dim3(T), dim3(256), 0, g_vt.stream, g_cd.qkv, p, l->q_norm, l->k_norm);
        else {
            CD_BY_CUTS(p.cuts, CALL);
            v = cd_v_rows{g_cd.qkv + 2 * CD_DIM, 3 * CD_DIM};
        }
#undef CALL
        if (T < CD_ATT_SPLIT_BELOW)
            hipLaunchKernelGGL(vt_codec_attention_split_kernel, dim3(T), dim3(64 * CD_HEADS), 0, g_vt.stream, g_cd.planes, g_cd.qkv, T, l->window, g_cd.slopes, scale);
        else if ((T + 15) / 16 <= g_vt.n_cu)
            hipLaunchKernelGGL(vt_codec_attention_kernel<2>, dim3((T + 15) / 16), dim3(64 * CD_HEADS), 0, g_vt.stream, g_cd.planes, g_cd.qkv, v, T, l->window, g_cd.slopes, scale);
        else
            hipLaunchKernelGGL(vt_codec_attention_kernel<4>, dim3((T + 31) / 32), dim3(64 * CD_HEADS), 0, g_vt.stream, g_cd.planes, g_cd.qkv, v, T, l->window, g_cd.slopes, scale);
        p = cd_gemm(T, l->wo);
        cd_row(p, false, g_cd.x, NULL, l->attn_scale, l->ffn_norm);
        p = cd_gemm(T, l->w13);
#define CALL(C) hipLaunchKernelGGL(vt_codec_swiglu_kernel<C>, dim3(T), dim3(256), 0, g_vt.stream, g_cd.planes, p)
        CD_BY_CUTS(p.cuts, CALL);
#undef CALL
        p = cd_gemm(T, l->w2);
        const int last_of_stage = (li & 1) == 1;
        cd_row(p, false, g_cd.x, NULL, l->ffn_scale, last_of_stage ? NULL : g_cd.layers[li + 1].attention_norm);
        if (last_of_stage && li < CD_LAYERS - 1) {
            const int st = li / 2;
            p = cd_gemm(T, g_cd.w_up[st]);
            cd_row(p, true, NULL, g_cd.b_up[st], NULL, g_cd.layers[li + 1].attention_norm);
            T *= 2;
        }
    }
    return cd_gemm(T, g_cd.w_out);
}

/* rows t0 .. t1 - 1 of the waveform from that product */
static int cd_wave(float *samples, const cd_product &p, int t0, int t1) {
#define CALL(C) hipLaunchKernelGGL(vt_codec_wave_kernel<C>, dim3(t1 - t0), dim3(64), 0, g_vt.stream, samples, p, g_cd.b_out, t0)
    CD_BY_CUTS(p.cuts, CALL);
#undef CALL
    return vt_check(hipGetLastError(), "codec launch");
}

static int cd_enqueue_all(const int *codes, int n_frames, float *d_samples) { return cd_wave(d_samples, cd_enqueue(codes, n_frames), 0, n_frames * 8); }

#define CD_MAX_FRAMES 4096
static int cd_ready(const char *who, int n_frames) {
    if (!g_vt.initialized || !g_cd.uploaded) { vt_set_error("%s: codec weights not uploaded", who); return -1; }
    if (n_frames < 1 || n_frames > CD_MAX_FRAMES) { vt_set_error("%s: n_frames %d out of range", who, n_frames); return -1; }
    if (cd_reserve(n_frames)) { vt_set_error("%s: out of device memory for %d frames", who, n_frames); return -1; }
    return 0;
}

/* pinned memory and the events of the waveform's parts.  The memory doubles at least, up to what the longest decode takes (32 MB):
 * decodes that slowly get longer pin it anew five times. */
#define CD_WAVE_PART_BYTES (480 << 10)
#define CD_HOST_FRAME_BYTES (sizeof(float) * 8 * CD_PATCH + sizeof(int) * 37)
static int cd_pin(int n_frames) {
    size_t bytes = n_frames * CD_HOST_FRAME_BYTES;
    for (int i = 0; i < CD_WAVE_PARTS; i++)
        if (!g_cd.written[i] && vt_check(hipEventCreateWithFlags(&g_cd.written[i], hipEventDisableTiming), "codec event")) return -1;
    if (bytes <= g_cd.host_bytes) return 0;
    (void)hipStreamSynchronize(g_vt.stream);
    if (g_cd.host) (void)hipHostFree(g_cd.host);
    const size_t longest = CD_MAX_FRAMES * CD_HOST_FRAME_BYTES, twice = 2 * g_cd.host_bytes > 1 << 20 ? 2 * g_cd.host_bytes : 1 << 20;
    bytes = bytes > twice ? bytes : twice < longest ? twice : longest;
    g_cd.host_bytes = 0;
    g_cd.host = NULL;
    if (vt_check(hipHostMalloc((void **)&g_cd.host, bytes, hipHostMallocDefault), "codec host memory")) { g_cd.host = NULL; return -1; }
    g_cd.host_bytes = bytes;
    return 0;
}

/* device codes -> device waveform (n_frames * 1920 floats), asynchronous on the library's stream */
extern "C" int tts_hip_codec_decode_device(const int *d_codes, int n_frames, float *d_samples) {
    if (cd_ready("tts_hip_codec_decode_device", n_frames)) return -1;
    if (!d_codes || !d_samples) { vt_set_error("tts_hip_codec_decode_device: NULL buffer"); return -1; }
    return cd_enqueue_all(d_codes, n_frames, d_samples);
}

/* replaces tts_codec_decode (voxtral_tts_codec.c:389): host codes [n_frames, 37] -> a malloc'ed
 * waveform the caller frees; NULL / 0 on failure. */
extern "C" void tts_hip_codec_decode(const int *codes, int n_frames, float **out_samples, int *out_n_samples) {
    if (out_samples) *out_samples = NULL;
    if (out_n_samples) *out_n_samples = 0;
    if (!codes || !out_samples || !out_n_samples) { vt_set_error("tts_hip_codec_decode: NULL argument"); return; }
    if (cd_ready("tts_hip_codec_decode", n_frames)) return;
    const int rows = n_frames * 8, n = rows * CD_PATCH;
    const size_t code_bytes = (size_t)n_frames * 37 * sizeof(int);
    if (cd_pin(n_frames)) { vt_set_error("tts_hip_codec_decode: out of host memory"); return; }
    float *s = (float *)malloc((size_t)n * sizeof(float));
    if (!s) { vt_set_error("tts_hip_codec_decode: out of host memory"); return; }
    /* Codes and samples cross through pinned memory that the kernels read and write themselves; the caller's buffer is filled
     * part by part behind the last kernel's launches.  Where the codes and the waveform were copied
     * from and into pageable memory, calls of 2 / 21 / 212 / 1003 frames took 508 / 737 / 1630 / 5020 us; 453 / 695 / 1596 / 4791
     * with this, of which 8 / 21 / 95 / 273 behind the device's work. */
    float *wave = (float *)g_cd.host;
    int *host_codes = (int *)(wave + n);
    if (vt_pageable(codes)) memcpy(host_codes, codes, code_bytes);
    else if (vt_check(hipMemcpyAsync(host_codes, codes, code_bytes, hipMemcpyDefault, g_vt.stream), "codes copy")) { free(s); return; }
    const cd_product p = cd_enqueue(host_codes, n_frames);
    int parts = (int)((size_t)n * sizeof(float) / CD_WAVE_PART_BYTES), bad = 0;
    parts = parts < 1 ? 1 : parts < CD_WAVE_PARTS ? parts : CD_WAVE_PARTS;
    auto first = [&](int i) { return (int)((long long)rows * i / parts); };
    for (int i = 0; i < parts && !bad; i++)
        bad = cd_wave(wave, p, first(i), first(i + 1)) || (i + 1 < parts && vt_check(hipEventRecord(g_cd.written[i], g_vt.stream), "codec decode"));
    for (int i = 0; i < parts && !bad; i++) {
        bad = vt_check(i + 1 < parts ? hipEventSynchronize(g_cd.written[i]) : hipStreamSynchronize(g_vt.stream), "codec decode");
        if (!bad) memcpy(s + (size_t)first(i) * CD_PATCH, wave + (size_t)first(i) * CD_PATCH, (size_t)(first(i + 1) - first(i)) * CD_PATCH * sizeof(float));
    }
    if (bad) {
        free(s);
        return;
    }
    *out_samples = s;
    *out_n_samples = n;
}

/* For other translation units of the library: one launch of the decoder's product kernel at the last
 * stage's 1600 rows with the q|k|v, output, gate|up or down matrix of layer 7 (which 0..3), or of the whole
 * decoder on 200 frames of resident codes (which 4), on the decoder's own work area and a waveform and codes of the
 * probe's.  vt_codec_probe_fill makes
 * the planes that which 0..3 read from fp32 values x [1600, k], k = 1024 or 4096. */
#define CD_PROBE_FRAMES 200
int vt_codec_probe_buffers(float **x, int **codes) {
    if (!g_cd.uploaded) { vt_set_error("codec weights not uploaded"); return -1; }
    if (cd_reserve(CD_PROBE_FRAMES)) { vt_set_error("codec: out of device memory"); return -1; }
    if (!g_cd.probe_wave && !(g_cd.probe_wave = (float *)vt_dev_alloc(sizeof(float) * CD_PROBE_FRAMES * 8 * CD_PATCH))) return -1;
    if (!g_cd.probe_codes && !(g_cd.probe_codes = (int *)vt_dev_alloc(sizeof(int) * CD_PROBE_FRAMES * 37))) return -1;
    *x = g_cd.part; *codes = g_cd.probe_codes;
    return 0;
}

__global__ void __launch_bounds__(256) vt_codec_probe_planes_kernel(cd_planes p, const float *x, int k) {
    __shared__ float red[4];
    float m = 0.f;
    for (int c = threadIdx.x * 4; c < k; c += 1024) m = fmaxf(m, cd_max4(*(const f32x4 *)(x + (size_t)blockIdx.x * k + c)));
    const int e = vt_f16_exp(cd_block_max(m, red));
    for (int c = threadIdx.x * 4; c < k; c += 1024) cd_put4(p, (size_t)blockIdx.x * k + c, *(const f32x4 *)(x + (size_t)blockIdx.x * k + c), e);
    if (threadIdx.x == 0) p.exp[blockIdx.x] = e;
}

void vt_codec_probe_fill(const float *x, int k) {
    hipLaunchKernelGGL(vt_codec_probe_planes_kernel, dim3(1600), dim3(256), 0, g_vt.stream, g_cd.planes, x, k);
}

int vt_codec_probe_launch(int which) {
    const int frames = CD_PROBE_FRAMES;
    const cd_layer_dev *l = &g_cd.layers[CD_LAYERS - 1];
    const cd_matrix *w[4] = {&l->wqkv, &l->wo, &l->w13, &l->w2};
    if (which == 4) return cd_enqueue_all(g_cd.probe_codes, frames, g_cd.probe_wave);
    if (which < 0 || which > 3) return -1;
    (void)cd_gemm(frames * 8, *w[which]);
    return 0;
}

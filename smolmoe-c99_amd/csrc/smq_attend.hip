/* Prefill attention (many tokens) in three launches over a workspace of
 * scores, for head sizes that are multiples of 8 and any context.
 *
 * The arithmetic is attend_f32's (kernels.c:1154-1176), bit for bit: every
 * product is rounded to f32 before it is added, and every sum has one order
 * (the 8-lane dot_f32 of kernels.c:1119-1127, the softmax total and the value
 * columns in position order). So the bound is the VALU: a multiply and an add
 * per element of K and of V for each row (token, query head). The multiplies
 * are taken off it: v_mfma_f32_16x16x1_4b with a zero accumulator forms four
 * 16 x 16 outer products, each element one f32 product rounded once
 * (denormals kept; an underflow to -0 instead of +0 changes no sum that holds
 * a nonzero term), and the VALU does the adds. A tile is 16 rows that share a
 * KV head, so each K and V row read serves 16 rows, and neither operand needs
 * a broadcast. Measured per wave with four on a SIMD: 8 such products and their
 * 128 adds 247 ns; 128 v_mul and 128 v_add 231 ns, but 302 ns when the common
 * operand comes by DPP, and scalar loads of it did not keep up.
 * 256 tokens at positions 3328-3583, 12 heads of 128 over 2 KV heads: 4220 us
 * with a workgroup per token, head and 32 columns -> 171 us (traced one by
 * one, with their own start and end, scores 72, softmax 29, values 90; the
 * products and adds alone need about 40 + 40 at four waves per SIMD, and this
 * many rows fill less than two). */
#include "smq_device.h"

namespace smq {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr uint32_t AP_ROWS = 16; /* rows per tile */
constexpr uint32_t AP_SW = 4;    /* row tiles (waves) per scores workgroup */
constexpr uint32_t AP_VW = 4;    /* 16-column tiles (waves) per values workgroup */
constexpr uint32_t AP_CH = 240;  /* positions per softmax chunk: a group of 16 for each of 15 waves */
constexpr uint32_t AP_CHP = AP_CH + 20; /* room for the read past a chunk; 4 mod 64: 16 rows meet every bank */
constexpr uint32_t AP_OOB = 0x80000000u; /* a buffer offset past every record: reads zeros */

struct PreArgs {
    const float *q, *k, *v; /* q and att from the slab's first token */
    float *att, *xd;
    int8_t *xq;
    int *flag;
    float *ws, *inv; /* scores, then exp(s - max) [kv][tile][16][stride]; 1 / total per row */
    uint32_t kv_heads, grp, hd, q_dim, kv_dim, window;
    uint32_t pos0; /* position of the slab's first token */
    uint32_t rows, tiles, stride, pc;
};

/* Row i of a KV head's rows: token i / grp, query head i % grp; rows past the end repeat the last. */
__device__ __forceinline__ uint32_t ap_row(const PreArgs &a, uint32_t i) { return i < a.rows ? i : a.rows - 1; }
__device__ __forceinline__ uint32_t ap_pos(const PreArgs &a, uint32_t i) { return a.pos0 + ap_row(a, i) / a.grp; }
__device__ __forceinline__ uint32_t ap_start(const PreArgs &a, uint32_t pos) {
    return a.window && pos >= a.window ? pos - a.window + 1 : 0; /* model.c:466-470 */
}
/* First position of a tile's score columns. A row keeps its columns in groups of 16 positions, position
 * 4j + b of a group in slot 4b + j: the four weights of a 16-byte read then belong to block b of the four
 * products j = 0..3 that k_ap_values adds one after the other. */
__device__ __forceinline__ uint32_t ap_base(const PreArgs &a, uint32_t tile) {
    return ap_start(a, ap_pos(a, tile * AP_ROWS)) & ~(AP_ROWS - 1);
}
__device__ __forceinline__ uint32_t ap_last(const PreArgs &a, uint32_t tile) {
    return ap_pos(a, tile * AP_ROWS + AP_ROWS - 1);
}

/* Four outer products a[blk][row] * b[blk][col]: lane L supplies a and b of block L/16, row or column
 * L%16, and receives element (row 4(L/16)+v, column L%16) of block m in component 4m+v. */
__device__ __forceinline__ v16f outer4(float a, float b) {
    const v16f zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, zero, 0, 0, 0);
}
/* The rows of one KV head up to position `last`, as a buffer: a read past them returns zeros. Offsets are
 * formed as voffset (lane) + soffset (uniform, at most the last row's). */
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ap_rows(const float *cache, uint32_t kh, uint32_t hd, uint32_t kv_dim,
                                                          uint32_t last) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)(cache + (size_t)kh * hd), 0, (int)((last * kv_dim + hd) * 4),
                                             0x00027000);
}
__device__ __forceinline__ f4v buf4(__amdgpu_buffer_rsrc_t s, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(s, voff, soff, 0));
}

/* Scaled scores of one row tile over a.pc positions, a wave per tile. Block b of a product is the group of
 * eight elements 4g + b, the product's index l in the group the dot's lane, so lane sum l adds its products
 * in element order over (g, b); groups past the head are zeros, which change no sum. q from LDS; the K rows
 * of the next 16 positions are requested as soon as a group's products are issued; the adds of a product
 * run while the next one forms. */
template <int NG>
__global__ __launch_bounds__(64 * AP_SW) __attribute__((amdgpu_waves_per_eu(NG <= 4 ? 4 : 2, 8))) void k_ap_scores(PreArgs a) {
    constexpr uint32_t QP = 32 * NG + 4;
    __shared__ __attribute__((aligned(16))) float qs[AP_SW][AP_ROWS * QP];
    const uint32_t L = threadIdx.x & 63u, r = L & 15u, b = L / 16, kh = blockIdx.z;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), tile = blockIdx.y * AP_SW + w;
    if (tile >= a.tiles) return; /* no barrier: each wave stages its own q */
    const uint32_t last = ap_last(a, tile), base = ap_base(a, tile), c0 = base + blockIdx.x * a.pc;
    if (c0 > last) return;
    const uint32_t c1 = c0 + a.pc < last + 1 ? c0 + a.pc : last + 1;
    const __amdgpu_buffer_rsrc_t src = ap_rows(a.k, kh, a.hd, a.kv_dim, last);
    const uint32_t off = (r * a.kv_dim + 8 * b) * 4, rowb = a.kv_dim * 4;
    const uint32_t offn = 32 * (NG - 1) + 8 * b < a.hd ? off : AP_OOB; /* the last group's, past the head zeros */
    f4v kv[NG][2];
    auto kload = [&](int g, uint32_t p) __attribute__((always_inline)) {
        const uint32_t o = (g == NG - 1 ? offn : off) + 128 * g;
        kv[g][0] = buf4(src, o, p * rowb);
        kv[g][1] = buf4(src, o + 16, p * rowb);
    };
#pragma unroll
    for (int g = 0; g < NG; ++g) kload(g, c0);
    {
        const uint32_t i = ap_row(a, tile * AP_ROWS + r);
        const float *qp = a.q + (size_t)(i / a.grp) * a.q_dim + (size_t)(kh * a.grp + i % a.grp) * a.hd;
        const f4v zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (uint32_t g = 0; g < NG; ++g) {
            const uint32_t e = 32 * g + 8 * b;
            *(f4v *)&qs[w][r * QP + e] = e < a.hd ? *(const f4v *)(qp + e) : zero;
            *(f4v *)&qs[w][r * QP + e + 4] = e < a.hd ? *(const f4v *)(qp + e + 4) : zero;
        }
    }
    const float *qr = &qs[w][r * QP + 8 * b];
    const float factor = 1.0f / sqrtf((float)a.hd);
    float *out = a.ws + ((size_t)(kh * a.tiles + tile) * AP_ROWS + 4 * b) * a.stride + (4 * (r & 3u) + r / 4);
    for (uint32_t p = c0; p < c1; p += 16) {
        const uint32_t pn = p + 16 < c1 ? p + 16 : p;
        float s[8][4];
        v16f d;
        f4v qn0 = *(const f4v *)qr, qn1 = *(const f4v *)(qr + 4);
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const f4v q0 = qn0, q1 = qn1;
            if (g + 1 < NG) {
                qn0 = *(const f4v *)(qr + 32 * (g + 1));
                qn1 = *(const f4v *)(qr + 32 * (g + 1) + 4);
            }
#pragma unroll
            for (int l = 0; l < 8; ++l) {
                const v16f n = outer4(l < 4 ? q0[l & 3] : q1[l & 3], l < 4 ? kv[g][0][l & 3] : kv[g][1][l & 3]);
                __builtin_amdgcn_sched_barrier(0);
                if (g || l) {
                    const int lp = (l + 7) & 7, first = l ? g == 0 : g == 1;
#pragma unroll
                    for (int m = 0; m < 4; ++m)
#pragma unroll
                        for (int v = 0; v < 4; ++v) s[lp][v] = first && m == 0 ? d[v] : s[lp][v] + d[4 * m + v];
                }
                __builtin_amdgcn_sched_barrier(0);
                d = n;
            }
            kload(g, pn);
        }
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v) s[7][v] = NG == 1 && m == 0 ? d[v] : s[7][v] + d[4 * m + v];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float p04 = s[0][v] + s[4][v], p15 = s[1][v] + s[5][v], p26 = s[2][v] + s[6][v],
                        p37 = s[3][v] + s[7][v];
            const float e2 = p04 + p26, o2 = p15 + p37;
            out[(size_t)v * a.stride + (p - base)] = (e2 + o2) * factor;
        }
    }
}

/* Softmax weights of one row tile. A wave per row finds the maximum (order-free; NaN never wins). Then 15
 * waves form exp_det(s - max), a group of 16 positions of every row each, written back and to LDS, two
 * chunks of 15 groups requested ahead; the last wave meanwhile adds the previous chunk, a lane per row, in
 * position order (the serial part: it sets the pace). A position outside a row's range adds +0.0, which
 * changes no total. */
__global__ __launch_bounds__(64 * AP_ROWS) void k_ap_softmax(PreArgs a) {
    __shared__ __attribute__((aligned(16))) float buf[2][AP_ROWS * AP_CHP];
    __shared__ float high[AP_ROWS];
    __shared__ uint64_t etab[32];
    const uint32_t tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid / 64), L = tid & 63u;
    const uint32_t tile = blockIdx.x, kh = blockIdx.y, base = ap_base(a, tile), span = ap_last(a, tile) - base + 1;
    float *rows = a.ws + (size_t)(kh * a.tiles + tile) * AP_ROWS * a.stride;
    if (tid < 32) etab[tid] = EXP2_TABLE[tid];
    const uint32_t groups = (span + 15) / 16;
    {
        const uint32_t pos = ap_pos(a, tile * AP_ROWS + w), lo = ap_start(a, pos) - base, hi = pos - base;
        const float *row = rows + (size_t)w * a.stride + 4 * (L & 3u);
        float m = -FLT_MAX;
        for (uint32_t g0 = 0; g0 < groups; g0 += 16 * 4) { /* four reads of 16 groups at once, clamped */
            f4v s[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const uint32_t g = g0 + 16 * u + L / 4;
                s[u] = *(const f4v *)(row + 16 * (g < groups ? g : groups - 1));
            }
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u)
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    const uint32_t p = 16 * (g0 + 16 * u + L / 4) + (L & 3u) + 4 * k;
                    const float v = p >= lo && p <= hi ? s[u][k] : -FLT_MAX;
                    m = v > m ? v : m;
                }
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const float o = __shfl_xor(m, off, 64);
            m = o > m ? o : m;
        }
        if (L == 0) high[w] = m;
    }
    __syncthreads();
    constexpr uint32_t CG = AP_CH / 16; /* groups per chunk: one per exp wave */
    const uint32_t nch = (groups + CG - 1) / CG;
    if (w < CG) {
        const uint32_t r = L / 4, pos = ap_pos(a, tile * AP_ROWS + r), lo = ap_start(a, pos) - base, hi = pos - base;
        const float m = high[r];
        /* a group past the last reads zeros and stores nothing: every step issues the same operations, so a
         * wait for the oldest load leaves the others in flight */
        const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(rows, 0, (int)(AP_ROWS * a.stride * 4), 0x00027000);
        const uint32_t cell = (r * a.stride + 4 * (L & 3u)) * 4;
        auto at = [&](uint32_t g) __attribute__((always_inline)) { return g < groups ? cell + 64 * g : AP_OOB; };
        auto load = [&](uint32_t c) __attribute__((always_inline)) { return buf4(src, at(c * CG + w), 0); };
        f4v n[2] = {load(0), load(1)};
        auto step = [&](uint32_t c, f4v &x) __attribute__((always_inline)) {
            const uint32_t g = c * CG + w, p = 16 * g + (L & 3u);
            f4v s;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                float e = exp_det_flat(x[k] - m, etab);
                asm("" : "+v"(e)); /* not sunk into a branch */
                s[k] = p + 4 * k >= lo && p + 4 * k <= hi ? e : 0.0f;
            }
            x = load(c + 2);
            *(f4v *)&buf[c & 1u][r * AP_CHP + 16 * w + 4 * (L & 3u)] = s;
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, s), src, at(g), 0, 0);
            __syncthreads();
        };
        for (uint32_t c = 0; c < nch; c += 2) {
            step(c, n[0]);
            if (c + 1 < nch) step(c + 1, n[1]);
        }
        return;
    }
    float t = 0.0f;
    __builtin_amdgcn_s_setprio(3); /* the chain before the three waves of its SIMD that form weights: 177 -> 171 us above */
    __syncthreads();
    for (uint32_t c = 0; c < nch; ++c) { /* chunk c, while the others form chunk c + 1 */
        const uint32_t left = groups - c * CG, n = left < CG ? left : CG;
        const f4v *x4 = (const f4v *)(buf[c & 1u] + (L & 15u) * AP_CHP); /* lanes 16.. repeat rows */
        f4v x[4], y[4];
        auto read = [&](f4v (&z)[4], uint32_t g) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < 4; ++k) z[k] = x4[4 * g + k];
            __builtin_amdgcn_sched_barrier(0);
        };
        auto add = [&](const f4v (&z)[4]) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int j = 0; j < 4; ++j) t = t + z[j][k];
            __builtin_amdgcn_sched_barrier(0);
        };
        read(x, 0);
        for (uint32_t g = 0; g < n; g += 2) { /* the next group's reads in flight (past the last: the next row's) */
            read(y, g + 1);
            add(x);
            if (g + 1 >= n) break;
            read(x, g + 2);
            add(y);
        }
        if (c + 1 < nch) __syncthreads();
    }
    if (L < AP_ROWS) a.inv[(size_t)(kh * a.tiles + tile) * AP_ROWS + L] = 1.0f / t;
}

/* Weighted values (exp_p * inv) * v_p[j] of one row tile (kernels.c:1165): a wave owns 16 columns; block b of
 * the j-th product of a group is position 4j + b, so the products' blocks are added in position order. V and
 * the weights are requested AP_PF groups ahead (both come from beyond the L2 as a rule). Groups that hold
 * positions outside some row's range (the batch's own last positions, a window's first) are added by a
 * select. Then the rows and their Q8 blocks (a half wave each). */
constexpr int AP_PF = 8;
template <bool MASK>
__device__ __forceinline__ void ap_add(float (&acc)[4], const v16f &d, uint32_t p, const uint32_t (&lo)[4],
                                       const uint32_t (&hi)[4]) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float t = acc[v] + d[4 * m + v];
            acc[v] = !MASK || (p + m >= lo[v] && p + m <= hi[v]) ? t : acc[v];
        }
}
template <bool MASK>
__device__ __forceinline__ void ap_group(float (&acc)[4], const f4v &w, const float (&v)[4], uint32_t p,
                                         const uint32_t (&lo)[4], const uint32_t (&hi)[4]) {
    v16f d0 = outer4(w[0], v[0]);
    const v16f d1 = outer4(w[1], v[1]);
    __builtin_amdgcn_sched_barrier(0);
    ap_add<MASK>(acc, d0, p, lo, hi);
    __builtin_amdgcn_sched_barrier(0);
    d0 = outer4(w[2], v[2]);
    __builtin_amdgcn_sched_barrier(0);
    ap_add<MASK>(acc, d1, p + 4, lo, hi);
    __builtin_amdgcn_sched_barrier(0);
    const v16f d3 = outer4(w[3], v[3]);
    __builtin_amdgcn_sched_barrier(0);
    ap_add<MASK>(acc, d0, p + 8, lo, hi);
    ap_add<MASK>(acc, d3, p + 12, lo, hi);
}
__global__ __launch_bounds__(64 * AP_VW) __attribute__((amdgpu_waves_per_eu(2, 8))) void k_ap_values(PreArgs a) {
    constexpr uint32_t OP = 16 * AP_VW + 4;
    __shared__ __attribute__((aligned(16))) float os[AP_ROWS * OP];
    const uint32_t tid = threadIdx.x, L = tid & 63u, r = L & 15u, b = L / 16;
    const uint32_t tile = blockIdx.x, kh = blockIdx.y, jw = blockIdx.z * 16 * AP_VW;
    const uint32_t j0 = jw + __builtin_amdgcn_readfirstlane(tid / 64) * 16;
    const uint32_t first = ap_pos(a, tile * AP_ROWS), last = ap_last(a, tile), base = ap_base(a, tile);
    const uint32_t edge = ap_start(a, last); /* [edge, first]: in every row's range */
    const size_t row0 = (size_t)(kh * a.tiles + tile) * AP_ROWS;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (j0 < a.hd) { /* uniform; a tile past the head has no columns */
        const __amdgpu_buffer_rsrc_t vsrc = ap_rows(a.v, kh, a.hd, a.kv_dim, last);
        const __amdgpu_buffer_rsrc_t wsrc =
            __builtin_amdgcn_make_buffer_rsrc((void *)(a.ws + row0 * a.stride), 0, (int)(AP_ROWS * a.stride * 4), 0x00027000);
        const uint32_t woff = (r * a.stride + 4 * b) * 4, rowb = a.kv_dim * 4;
        uint32_t voff[4]; /* product j: position 4j + b */
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) voff[j] = ((4 * j + b) * a.kv_dim + j0 + r) * 4;
        const float inv = a.inv[row0 + r];
        uint32_t lo[4], hi[4];
#pragma unroll
        for (uint32_t v = 0; v < 4; ++v) {
            hi[v] = ap_pos(a, tile * AP_ROWS + 4 * b + v);
            lo[v] = ap_start(a, hi[v]);
        }
        const uint32_t ng = (last - base) / 16 + 1;
        f4v wn[AP_PF];
        float vn[AP_PF][4];
        auto load = [&](int u, uint32_t g) __attribute__((always_inline)) {
            g = g < ng ? g : ng - 1;
            wn[u] = buf4(wsrc, woff, 64 * g);
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                vn[u][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(vsrc, voff[j], (base + 16 * g) * rowb, 0));
        };
#pragma unroll
        for (int u = 0; u < AP_PF; ++u) {
            load(u, u);
            __builtin_amdgcn_sched_barrier(0); /* issued in the loop's order: its waits count on it */
        }
        for (uint32_t g0 = 0; g0 < ng; g0 += AP_PF) {
#pragma unroll
            for (int u = 0; u < AP_PF; ++u) {
                const uint32_t g = g0 + u, p = base + 16 * g;
                const f4v w = wn[u] * inv;
                const float v[4] = {vn[u][0], vn[u][1], vn[u][2], vn[u][3]};
                __builtin_amdgcn_sched_barrier(0);
                load(u, g + AP_PF);
                __builtin_amdgcn_sched_barrier(0);
                if (p >= edge && p + 15 <= first) { /* uniform */
                    ap_group<false>(acc, w, v, p, lo, hi);
                } else if (g < ng) {
                    uint32_t pv = p;
                    asm("" : "+v"(pv)); /* selects, not a branch per product */
                    ap_group<true>(acc, w, v, pv, lo, hi);
                }
            }
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) os[(4 * b + v) * OP + tid / 64 * 16 + r] = acc[v];
    __syncthreads();
    for (uint32_t task = tid / 32; task < AP_ROWS * AP_VW / 2; task += AP_VW * 2) { /* a row's 32 columns */
        const uint32_t rr = task / (AP_VW / 2), jl = task % (AP_VW / 2) * 32 + (tid & 31u), j = jw + jl;
        const uint32_t i = tile * AP_ROWS + rr;
        if (i >= a.rows || j >= a.hd) continue; /* whole half waves where Q8 blocks are formed (hd % 32 == 0) */
        const uint32_t t = i / a.grp, head = kh * a.grp + i % a.grp;
        const float o = os[rr * OP + jl];
        a.att[(size_t)t * a.q_dim + (size_t)head * a.hd + j] = o;
        if (a.xd) { /* kernels.c:912-935 */
            const float av = fabsf(o);
            const bool bad = !(av <= FLT_MAX);
            const float scale = max32(av) / 127.0f;
            const float qinv = scale >= FLT_MIN ? 1.0f / scale : 0.0f;
            const float pq = o * qinv;
            int qi = (int)__builtin_rintf(pq);
            qi = qi > 127 ? 127 : (qi < -127 ? -127 : qi);
            const size_t blk = (size_t)t * (a.q_dim / QK) + (size_t)head * (a.hd / QK) + j / QK;
            a.xq[blk * QK + j % QK] = (int8_t)qi;
            if (j % QK == 0) a.xd[blk] = scale;
            if (bad && a.flag) *a.flag = 1;
        }
    }
}

}  // namespace

/* Score columns of a tile (its rows' positions from a multiple of 16; a multiple of 16) and the tokens whose
 * score rows fit the workspace with a float more per row for 1 / total. */
struct Slab {
    uint32_t stride, tokens;
};
static Slab attend_slab(const AttnShape &sh, uint32_t seen, size_t ws_bytes) {
    const uint32_t grp = sh.heads / sh.kv_heads;
    const uint32_t wide = sh.window < seen ? sh.window + AP_ROWS / grp + 2 + 16 : seen; /* a tile's tokens too */
    Slab z;
    z.stride = ((sh.window && wide < seen ? wide : seen) + 16 + 15) & ~15u;
    const size_t tiles = ws_bytes / sizeof(float) / ((size_t)AP_ROWS * (z.stride + 1)) / sh.kv_heads;
    z.tokens = (uint32_t)(tiles * AP_ROWS / grp);
    return z;
}

bool attend_tiles_ok(const AttnShape &sh, const float *q, const float *kcache, const float *vcache, uint32_t ntok,
                     uint32_t pos0, size_t ws_bytes) {
    return sh.head_dim % 8 == 0 && sh.head_dim <= MAX_HEAD_DIM && sh.heads % sh.kv_heads == 0 &&
           (((uintptr_t)q | (uintptr_t)kcache | (uintptr_t)vcache) & 15u) == 0 &&
           (uint64_t)sh.context * sh.kv_dim * 4 < AP_OOB && /* offsets into a cache */
           attend_slab(sh, pos0 + ntok, ws_bytes).tokens != 0;
}

template <int NG>
static void ap_scores(const PreArgs &a, dim3 grid, hipStream_t s) {
    hipLaunchKernelGGL(k_ap_scores<NG>, grid, dim3(64 * AP_SW), 0, s, a);
}

hipError_t launch_attend_tiles(const float *q, const float *kcache, const float *vcache, float *att, uint32_t ntok,
                               const AttnShape &sh, uint32_t pos0, int *flag, float *xd, int8_t *xq, float *ws,
                               size_t ws_bytes, hipStream_t s) {
    PreArgs a;
    a.k = kcache;
    a.v = vcache;
    a.flag = flag;
    a.kv_heads = sh.kv_heads;
    a.grp = sh.heads / sh.kv_heads;
    a.hd = sh.head_dim;
    a.q_dim = sh.q_dim;
    a.kv_dim = sh.kv_dim;
    a.window = sh.window;
    const Slab slab = attend_slab(sh, pos0 + ntok, ws_bytes);
    if (!slab.tokens) return hipErrorInvalidValue;
    a.stride = slab.stride;
    for (uint32_t t0 = 0; t0 < ntok;) {
        const uint32_t n = ntok - t0 < slab.tokens ? ntok - t0 : slab.tokens;
        a.q = q + (size_t)t0 * sh.q_dim;
        a.att = att + (size_t)t0 * sh.q_dim;
        a.xd = xd ? xd + (size_t)t0 * (sh.q_dim / QK) : nullptr;
        a.xq = xq ? xq + (size_t)t0 * sh.q_dim : nullptr;
        a.pos0 = pos0 + t0;
        a.rows = n * a.grp;
        a.tiles = (a.rows + AP_ROWS - 1) / AP_ROWS;
        a.ws = ws;
        a.inv = ws + (size_t)sh.kv_heads * a.tiles * AP_ROWS * a.stride;
        const uint32_t groups = (a.tiles + AP_SW - 1) / AP_SW;
        /* positions per wave: 256 unless that gives fewer than 1024 workgroups, at least 32 */
        a.pc = 256;
        while (a.pc > 32 && (uint64_t)((a.stride + a.pc - 1) / a.pc) * groups * sh.kv_heads < 1024) a.pc /= 2;
        const dim3 sgrid((a.stride + a.pc - 1) / a.pc, groups, sh.kv_heads);
        switch ((sh.head_dim + 31) / 32) {
        case 1: ap_scores<1>(a, sgrid, s); break;
        case 2: ap_scores<2>(a, sgrid, s); break;
        case 3: ap_scores<3>(a, sgrid, s); break;
        case 4: ap_scores<4>(a, sgrid, s); break;
        case 5: ap_scores<5>(a, sgrid, s); break;
        case 6: ap_scores<6>(a, sgrid, s); break;
        case 7: ap_scores<7>(a, sgrid, s); break;
        default: ap_scores<8>(a, sgrid, s); break;
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_ap_softmax, dim3(a.tiles, sh.kv_heads), dim3(64 * AP_ROWS), 0, s, a);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_ap_values, dim3(a.tiles, sh.kv_heads, (sh.head_dim + 16 * AP_VW - 1) / (16 * AP_VW)),
                           dim3(64 * AP_VW), 0, s, a);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        t0 += n;
    }
    return hipSuccess;
}

}  // namespace smq

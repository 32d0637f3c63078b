/* Q5 weight conversion on gfx950 (reference: src/kernels.c:1064-1117,
 * quantize_q5_row, as src/quantize_main.c:107-121 runs it row by row).
 *
 * Per 32-element block: the signed extreme (the first element of largest
 * magnitude; a NaN element is never chosen), then 21 candidate scales
 * d_k = f16(extreme / -(14.5 + 0.1k)) (f32 arithmetic, binary16 rounding to
 * nearest even, k = 0..20; a zero or non-finite d_k is skipped); each
 * candidate's squared error sum_j (x_j - clamp(rint(x_j * (1/d_k)), -16, 15) * d_k)^2
 * is formed in binary64 in element order; the first minimum wins (with a NaN
 * element every sum is NaN and the first kept candidate stays); codes q + 16
 * are packed as 16 nibble bytes (element j low, j + 16 high) after the f16
 * scale and the 32-bit plane of fifth bits (docs/FORMAT.md:124-134).
 *
 * Mapping: a wave takes six (few blocks in all: three) consecutive blocks and needs no
 * barrier. Eight lanes per block load four elements each and find the extreme; then a lane
 * per (block, candidate), 63 of them in each of two rounds (one), sums over the block's
 * elements in LDS; eight lanes per block quantize and pack, and the bytes go out as words
 * (half words: three blocks are 66 bytes).
 *
 * What bounds it is the 21 x 32 terms per block, so a term is as short as its value
 * allows. q * d is exact in binary32 (5 and 11 significant bits). x - q * d is exact too:
 * for q = 0 it is x; otherwise x lies within a factor of two of q * d (Sterbenz). For
 * |q| >= 2 and the clamped ends that is plain: |x / d| is at most 24.75, even where d is
 * a subnormal half. For |q| = 1, rint gave 1, so p = fl(x * dinv) is at least 1/2 + 2^-24
 * and, with both roundings below 2^-24, x / d at least 1/2 (1 - 2^-48): as x and d / 2 are
 * binary32 numbers, x >= d / 2. The square of a binary32 number is exact in binary64, so
 * one fused multiply-add is the reference's square, then sum.
 *
 * The sums are formed in binary32 first: 32 fused steps of terms >= 0 are within 2^-19 of the
 * exact sum, so a candidate more than a factor 1 + 2^-17 above the smallest is not the minimum
 * (below 2^-99, where a square may underflow, all are kept). Only where another candidate is
 * within that are the kept ones summed in binary64; one block in some thousand of N(0, s).
 * A term is five binary32 operations, which at full rate take 37 us of 8960 x 1536. Measured
 * there: half a wave per block and four binary64 operations a term 253 us; a workgroup per 24
 * blocks, a conversion and a binary64 fma a term 71.2; binary32 sums 67.6; a wave per six blocks
 * 63.1; the winner's scale from its lane, scalar row division, no half operands 55.4.
 */
#include <float.h>

#include "smq_device.h"
#include "smq_internal.h"

namespace smq {
namespace {

constexpr uint32_t CV_WG = 256;
constexpr uint32_t CV_K = 21;
constexpr uint32_t CV_PITCH = 36; /* floats per block: a round's three blocks on distinct banks */

/* lrintf(v * inv) clamped to the 5-bit range (kernels.c:1064-1067). A NaN product takes
 * -16: x86-64's lrintf returns LONG_MIN for it (cvtss2si's "integer indefinite"), which the
 * clamp turns into -16 on the host the reference and the oracle run on. */
__device__ __forceinline__ int q5_level(float v, float inv) {
    const float p = v * inv;
    const float r = __builtin_rintf(p);
    return !(r >= -16.0f) ? -16 : (r > 15.0f ? 15 : (int)r);
}

/* binary32 -> binary16 bits, round to nearest even, overflow to infinity,
 * subnormal results kept (one v_cvt_f16_f32; f16 denormals are on). */
__device__ __forceinline__ uint32_t to_half_bits(float f) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)f);
}

/* Candidate k's scale as a half (0 or non-finite: skipped). */
__device__ __forceinline__ uint32_t q5_candidate(float extreme, uint32_t k) {
    const float t = 0.1f * (float)k;
    const float divisor = -(14.5f + t);
    return to_half_bits(extreme / divisor);
}

/* LDS written by this wave's lanes, read by its other lanes (LDS serves a wave in order). */
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
template <int CTRL>
__device__ __forceinline__ uint32_t or_dpp(uint32_t v) {
    return v | (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}

/* quad: rows of whole quads of elements at 16-byte addresses (one read per lane). ROUNDS: one of 63 candidates a wave
 * where the blocks leave the chip idle, so that a wave's serial chain is half as long. */
template <uint32_t ROUNDS>
__global__ __launch_bounds__(CV_WG) void k_quantize_q5(const float *x, uint32_t blocks, uint32_t nb, uint32_t cols,
                                                       bool quad, unsigned char *out) {
    constexpr uint32_t W = CV_WG / 64, CV_BLOCKS = 3 * ROUNDS; /* per wave: 21 candidates of three blocks a round */
    __shared__ __attribute__((aligned(16))) float s_x[W][CV_BLOCKS * CV_PITCH];
    __shared__ double s_exact[W][CV_BLOCKS * CV_K];
    __shared__ float s_scale[W][CV_BLOCKS][2];
    __shared__ unsigned long long s_best[W][CV_BLOCKS]; /* bits of the smallest sum, then its candidate */
    __shared__ __attribute__((aligned(4))) unsigned char s_bytes[W][CV_BLOCKS * Q5_BYTES];
    const uint32_t L = threadIdx.x & 63u, w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint64_t first = ((uint64_t)blockIdx.x * W + w) * CV_BLOCKS;
    if (first >= blocks) return; /* no barrier below */
    const uint32_t b0 = (uint32_t)first, left = blocks - b0, slot = L / 8, t = L % 8;
    float *xs = s_x[w];
    double *exact = s_exact[w];
    unsigned long long *best = s_best[w];
    unsigned char *bytes = s_bytes[w];

    uint32_t row = b0 / nb, col = b0 - row * nb + slot; /* scalar, then this lane's block */
    if (nb >= 8) { /* slot < 8: at most one row further */
        row += col >= nb;
        col -= col >= nb ? nb : 0;
    } else {
        row += col / nb;
        col %= nb;
    }
    const uint32_t c = col * 32 + 4 * t;
    const bool live = slot < CV_BLOCKS && slot < left;
    const float *src = x + (size_t)row * cols + c;
    f4v v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (quad) {
        if (live && c < cols) v = *(const f4v *)src;
    } else {
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if (live && c + i < cols) v[i] = src[i];
    }
    /* the signed extreme: largest |x|, first on ties (kernels.c:1090-1091); a NaN never wins
     * (fabsf(NaN) > m is false there), so it enters as -1 and an all-NaN block keeps extreme 0 */
    float m = -1.0f, own = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const float av = fabsf(v[i]);
        own = av > m ? v[i] : own;
        m = av > m ? av : m;
    }
    float m8 = m, o = dpp_f<0xB1>(m8); /* the block's eight lanes */
    m8 = o > m8 ? o : m8;
    o = dpp_f<0x4E>(m8);
    m8 = o > m8 ? o : m8;
    o = dpp_f<0x141>(m8);
    m8 = o > m8 ? o : m8;
    const uint32_t at = (uint32_t)(__ballot(m == m8) >> (8 * slot)) & 255u;
    const float e8 = __shfl(own, (int)(8 * slot + (uint32_t)__builtin_ctz(at | 256u)), 64);
    const float extreme8 = m8 > 0.0f ? e8 : 0.0f; /* this lane's block's */
    if (slot < CV_BLOCKS) *(f4v *)&xs[slot * CV_PITCH + 4 * t] = v;
    if (L < CV_BLOCKS) best[L] = ~0ull;
    wave_sync();

    auto diff = [&](float e, float d, float dinv) __attribute__((always_inline)) {
        const float q = __builtin_amdgcn_fmed3f(__builtin_rintf(e * dinv), -16.0f, 15.0f);
        return __builtin_fmaf(-q, d, e);
    };
    /* the sums in binary32 (a NaN element makes every kept candidate's sum NaN; the zeros past a short
     * block's end add zeros), then the first minimum over the kept candidates, as
     * `best < 0 || err < best` (kernels.c:1099): the first kept one is taken whatever its error, so NaN sums
     * leave the first kept candidate */
    const uint32_t kb = L / CV_K, k = L - kb * CV_K; /* lane 63: no candidate */
    float err[ROUNDS], dk[ROUNDS], ik[ROUNDS]; /* sum, scale and its inverse */
#pragma unroll
    for (uint32_t r = 0; r < ROUNDS; ++r) {
        const uint32_t s = 3 * r + (kb < 3 ? kb : 2);
        const float extreme = __shfl(extreme8, (int)(8 * s), 64);
        float d = half_to_float(q5_candidate(extreme, k));
        asm("" : "+v"(d)); /* a binary32 register, not a half operand of every fma */
        const bool kept = kb < 3 && extreme != 0.0f && d != 0.0f && fabsf(d) <= FLT_MAX;
        const float dinv = 1.0f / d;
        float acc = 0.0f;
        const f4v *x4 = (const f4v *)&xs[s * CV_PITCH];
#pragma unroll
        for (uint32_t g = 0; g < 8; ++g) {
            const f4v xv = x4[g];
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                const float de = diff(xv[i], d, dinv);
                acc = __builtin_fmaf(de, de, acc);
            }
        }
        err[r] = kept ? acc : -1.0f; /* skipped: no sum of squares is -1 */
        dk[r] = d;
        ik[r] = dinv;
        const uint32_t bits = acc == acc ? __float_as_uint(acc) : 0x7fc00000u;
        if (kept) atomicMin(&best[s], (unsigned long long)bits << 32 | k);
    }
    wave_sync();
    bool near[ROUNDS], close = false;
#pragma unroll
    for (uint32_t r = 0; r < ROUNDS; ++r) {
        const unsigned long long key = best[3 * r + (kb < 3 ? kb : 2)];
        const float wide = __uint_as_float((uint32_t)(key >> 32)) * (1.0f + 0x1p-17f), lim = wide < 0x1p-99f ? 0x1p-99f : wide;
        near[r] = err[r] >= 0.0f && err[r] <= lim;
        close |= near[r] && k != (uint32_t)key;
    }
    if (__ballot(close)) { /* uniform: in element order, as the reference sums */
#pragma unroll
        for (uint32_t r = 0; r < ROUNDS; ++r) {
            const uint32_t s = 3 * r + (kb < 3 ? kb : 2);
            double acc = 0.0;
#pragma unroll 8
            for (uint32_t i = 0; i < 32; ++i) {
                const double de = (double)diff(xs[s * CV_PITCH + i], dk[r], ik[r]);
                acc = __builtin_fma(de, de, acc);
            }
            if (kb < 3) exact[s * CV_K + k] = near[r] ? acc : -1.0;
        }
        wave_sync();
        if (L < CV_BLOCKS) {
            double low = -1.0;
            uint32_t win = CV_K;
            for (uint32_t i = 0; i < CV_K; ++i) {
                const double e = exact[L * CV_K + i];
                if (e != -1.0 && (low < 0.0 || e < low)) {
                    low = e;
                    win = i;
                }
            }
            if (win < CV_K) best[L] = win;
        }
        wave_sync();
    }

    /* pack: high plane bit j = bit 4 of code j; byte 6 + j (j < 16) = code j | code j+16 << 4 */
#pragma unroll
    for (uint32_t r = 0; r < ROUNDS; ++r) { /* the winner's lane leaves its scale and inverse */
        const uint32_t s = 3 * r + kb;
        if (kb < 3 && k == (uint32_t)best[s]) {
            s_scale[w][s][0] = dk[r];
            s_scale[w][s][1] = ik[r];
        }
    }
    wave_sync();
    const bool won = slot < CV_BLOCKS && (uint32_t)best[slot] < CV_K; /* else no scale was kept */
    const uint32_t ss = slot < CV_BLOCKS ? slot : 0;
    const float inv = won ? s_scale[w][ss][1] : 0.0f;
    const uint32_t half = won ? to_half_bits(s_scale[w][ss][0]) : 0u;
    uint32_t low = 0, high = 0;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t q = (uint32_t)((c + i < cols && inv != 0.0f ? q5_level(v[i], inv) : 0) + 16);
        low |= (q & 15u) << (8 * i);
        high |= (q >> 4) << (4 * t + i);
    }
    high = or_dpp<0x141>(or_dpp<0x4E>(or_dpp<0xB1>(high)));
    const uint32_t word = low | __shfl_down(low, 4, 8) << 4; /* of lanes 0-3 */
    if (slot < CV_BLOCKS) {
        uint16_t *o16 = (uint16_t *)(bytes + slot * Q5_BYTES);
        if (t < 4) {
            o16[3 + 2 * t] = (uint16_t)word;
            o16[4 + 2 * t] = (uint16_t)(word >> 16);
        } else if (t == 4) {
            o16[0] = (uint16_t)half;
        } else if (t < 7) {
            o16[t - 4] = (uint16_t)(high >> (16 * (t - 5)));
        }
    }
    wave_sync();
    const uint32_t n = (left < CV_BLOCKS ? left : CV_BLOCKS) * Q5_BYTES;
    unsigned char *dst = out + (size_t)b0 * Q5_BYTES;
    if (ROUNDS == 2 && ((uintptr_t)out & 3u) == 0) { /* b0 * 22 is a multiple of 132 */
        if (L < n / 4) ((uint32_t *)dst)[L] = ((const uint32_t *)bytes)[L];
        else if (L == n / 4 && n % 4) *(uint16_t *)(dst + (n & ~3u)) = *(const uint16_t *)(bytes + (n & ~3u));
    } else if (ROUNDS == 1 && ((uintptr_t)out & 1u) == 0) { /* 66 bytes */
        if (L < n / 2) ((uint16_t *)dst)[L] = ((const uint16_t *)bytes)[L];
    } else {
        for (uint32_t i = L; i < n; i += 64) dst[i] = bytes[i];
    }
}

}  // namespace

template <uint32_t ROUNDS>
static hipError_t launch_q5_rounds(const float *x, uint32_t blocks, uint32_t cols, bool quad, unsigned char *out, hipStream_t s) {
    constexpr uint32_t per = 3 * ROUNDS * (CV_WG / 64);
    hipLaunchKernelGGL(k_quantize_q5<ROUNDS>, dim3((uint32_t)(((uint64_t)blocks + per - 1) / per)), dim3(CV_WG), 0, s, x, blocks,
                       (cols + 31) / 32, cols, quad, out);
    return hipGetLastError();
}

hipError_t launch_quantize_q5(const float *x, uint32_t rows, uint32_t cols, unsigned char *out, hipStream_t s) {
    const uint64_t blocks = (uint64_t)rows * ((cols + 31) / 32);
    if (!blocks) return hipSuccess;
    const bool quad = cols % 4 == 0 && ((uintptr_t)x & 15u) == 0;
    if (blocks > 0xffffffffu) return hipErrorInvalidValue; /* more than the device memory holds */
    /* one round while about four such waves per SIMD hold every block. Measured on MI355X (us, one round / two): 1 block
     * 2.8 / 3.3, 500 4.3 / 5.3, 5000 4.7 / 5.6, 20000 6.5 / 7.0, 30000 8.25 / 8.2, 50000 11.2 / 10.1 */
    if (blocks <= 28000) return launch_q5_rounds<1>(x, (uint32_t)blocks, cols, quad, out, s);
    return launch_q5_rounds<2>(x, (uint32_t)blocks, cols, quad, out, s);
}

}  // namespace smq

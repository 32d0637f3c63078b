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
 * Mapping: a workgroup takes 24 consecutive blocks. Half a wave per block finds the
 * extreme; then a lane per (block, candidate), 504 of them in two rounds over the 256
 * threads, runs the binary64 sum over the block's elements in LDS; one lane per block
 * picks the winner; half a wave per block quantizes and packs into LDS, and the 528
 * bytes go out as words.
 *
 * What bounds it is the 21 x 32 terms per block, so a term is as short as its value
 * allows. q * d is exact in binary32 (5 and 11 significant bits). x - q * d is exact too:
 * for q = 0 it is x; otherwise x lies within a factor of two of q * d (Sterbenz). For
 * |q| >= 2 and the clamped ends that is plain: |x / d| is at most 24.75, even where d is
 * a subnormal half. For |q| = 1, rint gave 1, so p = fl(x * dinv) is at least 1/2 + 2^-24
 * and, with both roundings below 2^-24, x / d at least 1/2 (1 - 2^-48): as x and d / 2 are
 * binary32 numbers, x >= d / 2. The square of a binary32 number is exact in binary64, so
 * one fused multiply-add is the reference's square, then sum. A term is four binary32
 * operations, a conversion and that fma. 8960 x 1536: 253.4 us with half a wave per block (21 of 32 lanes) and four
 * binary64 operations a term -> 71.2 us.
 */
#include <float.h>

#include "smq_device.h"
#include "smq_internal.h"

namespace smq {
namespace {

constexpr uint32_t CV_WG = 256;
constexpr uint32_t CV_BLOCKS = 24; /* 21 candidates of each: 504 lanes of two rounds */
constexpr uint32_t CV_K = 21;
constexpr uint32_t CV_PITCH = 36; /* floats per block: a wave's three or four blocks on distinct banks */

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

__global__ __launch_bounds__(CV_WG) void k_quantize_q5(const float *x, uint32_t blocks, uint32_t nb, uint32_t cols,
                                                       unsigned char *out) {
    __shared__ __attribute__((aligned(16))) float xs[CV_BLOCKS * CV_PITCH];
    __shared__ double errs[CV_BLOCKS * CV_K];
    __shared__ float ext[CV_BLOCKS], winv[CV_BLOCKS];
    __shared__ uint32_t whalf[CV_BLOCKS];
    __shared__ __attribute__((aligned(4))) unsigned char bytes[CV_BLOCKS * Q5_BYTES];
    const uint32_t tid = threadIdx.x, j = tid % 32, b0 = blockIdx.x * CV_BLOCKS;
    constexpr uint32_t U = CV_BLOCKS * 32 / CV_WG;
    float v[U];
    bool valid[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
        const uint32_t blk = b0 + u * (CV_WG / 32) + tid / 32, row = blk / nb, c = (blk - row * nb) * 32 + j;
        valid[u] = blk < blocks && c < cols;
        v[u] = valid[u] ? x[(size_t)row * cols + c] : 0.0f;
    }
    /* the signed extreme: largest |x|, first on ties (kernels.c:1090-1091); a NaN never wins
     * (fabsf(NaN) > m is false there), so it enters as -1 and an all-NaN block keeps extreme 0 */
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
        const uint32_t slot = u * (CV_WG / 32) + tid / 32;
        xs[slot * CV_PITCH + j] = v[u];
        const float av = v[u] == v[u] ? fabsf(v[u]) : -1.0f, m = max32(av);
        const uint64_t at = __ballot(av == m);
        const uint32_t first = (uint32_t)__builtin_ctz((uint32_t)((tid & 63u) < 32 ? at : at >> 32));
        const float e = __shfl(v[u], (int)first, 32);
        if (j == 0) ext[slot] = m > 0.0f ? e : 0.0f;
    }
    __syncthreads();

    /* error sums in element order (a NaN element makes every kept candidate's sum NaN; the zeros past a
     * short block's end add zeros) */
    for (uint32_t id = tid; id < CV_BLOCKS * CV_K; id += CV_WG) {
        const uint32_t slot = id / CV_K, k = id - slot * CV_K;
        const float extreme = ext[slot];
        double err = -1.0; /* skipped: no sum of squares is -1 */
        const float d = half_to_float(q5_candidate(extreme, k));
        if (extreme != 0.0f && d != 0.0f && fabsf(d) <= FLT_MAX) {
            const float dinv = 1.0f / d;
            const float4 *x4 = (const float4 *)&xs[slot * CV_PITCH];
            double acc = 0.0;
#pragma unroll
            for (uint32_t g = 0; g < 8; ++g) {
                const float4 xv = x4[g];
                const float e4[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) {
                    const float q = __builtin_amdgcn_fmed3f(__builtin_rintf(e4[i] * dinv), -16.0f, 15.0f);
                    const double de = (double)__builtin_fmaf(-q, d, e4[i]);
                    acc = __builtin_fma(de, de, acc);
                }
            }
            err = acc;
        }
        errs[id] = err;
    }
    __syncthreads();
    /* first minimum over the kept candidates, as `best < 0 || err < best` (kernels.c:1099): the
     * first kept one is taken whatever its error, so NaN sums leave the first kept candidate */
    if (tid < CV_BLOCKS) {
        uint32_t win = CV_K;
        double best = -1.0;
#pragma unroll
        for (uint32_t k = 0; k < CV_K; ++k) {
            const double e = errs[tid * CV_K + k];
            if (e != -1.0 && (best < 0.0 || e < best)) {
                best = e;
                win = k;
            }
        }
        const uint32_t h = win < CV_K ? q5_candidate(ext[tid], win) : 0u;
        whalf[tid] = h;
        winv[tid] = win < CV_K ? 1.0f / half_to_float(h) : 0.0f; /* 0: no scale was kept */
    }
    __syncthreads();

    /* pack: high plane bit j = bit 4 of code j; byte 6 + j (j < 16) = code j | code j+16 << 4 */
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
        const uint32_t slot = u * (CV_WG / 32) + tid / 32;
        const float inv = winv[slot];
        const uint32_t q = (uint32_t)((valid[u] && inv != 0.0f ? q5_level(v[u], inv) : 0) + 16);
        const uint64_t hb = __ballot((q >> 4) & 1u);
        const uint32_t high = (uint32_t)((tid & 63u) < 32 ? hb : hb >> 32), half = whalf[slot];
        const uint32_t upper = __shfl_down(q, 16, 32);
        unsigned char *o = bytes + slot * Q5_BYTES;
        if (j < 16) o[6 + j] = (unsigned char)((q & 15u) | ((upper & 15u) << 4));
        else if (j < 18) o[j - 16] = (unsigned char)(half >> (8 * (j - 16)));
        else if (j < 22) o[2 + (j - 18)] = (unsigned char)(high >> (8 * (j - 18)));
    }
    __syncthreads();
    const uint32_t live = (blocks - b0 < CV_BLOCKS ? blocks - b0 : CV_BLOCKS) * Q5_BYTES;
    unsigned char *o = out + (size_t)b0 * Q5_BYTES;
    if (((uintptr_t)out & 3u) == 0) { /* b0 * 22 is a multiple of 528 */
        if (tid < live / 4) ((uint32_t *)o)[tid] = ((const uint32_t *)bytes)[tid];
        else if (tid == live / 4 && live % 4) *(uint16_t *)(o + (live & ~3u)) = *(const uint16_t *)(bytes + (live & ~3u));
    } else {
        for (uint32_t i = tid; i < live; i += CV_WG) o[i] = bytes[i];
    }
}

}  // namespace

hipError_t launch_quantize_q5(const float *x, uint32_t rows, uint32_t cols, unsigned char *out, hipStream_t s) {
    const uint64_t blocks = (uint64_t)rows * ((cols + 31) / 32);
    if (!blocks) return hipSuccess;
    const uint64_t grid = (blocks + CV_BLOCKS - 1) / CV_BLOCKS;
    if (blocks > 0xffffffffu - CV_BLOCKS) return hipErrorInvalidValue; /* more than the device memory holds */
    hipLaunchKernelGGL(k_quantize_q5, dim3((uint32_t)grid), dim3(CV_WG), 0, s, x, (uint32_t)blocks, (cols + 31) / 32, cols,
                       out);
    return hipGetLastError();
}

}  // namespace smq

// cgh_common.hpp -- outputs and helpers shared by the direct CGH kernels (olx_cgh.hip) and
// the matrix-core Fresnel form (olx_cgh_mfma.hip).
#pragma once
#include "img_common.hpp"
#include "olx_common.hpp"

namespace olx {

// The outputs of a CGH kernel, any of them null: the field (added to what U holds
// with accumulate), its phase atan2(im, re), its amplitude, and the phase8bit byte of
// that phase (include/olimg.h:205-213; img_offset: the +pi form) fused into the
// epilogue in place of a phase array and a second pass.
struct CghOut {
    float2* U;
    float* phase;
    float* amp;
    uint8_t* img;
    int img_offset;
    int accumulate;
};

__device__ __forceinline__ void cgh_store(const CghOut& o, size_t idx, float2 v) {
    if (o.accumulate && o.U) {
        const float2 q = o.U[idx];
        v = make_float2(v.x + q.x, v.y + q.y);
    }
    if (o.U) o.U[idx] = v;
    if (o.phase || o.img) {
        const float ph = atan2f(v.y, v.x);
        if (o.phase) o.phase[idx] = ph;
        if (o.img) o.img[idx] = phase8_one<float>(ph, o.img_offset);
    }
    if (o.amp) o.amp[idx] = sqrtf(v.x * v.x + v.y * v.y);
}

// sin / cos of t revolutions: the hardware units take revolutions; t is first
// reduced to [0, 1) with one v_fract (exact for a float)
__device__ __forceinline__ void sincos_rev(float t, float* s, float* c) {
    t = __builtin_amdgcn_fractf(t);
    *s = __builtin_amdgcn_sinf(t);
    *c = __builtin_amdgcn_cosf(t);
}

// Partial maxima of |amp| over the cloud (olx_cgh_mfma.hip), as float bits
constexpr int AMP_PARTS = 64;
// the cloud's maximum, taken by every lane of a wave from the AMP_PARTS partials
__device__ __forceinline__ uint32_t amp_max(const uint32_t* __restrict__ parts) {
    uint32_t m = parts[threadIdx.x & 63];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 64));
    return m;
}
constexpr uint32_t AMP_INF = 0x7f800000u;  // at or above: an infinite or NaN amplitude

constexpr int FAC_EXP = 5;  // 16-bit factors are scaled to at most 2^FAC_EXP
// exponent of the power of two that amplitudes are multiplied by: the largest goes below 2^FAC_EXP
__device__ __forceinline__ int amp_exp(uint32_t mx) { return min(126, FAC_EXP + 126 - (int)(mx >> 23)); }
__global__ void k_amp_parts(const olx_point* pts, int n, uint32_t* parts);
// adds S planes of np values in order, undoes the scaling of both factors and stores the outputs
__global__ void k_cgh_sum_scaled(const float2* part, int S, int64_t np, CghOut o, const uint32_t* amp_parts);

// The Fresnel sum on the matrix cores; under capture, where its workspace could not grow, it leaves the call
// to the vector kernels.  *done tells whether it ran; then *amp_parts are the
// AMP_PARTS partials, and an infinite or NaN maximum leaves the outputs unwritten for the
// separable kernel (olx_cgh_mfma.hip).
int cgh_fresnel_mfma(olx_ctx* ctx, const olx_point* d_pts, int64_t n, const CghOut& o, int64_t ny,
                     int64_t nx, double py, double px, double lambda, bool* done,
                     const uint32_t** amp_parts);
// Points that the exact-r sum on the matrix cores leaves, in the 64 x 64 tile at (w0, h0), to the
// per-pixel kernel: the condition of olx_cgh_exact.hip, each operation rounded, so that the two
// kernels agree.
constexpr int EXT = 64;            // tile side; points a block
// Largest cross phase, radians.  The first term left out, eps^4 / 24, is 8.6e-6 of a point's term at the tile's corner
// there (and grows with the fourth power: 1e-4 at 0.22).  Clouds of 600 points just below it (128 x 128, z = 1 mm
// to 0.3 m, pitch 1 to 8 um, 405 and 633 nm) are as near to FP64 as with the per-pixel kernel or nearer, in norm
// and at the worst pixel; at 0.15 the worst pixel was up to 1.7 times as far off (z = 10 mm), at 0.22 4.4 times.
constexpr double EX_EPS = 0.12;
constexpr double EX_E4K = 1.0e-6;  // (5/128) e^4 r0 / lambda <= 4e-8 cycles
__device__ __forceinline__ bool ex_near(const olx_point& p, int w0, int h0, double py, double px, double lambda) {
#pragma clang fp contract(off)
    const double dx = px * (w0 + EXT / 2) - p.x, dy = py * (h0 + EXT / 2) - p.y;
    const double hx = EXT / 2 * px, hy = EXT / 2 * py;
    const double r2 = dx * dx + dy * dy + p.z * p.z, rl = sqrt(r2) / lambda, i2 = 1.0 / r2;
    const double e1 = (2.0 * fabs(dx) * hx + hx * hx) * i2, e2 = (2.0 * fabs(dy) * hy + hy * hy) * i2;
    const double em = fmax(e1, e2), em2 = em * em;
    return !(em <= 0.01 && em2 * em2 * rl <= EX_E4K && 0.5 * M_PI * rl * e1 * e2 <= EX_EPS);
}
// What that sum leaves of a tile and slice: nothing, the points of ex_near, or all points
constexpr uint32_t EX_NONE = 0, EX_SOME = 1, EX_ALL = 2;
// What that sum leaves (olx_cgh.hip), added to the S planes of `slice` points each; all points, into the
// outputs, of a cloud with an infinite or NaN amplitude.  parts: the AMP_PARTS maxima, and after them a word a
// tile and slice.
void cgh_exact_rest(hipStream_t s, const olx_point* d_pts, int64_t n, const CghOut& o, int64_t ny, int64_t nx,
                    double py, double px, double lambda, float2* part, int S, int slice, const uint32_t* parts);
// the exact-r sum (olx_cgh_exact.hip)
int cgh_exact_mfma(olx_ctx* ctx, const olx_point* d_pts, int64_t n, const CghOut& o, int64_t ny, int64_t nx,
                   double py, double px, double lambda, bool* done);

}  // namespace olx

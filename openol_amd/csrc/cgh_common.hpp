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

// The Fresnel sum on the matrix cores.  *done tells whether it ran; then *amp_parts are the
// AMP_PARTS partials, and an infinite or NaN maximum leaves the outputs unwritten for the
// separable kernel (olx_cgh_mfma.hip).
int cgh_fresnel_mfma(olx_ctx* ctx, const olx_point* d_pts, int64_t n, const CghOut& o, int64_t ny,
                     int64_t nx, double py, double px, double lambda, bool* done,
                     const uint32_t** amp_parts);

}  // namespace olx

// olx_cgh_mfma.hip -- the direct Fresnel CGH on the matrix cores.
//
// theta = c (px w - x_j)^2 + phi_j / 2 pi + c (py h - y_j)^2, c = 1 / (2 lambda z_j), separates,
// so U = Y X^T with X_j(w) = A_j e^{2 pi i (c (px w - x_j)^2 + phi_j / 2 pi)} and
// Y_j(h) = e^{2 pi i c (py h - y_j)^2}: one complex product over the points (mfma_gemm.hpp).
//
// Each factor's phase is taken in FP64 and its sine / cosine by the hardware unit, in FP32;
// the value is then split into FP16 hi + lo.  Scaled so that the largest is near 32, lo
// (at most 2^-7) stays a normal FP16 number with 2^-18 spacing, so hi + lo is off by at most
// 2^-19 of 32, that is 2^-24: the rounding of an FP32 value.  The dropped lo lo product is
// below 2^-24 too.  The largest amplitude (a power of two above it) is divided out of X and
// multiplied back exactly at the end, so any finite FP32 amplitudes are taken; a cloud with an
// infinite or NaN amplitude is left to the separable kernel.  Sums run in FP32 over at most
// FAC_CHAIN points and are added and subtracted in turn (mfma_gemm.hpp); slices' planes are added in FP64.
//
// Why matrix cores: the separable kernel spends 6.25 vector operations per point and pixel at 92%
// of the issue peak, 5.8 Tpt px/s.  The three FP16 products cost 24 flop per point and pixel on a
// unit that gives 1.2 PFLOP/s here.  Measured: 5,197 points into 1080 x 1920 1865 -> 311 us (2.0e-6
// -> 4.0e-7 off FP64), 10,000 into 2048^2 7.26 -> 0.96 ms, 5,197 into 300 x 400 1207 -> 56 us.
// The product is 277 us of the 311, the factors 21, the planes' sum 13.
#include "cgh_common.hpp"
#include "mfma_gemm.hpp"

namespace olx {

// Points summed in one FP32 accumulator.  5197 points into 1080 x 1920 and the error of 20,000 into
// 500^2 (3.74 um; the separable kernel's is 4.7e-7): runs of 1024 303 us, 4.9e-7; 768 328, 4.3e-7; 640 329; 512 349,
// 3.7e-7.
constexpr int FAC_CHAIN = 640;
constexpr int FAC_RB = 16;       // factor rows per thread

__global__ void __launch_bounds__(1024)
k_amp_parts(const olx_point* __restrict__ pts, int n, uint32_t* __restrict__ parts) {
    __shared__ uint32_t wm[16];
    uint32_t m = 0;
    for (int64_t j = blockIdx.x * 1024 + threadIdx.x; j < n; j += AMP_PARTS * 1024)
        m = max(m, __float_as_uint(pts[j].amp) & 0x7fffffffu);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 64));
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; w++) m = max(m, wm[w]);
        parts[blockIdx.x] = m;
    }
}

// Factor rows of points [j0, j0 + kc), in the split row layout (ldw 32-bit words a row): row
// blocks [0, yb) are Y's (h, as A: Re, Im), the others X's (w, as Br: Re, -Im).  A thread
// owns one point and FAC_RB consecutive rows; 16 lanes write 64 contiguous bytes of hi and of
// lo, the 256 threads of a group 2 KiB a row.
__global__ void __launch_bounds__(256)
k_cgh_factors(const olx_point* __restrict__ pts, int j0, int n, int kc, double py, double px,
              double lambda, int ny, int nx, int yb, uint32_t* __restrict__ Y, uint32_t* __restrict__ X,
              int ldw, const uint32_t* __restrict__ amp_parts, int kslice) {
    const uint32_t mx = amp_max(amp_parts);
    if (mx >= AMP_INF) return;
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= kc) return;
    const bool isy = (int)blockIdx.y < yb;
    const int rb = ((int)blockIdx.y - (isy ? 0 : yb)) * FAC_RB;
    const int rows = isy ? ny : nx;
    double c = 0.0, p0 = 0.0, ph = 0.0;
    float amp = 0.f;  // points past the cloud's end add nothing
    if (j0 + j < n) {
        const olx_point p = pts[j0 + j];
        c = 1.0 / (2.0 * lambda * p.z);
        p0 = isy ? p.y : p.x;
        // half a cycle more in the runs that the product subtracts
        constexpr int SP = stage_pts<true>();
        const int st = j / SP, z = st / kslice, odd = (z + (st - z * kslice) / (FAC_CHAIN / SP)) & 1;
        ph = isy ? 0.0 : (double)p.phase * (0.5 / M_PI) + 0.5 * odd;
        amp = isy ? ldexpf(1.f, FAC_EXP) : ldexpf(p.amp, amp_exp(mx));
    }
    const double d = isy ? py : px;
    const float sgn = isy ? amp : -amp;
    uint32_t* out = (isy ? Y : X) + (size_t)rb * ldw + fac_word<true>(j);
    const int nr = min(FAC_RB, rows - rb);
    for (int q = 0; q < nr; q++) {
        const double x = d * (rb + q) - p0;
        double th = fma(c * x, x, ph);
        th -= rint(th);
        const float t = (float)th;
        const float re = amp * __builtin_amdgcn_cosf(t), im = sgn * __builtin_amdgcn_sinf(t);
        float hr, hi, lr, li;
        out[0] = pack2<_Float16>(re, im, &hr, &hi);
        out[16] = pack2<_Float16>(re - hr, im - hi, &lr, &li);
        out += ldw;
    }
}

// adds the slices' planes in slice order, in FP64 (64 FP32 sums added 1.4e-7), undoes the scaling and stores the
// outputs
__global__ void __launch_bounds__(256)
k_cgh_sum_scaled(const float2* __restrict__ part, int S, int64_t np, CghOut o,
                 const uint32_t* __restrict__ amp_parts) {
    const uint32_t mx = amp_max(amp_parts);
    if (mx >= AMP_INF) return;
    const int e = -FAC_EXP - amp_exp(mx);
    for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < np; i += (int64_t)gridDim.x * 256) {
        double x = 0.0, y = 0.0;
        for (int s = 0; s < S; s++) {
            const float2 w = part[(size_t)s * np + i];
            x += w.x;
            y += w.y;
        }
        cgh_store(o, (size_t)i, make_float2(ldexpf((float)x, e), ldexpf((float)y, e)));
    }
}

int cgh_fresnel_mfma(olx_ctx* ctx, const olx_point* d_pts, int64_t n, const CghOut& o, int64_t ny,
                     int64_t nx, double py, double px, double lambda, bool* done,
                     const uint32_t** amp_parts) {
    *done = false;
    // The separable kernel takes 0.43 us a point where its tiles do not fill the GPU and 5.8
    // point-pixel pairs a ps where they do; this form's five launches take about 33 us plus
    // 24 bytes a pixel of planes at 5 TB/s before any product (both in us here).  Measured on
    // either side: 284 points, 512^2: 127 us there, 31 here; 64 points, 512^2: 29 there, 30 here.
    // Sides above 32768 keep the kernel that needs no workspace.
    const double px_n = (double)ny * (double)nx;
    const double t_sep = std::max(0.43 * n, n * px_n / 5.8e6), t_mfma = 33.0 + px_n * 24.0 / 5.0e6;
    if (ny > 32768 || nx > 32768 || t_sep <= t_mfma || capturing(ctx->stream)) return OLX_OK;
    auto up = [](int64_t v, int64_t m) { return (v + m - 1) / m * m; };
    constexpr int SP = stage_pts<true>();
    const size_t np = (size_t)ny * (size_t)nx;
    const int64_t rows = up(ny, 256) + up(nx, GTN);
    // chunks of points: factors of at most 1 GiB (8 bytes per row and point)
    const int64_t kmax = std::max<int64_t>(FAC_CHAIN, ((int64_t)1 << 30) / (8 * rows) / SP * SP);
    const int64_t nchunk = (n + kmax - 1) / kmax;
    const int kc = (int)up((n + nchunk - 1) / nchunk, SP), stages = kc / SP;
    // partial planes of at most 2 GiB
    const int smax = (int)std::min<size_t>(64, ((size_t)2 << 30) / (sizeof(float2) * np));
    if (smax < 1) return OLX_OK;
    const GemmPlan g = gemm_plan(ny, nx, stages, true, smax, 0.0);
    const int ldk = 4 * kc;
    const size_t ybytes = sizeof(uint16_t) * (size_t)up(ny, 64 * g.wr) * ldk;
    const size_t xbytes = sizeof(uint16_t) * (size_t)up(nx, GTN) * ldk;
    if (spare(ctx, ctx->lay_counts, ybytes + xbytes + sizeof(uint32_t) * AMP_PARTS) != OLX_OK ||
        spare(ctx, ctx->cgh_part, sizeof(float2) * np * (size_t)g.slices) != OLX_OK)
        return OLX_OK;  // no room for the workspace: the separable kernel needs none
    uint32_t* Y = (uint32_t*)ctx->lay_counts.p;
    uint32_t* X = (uint32_t*)((char*)ctx->lay_counts.p + ybytes);
    uint32_t* parts = (uint32_t*)((char*)ctx->lay_counts.p + ybytes + xbytes);
    float2* part = (float2*)ctx->cgh_part.p;
    hipStream_t s = ctx->stream;
    TimedLaunch tl(ctx, "cgh_f32_fresnel");
    k_amp_parts<<<AMP_PARTS, 1024, 0, s>>>(d_pts, (int)n, parts);
    const int yb = (int)((ny + FAC_RB - 1) / FAC_RB), xb = (int)((nx + FAC_RB - 1) / FAC_RB);
    for (int64_t j0 = 0, c = 0; j0 < n; j0 += kc, c++) {
        const int kn = (int)std::min<int64_t>(kc, up(n - j0, SP)), st = kn / SP;
        k_cgh_factors<<<dim3((unsigned)((kn + 255) / 256), (unsigned)(yb + xb)), 256, 0, s>>>(
            d_pts, (int)j0, (int)n, kn, py, px, lambda, (int)ny, (int)nx, yb, Y, X, ldk / 2, parts, g.kslice);
        cgemm<_Float16, true>(s, g.wr, (st + g.kslice - 1) / g.kslice, Y, X, ldk, st, g.kslice,
                              FAC_CHAIN / SP, part, np, ny, nx, c > 0, 4, 1);
    }
    const int64_t blocks = std::min<int64_t>(((int64_t)np + 255) / 256, 65536);
    k_cgh_sum_scaled<<<(unsigned)blocks, 256, 0, s>>>(part, g.slices, (int64_t)np, o, parts);
    *done = true;
    *amp_parts = parts;
    return check_launch("cgh fresnel (matrix cores)");
}

}  // namespace olx

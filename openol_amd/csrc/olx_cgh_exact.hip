// olx_cgh_exact.hip -- the direct exact-r CGH on the matrix cores.
//
// Over a tile of pixels around (w0, h0), with X = r^2 along x minus r0^2 (at v = 0), Y along y:
//   r = sqrt(r0^2 + X + Y) = sqrt(r0^2 + X) + sqrt(r0^2 + Y) - r0 - (r0 / 4) a b + ...,
//   e1 = X / r0^2, a = e1 (1 - 3/4 e1), and b from e2 = Y / r0^2 alike,
// exact to third order in e.  The separable part gives one factor a column and one a row, and the
// cross term's phase, eps = -(pi r0 / 2 lambda) a b, is small over 64 x 64 pixels, so
//   exp(i eps) = sum_m (i p)^m q^m / m!,   p q = eps,
// and the tile is a product over (point, m), m < 4: U = sum_m Y_m X_m^T with X_m = X_0 (i p)^m and
// Y_m = Y_0 q^m / m!.  A wave owns the tile and forms the factors in registers, in the lane layout of
// its matrix operands: 128 phases a point in place of 4096.
//
// Precision.  Phases: r0 / lambda and the slope per pixel in FP64, reduced mod 1 (pixel offsets are
// integers); the slope's upper 18 bits times the offset are exact in FP32, the rest of the phase is
// below about a cycle.  m = 0 and 1 are carried as FP16 hi + lo (three products, 2^-24 as in
// olx_cgh_mfma.hip), m = 2 and 3, at most 0.7% of m = 0 and far less mostly, as one FP16 value.  A
// point is taken this way in a tile where |eps| <= EX_EPS at the tile's corner and the one-axis series ends
// below 4e-8 cycles; the others (ex_near: near field, wide angles) are left to
// k_cgh_exact, which adds them to the same planes.
//
// Bound by the vector work of the factors (about 580 instructions for 8 points and 64 matrix
// instructions, with the sums of the runs 71% of the issue slots, the matrix unit 46% busy) at the
// clock this mix leaves (1.85 GHz).  10,000 points into 2048^2: 12200 us with the per-pixel kernel (10.8
// vector operations a point and pixel, 94% of the issue peak, 3.8e-6 off FP64), 3060 here (4.5e-7; 85
// of them the points left to the per-pixel kernel); 5000 into 1080 x 1920 3190 -> 740, 20,000 into 300 x 300
// 789 -> 167; a cloud of near points only (2000, 2160^2, z 2 to 10 mm) 8350 -> 8110.
#include <algorithm>

#include "cgh_common.hpp"
#include "mfma_gemm.hpp"

namespace olx {

// Points summed in one FP32 accumulator; runs of them are added and subtracted in turn (mfma_gemm.hpp).  10,000
// points into 2048^2 and the error of 20,000 into 500^2 (3.74 um; the per-pixel kernel's is 4.0e-7): runs of 1024 2985 us,
// 4.8e-7; 512 3100, 4.0e-7; 256 3260, 3.2e-7; 128 3630.
constexpr int EX_CHAIN = 256;

struct ExAxis {  // phase along one axis at pixel offset i: sh i mod 1 + i (sl + c2 i) + K8 e^2 + K16 e^3
    float sh, sl, c2, g1, g2;  // e = i (g1 + g2 i)
};
struct ExPt {    // per-(tile, point) constants; 16 floats
    ExAxis x, y;
    float ph, amp, G, K8, K16, pad;
};
__device__ __forceinline__ ExAxis ex_axis(double D, double p, double r0, double ir2, double rl) {
    ExAxis a;
    double s = D * p * ir2 * rl;  // cycles a pixel
    s -= rint(s);
    const double sh = rint(s * 262144.0) * (1.0 / 262144.0);
    a.sh = (float)sh;
    a.sl = (float)(s - sh);
    a.c2 = (float)(0.5 * p * p * ir2 * rl);
    a.g1 = (float)(2.0 * D * p * ir2);
    a.g2 = (float)(p * p * ir2);
    return a;
}

// cos and sin of the axis' phase (+ ph) at offset i, and G a(e)
template <bool PH>
__device__ __forceinline__ void ex_eval(const ExAxis& a, float K8, float K16, float G, float ph, float i,
                                        float* c, float* s, float* q) {
    const float e = i * fmaf(a.g2, i, a.g1);
    // sh i is exact; within 1/2 of zero, small slopes keep small phases, whose rounding is finer
    const float u = a.sh * i;
    float t = fmaf(i, fmaf(a.c2, i, a.sl), u - rintf(u));
    if constexpr (PH) t += ph;
    t = fmaf(e * e, fmaf(e, K16, K8), t);
    *c = __builtin_amdgcn_cosf(t);
    *s = __builtin_amdgcn_sinf(t);
    *q = G * e * fmaf(-0.75f, e, 1.f);
}

typedef _Float16 ex_half2 __attribute__((ext_vector_type(2)));
typedef float ex_float2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk16(float a, float b) {
    const ex_float2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, ex_half2));
}
// FP16 hi and lo of a word's two values; with B also of the word (-b, a), the Im product's operand
template <bool B>
__device__ __forceinline__ void ex_split(float a, float b, uint32_t* hi, uint32_t* lo, uint32_t* hb, uint32_t* lb) {
    const ex_float2 v = {a, b};
    const ex_half2 h = __builtin_convertvector(v, ex_half2);
    const float ra = fmaf((float)h[0], -1.f, a), rb = fmaf((float)h[1], -1.f, b);
    *hi = __builtin_bit_cast(uint32_t, h);
    *lo = pk16(ra, rb);
    if constexpr (B) {
        *hb = pk16(-b, a);
        *lb = pk16(-rb, ra);
    }
}
__device__ __forceinline__ uint4 ex_u4(const uint32_t* w) { return make_uint4(w[0], w[1], w[2], w[3]); }

// Grid: tiles (x), slices of the points (y).  One wave a work-group; plane y of part takes its sum, left what
// it leaves to k_cgh_exact.
__global__ void __launch_bounds__(64, 2)
k_cgh_exact_mfma(const olx_point* __restrict__ pts, int n, int slice, int tiles_x, int ny, int nx, double py,
                 double px, double lambda, float2* __restrict__ part,
                 const uint32_t* __restrict__ amp_parts, uint32_t* __restrict__ left) {
    const uint32_t mx = amp_max(amp_parts);
    if (mx >= AMP_INF) return;
    const int ae = amp_exp(mx);
    __shared__ ExPt sp[EXT];
    const int lane = threadIdx.x, li = lane & 31, hf = lane >> 5;
    const int w0 = (int)(blockIdx.x % tiles_x) * EXT, h0 = (int)(blockIdx.x / tiles_x) * EXT;
    const int beg = (int)blockIdx.y * slice, end = min(n, beg + slice);
    float2* U = part + (size_t)blockIdx.y * ny * nx;
    // a tile that more than two thirds of the first block's points are too near for is left as a whole: the
    // other third takes the vector kernel no longer than this one takes all of them
    if (3 * __popcll(__ballot(beg + lane < end && ex_near(pts[min(beg + lane, end - 1)], w0, h0, py, px, lambda))) >
        2 * min(EXT, end - beg)) {
        for (int h = h0; h < min(h0 + EXT, ny); h++)
            if (w0 + lane < nx) U[(size_t)h * nx + w0 + lane] = make_float2(0.f, 0.f);
        if (lane == 0) left[blockIdx.x * gridDim.y + blockIdx.y] = EX_ALL;
        return;
    }
    const float o0 = (float)(li - EXT / 2), o1 = (float)li;  // offsets of the two fragments' rows and columns
    f16v_t accr[2][2], acci[2][2];
    bool accumulate = false;
    unsigned long long some = 0;
    int odd = blockIdx.y & 1;  // of the runs: the other way round in every second slice
    for (int c0 = beg; c0 < end || !accumulate; c0 += EX_CHAIN) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) accr[i][j][v] = acci[i][j][v] = 0.f;
        const int c1 = min(end, c0 + EX_CHAIN);
        for (int b0 = c0; b0 < c1; b0 += EXT) {
            // one point a lane: its constants for the tile
            ExPt P = {};
            bool near = false;
            if (b0 + lane < c1) {
                const olx_point p = pts[b0 + lane];
                near = ex_near(p, w0, h0, py, px, lambda);
                if (!near) {
                    const double dx = px * (w0 + EXT / 2) - p.x, dy = py * (h0 + EXT / 2) - p.y;
                    const double r2 = dx * dx + dy * dy + p.z * p.z, r0 = sqrt(r2), ir2 = 1.0 / r2, rl = r0 / lambda;
                    P.amp = ldexpf(p.amp, ae);
                    P.x = ex_axis(dx, px, r0, ir2, rl);
                    P.y = ex_axis(dy, py, r0, ir2, rl);
                    P.K8 = (float)(-0.125 * rl);
                    P.K16 = (float)(0.0625 * rl);
                    P.G = (float)sqrt(0.5 * M_PI * rl);
                    const double th = rl + (double)p.phase * (0.5 / M_PI) + 0.5 * odd;
                    P.ph = (float)(th - rint(th));
                }
            }
            some |= __ballot(near);
            __syncthreads();  // the last block's readers
            sp[lane] = P;
            if (__ballot(P.G != 0.f) == 0) continue;
            __syncthreads();
#pragma unroll 1
            for (int k0 = 0; k0 < EXT; k0 += 8) {
                // (yr, yi): Y_m; (xr, xn): X_m's real part and minus its imaginary part
                float yr[2][4], yi[2][4], yq[2][4], xr[2][4], xn[2][4], xq[2][4];
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const ExPt& Q = sp[k0 + 4 * hf + t];
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const float o = i ? o1 : o0;
                        float c, s;
                        ex_eval<false>(Q.y, Q.K8, Q.K16, Q.G, 0.f, o, &c, &s, &yq[i][t]);
                        yr[i][t] = c * (float)(1 << FAC_EXP);
                        yi[i][t] = s * (float)(1 << FAC_EXP);
                        ex_eval<true>(Q.x, Q.K8, Q.K16, Q.G, Q.ph, o, &c, &s, &xq[i][t]);
                        xr[i][t] = c * Q.amp;
                        xn[i][t] = -(s * Q.amp);
                    }
                }
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    // A (Y), B (X, for Re) and C (X, for Im) operands, hi and lo
                    uint32_t ah[2][4], al[2][4], bh[2][4], bl[2][4], ch[2][4], cl[2][4];
#pragma unroll
                    for (int i = 0; i < 2; i++)
#pragma unroll
                        for (int t = 0; t < 4; t++) {
                            if (m > 0) {  // p = -xq: i p (xr - i xn) = p xn + i p xr
                                const float q = yq[i][t] * (1.f / m), x = xr[i][t];
                                yr[i][t] *= q;
                                yi[i][t] *= q;
                                xr[i][t] = -xq[i][t] * xn[i][t];
                                xn[i][t] = xq[i][t] * x;
                            }
                            if (m < 2) {
                                ex_split<false>(yr[i][t], yi[i][t], &ah[i][t], &al[i][t], nullptr, nullptr);
                                ex_split<true>(xr[i][t], xn[i][t], &bh[i][t], &bl[i][t], &ch[i][t], &cl[i][t]);
                            } else {
                                ah[i][t] = pk16(yr[i][t], yi[i][t]);
                                bh[i][t] = pk16(xr[i][t], xn[i][t]);
                                ch[i][t] = pk16(-xn[i][t], xr[i][t]);
                            }
                        }
#pragma unroll
                    for (int j = 0; j < 2; j++)
#pragma unroll
                        for (int i = 0; i < 2; i++) {
                            accr[i][j] = mfma<_Float16>(ex_u4(ah[i]), ex_u4(bh[j]), accr[i][j]);
                            acci[i][j] = mfma<_Float16>(ex_u4(ah[i]), ex_u4(ch[j]), acci[i][j]);
                        }
                    if (m < 2)
#pragma unroll
                        for (int j = 0; j < 2; j++)
#pragma unroll
                            for (int i = 0; i < 2; i++) {
                                accr[i][j] = mfma<_Float16>(ex_u4(al[i]), ex_u4(bh[j]), accr[i][j]);
                                acci[i][j] = mfma<_Float16>(ex_u4(al[i]), ex_u4(ch[j]), acci[i][j]);
                                accr[i][j] = mfma<_Float16>(ex_u4(ah[i]), ex_u4(bl[j]), accr[i][j]);
                                acci[i][j] = mfma<_Float16>(ex_u4(ah[i]), ex_u4(cl[j]), acci[i][j]);
                            }
                }
            }
        }
        // lane holds column l % 32 and rows 8 (v / 4) + 4 (l / 32) + v % 4 of each 32 x 32 quarter
        int hb = h0, wb = w0, ln = lane;
        const float sg = odd ? -1.f : 1.f;
        asm volatile("" : "+s"(hb), "+s"(wb), "+v"(ln));
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int h = hb + i * 32 + 8 * (v >> 2) + 4 * (ln >> 5) + (v & 3), w = wb + j * 32 + (ln & 31);
                    if (h >= ny || w >= nx) continue;
                    float2* p = &U[(size_t)h * nx + w];
                    float2 o = make_float2(sg * accr[i][j][v], sg * acci[i][j][v]);
                    if (accumulate) {
                        const float2 u = *p;
                        o.x += u.x;
                        o.y += u.y;
                    }
                    *p = o;
                }
        accumulate = true;
        odd ^= 1;
    }
    if (lane == 0) left[blockIdx.x * gridDim.y + blockIdx.y] = some ? EX_SOME : EX_NONE;
}

int cgh_exact_mfma(olx_ctx* ctx, const olx_point* d_pts, int64_t n, const CghOut& o, int64_t ny, int64_t nx,
                   double py, double px, double lambda, bool* done) {
    *done = false;
    const size_t np = (size_t)ny * (size_t)nx;
    const int64_t tx = (nx + EXT - 1) / EXT, tiles = tx * ((ny + EXT - 1) / EXT);
    if (n < 1 || n > (1 << 30) || tiles > INT32_MAX / 2 || capturing(ctx->stream)) return OLX_OK;
    // Slices of the points, with planes of at most 2 GiB.  A block of 64 points takes a wave 18.5 us at full
    // throughput, 27 alone on its SIMD; the planes, their sum and the output 9e-6 us a pixel (11e-6 past the
    // last-level cache) and 2.2e-6 for each further plane, 0.1 us a plane at least.
    const int64_t smax = std::min<int64_t>({256, (int64_t)(((size_t)2 << 30) / (sizeof(float2) * np)), (n + EXT - 1) / EXT});
    if (smax < 1) return OLX_OK;
    const double px_n = (double)np;
    int64_t S = 1;
    double best = 0.0;
    for (int64_t s = 1; s <= smax; s++) {
        const int64_t r = (tiles * s + 1023) / 1024, blocks = ((n + s - 1) / s + EXT - 1) / EXT;
        const double t = (r > 1 ? 18.5 * r : 27.0) * blocks + px_n * ((px_n < 3.4e7 ? 9e-6 : 11e-6) + 2.2e-6 * (s - 1)) + 0.1 * s;
        if (s == 1 || t < best) {
            best = t;
            S = s;
        }
    }
    // The vector kernel takes 0.12 us a point where its tiles do not fill the GPU and 3.1 point-pixel pairs a
    // ps where they do; this form's four launches 26 us at least.  Vector / this form, us: 250 points, 256 x 256
    // 32 / 26; 400, 700 x 700 75 / 49; 1000 x 1000 100 points 37 / 36, 250 86 / 52; 32 points, 2048^2 47 / 74, 64
    // 85 / 74; 8192^2 32 670 / 965, 64 1283 / 1077.
    const double t_vec = std::max(0.12 * (double)n, (double)n * px_n / 3.1e6);
    // Points too near for this form go to the vector kernel after all, which takes 0.33 us and 0.95 pairs for them:
    // a cloud of them only is slowed by the other launches and planes.  Where that is more than about a tenth the
    // vector kernel keeps the call.  100 points at z = 4 to 8 mm into
    // 2048^2: 365 us there, 418 with this form's launches; at 30 to 60 mm, where about half are too near, 204 and 254.
    const double t_near = std::max(0.33 * (double)n, (double)n * px_n / 0.95e6);
    if (t_vec <= std::max(30.0, best) || t_near <= 75.0 + std::min(px_n, 5e5) * 250e-6 + px_n * 100e-6) return OLX_OK;
    const int slice = (int)(((n + S - 1) / S + EXT - 1) / EXT * EXT);
    S = (n + slice - 1) / slice;
    if (spare(ctx, ctx->lay_counts, sizeof(uint32_t) * (size_t)(AMP_PARTS + tiles * S)) != OLX_OK ||
        spare(ctx, ctx->cgh_part, sizeof(float2) * np * (size_t)S) != OLX_OK)
        return OLX_OK;  // no room for the planes
    uint32_t* parts = (uint32_t*)ctx->lay_counts.p;
    float2* part = (float2*)ctx->cgh_part.p;
    hipStream_t s = ctx->stream;
    TimedLaunch tl(ctx, "cgh_f32_exact");
    k_amp_parts<<<AMP_PARTS, 1024, 0, s>>>(d_pts, (int)n, parts);
    k_cgh_exact_mfma<<<dim3((unsigned)tiles, (unsigned)S), 64, 0, s>>>(
        d_pts, (int)n, slice, (int)tx, (int)ny, (int)nx, py, px, lambda, part, parts, parts + AMP_PARTS);
    cgh_exact_rest(s, d_pts, n, o, ny, nx, py, px, lambda, part, (int)S, slice, parts);
    const int64_t blocks = std::min<int64_t>(((int64_t)np + 255) / 256, 65536);
    k_cgh_sum_scaled<<<(unsigned)blocks, 256, 0, s>>>(part, (int)S, (int64_t)np, o, parts);
    *done = true;
    return check_launch("cgh exact (matrix cores)");
}

}  // namespace olx

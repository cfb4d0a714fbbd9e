// olx_layered.hip -- layered Fresnel CGH as complex GEMMs on MFMA (gfx950).
//
// Points are snapped to the centres z_l of nlayers uniform layers.  For a point
// j in layer l (c_l = 1 / (lambda z_l)) the Fresnel term factorises:
//   exp(i pi ((x_w - x_j)^2 + (y_h - y_j)^2) c_l + i phi_j) A_j
//     = [cy_l(h) e^{-2 pi i h beta_j} a_j] [cx_l(w) e^{-2 pi i w alpha_j}]
// with the layer chirps cx_l(w) = e^{i pi (px w)^2 c_l}, cy_l(h) likewise, the
// cycles per pixel alpha_j = px x_j c_l, beta_j = py y_j c_l, and the point
// factor a_j = A_j e^{i (phi_j + pi (x_j^2 + y_j^2) c_l)}.  Hence
//   U = Y X^T,  Y[h, j] = cy_l(h) e^{-2 pi i h beta_j} a_j,  X[w, j] = cx_l(w) e^{-2 pi i w alpha_j},
// one complex GEMM with K = number of points, each layer's chirp folded into its
// points' factors (so no per-layer epilogue).  The complex product is two real
// MFMA GEMMs over K' = 2K interleaved (re, im) columns:
//   Re U = A Br^T,  Im U = A Bi^T,  A = [Re Y, Im Y],  Br = [Re X, -Im X],  Bi = [Im X, Re X].
// Phases are reduced exactly before quantisation: chirps in FP64 tables, and
// w alpha_j mod 1 as w alpha_hi (exact in FP32, alpha_hi has few fraction bits)
// plus w alpha_lo.  Factors are stored FP16, BF16, or split BF16 (hi + lo, three
// products Yh Xh + Yh Xl + Yl Xh); accumulation is FP32 throughout.
#include <climits>

#include "mfma_gemm.hpp"

namespace olx {

struct LayPt {       // 32 bytes
    int layer;
    float ahi, alo;  // alpha_j = ahi + alo (cycles per pixel along w), mod 1
    float bhi, blo;  // beta_j along h
    float2 a;        // point factor a_j
    float pad;
};

constexpr int KC_PTS = 32768;  // points per factor chunk
// Longest FP32 accumulation of a split product, in points: it adds three times per point, and
// the small terms lose bits beside a large running sum.  Relative error against FP64 at 200,000
// points, 2160 x 3840: 7.05e-6 with 8192, 6.88e-6 with 4096, and 6.93e-6 for the three products
// one after the other over 32768 points (factor rounding alone: 6.76e-6).
constexpr int CHAIN_SPLIT = 4096;

__host__ __device__ inline int layer_of(double z, double zmin, double zmax, int nl) {
    double f = floor((z - zmin) / (zmax - zmin) * nl);
    if (!(f >= 0.0)) f = 0.0;
    if (f > nl - 1) f = nl - 1;
    return (int)f;
}

// split v mod 1 into hi (nb fraction bits) + lo
__device__ inline void split_cycles(double v, int nb, float* hi, float* lo) {
    v -= floor(v);
    const double s = ldexp(1.0, nb);
    const double h = floor(v * s) / s;
    *hi = (float)h;
    *lo = (float)(v - h);
}

__global__ void k_lay_prep(const olx_point* __restrict__ pts, int n, LayPt* __restrict__ out,
                           double px, double py, double lambda, double zmin, double zmax, int nl,
                           int nb) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const olx_point p = pts[j];
    const int l = layer_of(p.z, zmin, zmax, nl);
    const double zl = zmin + ((double)l + 0.5) * (zmax - zmin) / nl;
    const double c = 1.0 / (lambda * zl);
    LayPt q;
    q.layer = l;
    split_cycles(px * p.x * c, nb, &q.ahi, &q.alo);
    split_cycles(py * p.y * c, nb, &q.bhi, &q.blo);
    double cyc = 0.5 * (p.x * p.x + p.y * p.y) * c + (double)p.phase * (0.5 / M_PI);
    cyc -= rint(cyc);
    double s, co;
    sincospi(2.0 * cyc, &s, &co);
    q.a = make_float2((float)(p.amp * co), (float)(p.amp * s));
    q.pad = 0.f;
    out[j] = q;
}

// per-layer chirp tables: ch[l * n + i] = exp(i pi (d i)^2 c_l), and the chirp's
// half-step in cycles per pixel^2, cd2[l] = d^2 c_l / 2
__global__ void k_lay_chirp(float2* __restrict__ ch, float* __restrict__ cd2, int n, int nl,
                            double d, double lambda, double zmin, double zmax) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, l = blockIdx.y;
    if (i >= n) return;
    const double zl = zmin + ((double)l + 0.5) * (zmax - zmin) / nl;
    if (i == 0) cd2[l] = (float)(0.5 * d * d / (lambda * zl));
    const double x = d * i;
    double cyc = 0.5 * x * x / (lambda * zl);
    cyc -= rint(cyc);
    double s, c;
    sincospi(2.0 * cyc, &s, &c);
    ch[(size_t)l * n + i] = make_float2((float)c, (float)s);
}

constexpr int GEN_RB = 16;  // rows per thread (one exact anchor, then a recurrence)

// factor rows: for rows r (h for Y, w for X) and chunk points j in [0, kc):
//   Y: A[r][2j] = Re, A[r][2j+1] = Im of cy_l(r) e^{-2 pi i r beta} a
//   X: B[r][2j] = Re, B[r][2j+1] = -Im of cx_l(r) e^{-2 pi i r alpha}
// A thread owns one point and GEN_RB consecutive rows: the phase e^{-2 pi i r alpha}
// is evaluated exactly (reduced) at the first row and advanced by the exact step
// e^{-2 pi i alpha} (rounding drift ~1e-6 over the run, far below FP16/BF16 ulps).
// SPLIT: hi = the rounded value and lo = value - hi, in the split row layout; a row is ldw
// 32-bit words.
template <typename T, bool ISY, bool SPLIT>
__global__ void k_lay_gen(const LayPt* __restrict__ pts, int j0, int n, int kc,
                          const float2* __restrict__ chirp, const float* __restrict__ chd2,
                          int rows, uint32_t* __restrict__ out, int ldw) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;  // chunk-local point
    const int rb = blockIdx.y * GEN_RB;
    if (j >= kc) return;
    const bool live = j0 + j < n;
    LayPt p;
    if (live) p = pts[j0 + j];
    else { p.layer = 0; p.ahi = p.alo = p.bhi = p.blo = 0.f; p.a = make_float2(0.f, 0.f); }
    const float hi = ISY ? p.bhi : p.ahi, lo = ISY ? p.blo : p.alo;
    // anchor e^{-2 pi i rb alpha} and step e^{-2 pi i alpha}
    const float fr = (float)rb;
    float t = fr * hi;  // exact: hi has few fraction bits
    t = (t - floorf(t)) + fr * lo;
    t = -(t - rintf(t));
    float2 e = make_float2(__builtin_amdgcn_cosf(t), __builtin_amdgcn_sinf(t));
    float ts = hi + lo;
    ts = -(ts - rintf(ts));
    const float2 stp = make_float2(__builtin_amdgcn_cosf(ts), __builtin_amdgcn_sinf(ts));
    // layer chirp e^{i pi c (d r)^2}: the FP64-built table gives the anchor at rb;
    // the next rows follow from ch(r+1) = ch(r) g(r), g(r) = e^{i pi c d^2 (2r+1)},
    // g(r+1) = g(r) e^{2 pi i c d^2}; their phases are at most a few cycles, exact
    // enough in FP32 (c d^2 = cd2 cycles per pixel^2 over 2)
    float2 ch = chirp[(size_t)p.layer * rows + rb];
    const float cd2 = chd2[p.layer];
    float tg = cd2 * (2.0f * fr + 1.0f);
    tg -= rintf(tg);
    float2 gr = make_float2(__builtin_amdgcn_cosf(tg), __builtin_amdgcn_sinf(tg));
    float tgg = 2.0f * cd2;
    tgg -= rintf(tgg);
    const float2 gg = make_float2(__builtin_amdgcn_cosf(tgg), __builtin_amdgcn_sinf(tgg));
    for (int q = 0; q < GEN_RB; q++) {
        const int r = rb + q;
        if (r >= rows) break;
        float2 v = make_float2(ch.x * e.x - ch.y * e.y, ch.x * e.y + ch.y * e.x);
        if (ISY) v = make_float2(v.x * p.a.x - v.y * p.a.y, v.x * p.a.y + v.y * p.a.x);
        else v.y = -v.y;
        if (!live) v = make_float2(0.f, 0.f);
        uint32_t* o = out + (size_t)r * ldw + fac_word<SPLIT>(j);  // 2 halves a word
        float hx, hy;
        o[0] = pack2<T>(v.x, v.y, &hx, &hy);
        if (SPLIT) {
            float dx_, dy_;
            o[16] = pack2<T>(v.x - hx, v.y - hy, &dx_, &dy_);
        }
        e = make_float2(e.x * stp.x - e.y * stp.y, e.x * stp.y + e.y * stp.x);
        ch = make_float2(ch.x * gr.x - ch.y * gr.y, ch.x * gr.y + ch.y * gr.x);
        gr = make_float2(gr.x * gg.x - gr.y * gg.y, gr.x * gg.y + gr.y * gg.x);
    }
}

// the K slices' planes added in slice order, to what U holds with accumulate
__global__ void k_lay_sum(const float2* __restrict__ part, int S, int64_t np, float2* __restrict__ U,
                          int accumulate) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < np;
         i += (int64_t)gridDim.x * blockDim.x) {
        float2 v = part[i];
        for (int z = 1; z < S; z++) {
            const float2 w = part[(size_t)z * np + i];
            v = make_float2(v.x + w.x, v.y + w.y);
        }
        if (accumulate) v = make_float2(v.x + U[i].x, v.y + U[i].y);
        U[i] = v;
    }
}

static int nbits_for(int64_t P) {
    int lg = 0;
    while ((1ll << lg) < P) lg++;
    return 24 - lg;
}

}  // namespace olx

using namespace olx;

extern "C" double olx_layer_depth(double z, double zmin, double zmax, int nlayers) {
    const int l = layer_of(z, zmin, zmax, nlayers);
    return zmin + ((double)l + 0.5) * (zmax - zmin) / nlayers;
}

extern "C" int olx_cgh_layered_c64(olx_ctx* ctx, const olx_point* d_pts, int64_t n, void* d_U,
                                   int64_t ny, int64_t nx, double py, double px, double lambda,
                                   int nlayers, double zmin, double zmax, int precision,
                                   uint32_t flags) {
    if (!ctx || !d_U) OLX_FAIL(OLX_EINVAL, "layered: null argument");
    if (n < 0 || (n > 0 && !d_pts)) OLX_FAIL(OLX_EINVAL, "layered: bad point array");
    if (n > INT32_MAX / 2) OLX_FAIL(OLX_EUNSUPPORTED, "layered: too many points");
    if (ny <= 0 || nx <= 0 || ny > 8192 || nx > 8192)
        OLX_FAIL(OLX_EUNSUPPORTED, "layered: hologram sides must be in [1, 8192]");
    if (!(py > 0) || !(px > 0) || !(lambda > 0) || nlayers < 1 || !(zmax > zmin) || !(zmin > 0))
        OLX_FAIL(OLX_EINVAL, "layered: need pitch, lambda > 0, nlayers >= 1, 0 < zmin < zmax");
    if (precision < OLX_LAYERED_F16 || precision > OLX_LAYERED_BF16X3)
        OLX_FAIL(OLX_EINVAL, "layered: unknown precision %d", precision);
    hipStream_t s = ctx->stream;
    const bool acc0 = (flags & OLX_CGH_ACCUMULATE) != 0;
    if (n == 0) {
        if (!acc0) OLX_HIP(hipMemsetAsync(d_U, 0, sizeof(float2) * ny * nx, s));
        return OLX_OK;
    }
    // point records and chirp tables
    const size_t pts_bytes = sizeof(LayPt) * (size_t)n;
    const size_t cx_off = (pts_bytes + 255) & ~(size_t)255;
    const size_t cy_off = cx_off + sizeof(float2) * (size_t)nlayers * nx;
    const size_t dx_off = cy_off + sizeof(float2) * (size_t)nlayers * ny;
    const size_t dy_off = dx_off + sizeof(float) * (size_t)nlayers;
    const size_t meta_bytes = dy_off + sizeof(float) * (size_t)nlayers;
    OLX_TRY(ctx->lay_pts.reserve(meta_bytes, ctx));
    char* meta = (char*)ctx->lay_pts.p;
    LayPt* lp = (LayPt*)meta;
    float2* cx = (float2*)(meta + cx_off);
    float2* cy = (float2*)(meta + cy_off);
    float* cdx = (float*)(meta + dx_off);
    float* cdy = (float*)(meta + dy_off);
    const int nb = nbits_for(std::max(nx, ny));
    {
        TimedLaunch tl(ctx, "layered_prep");
        k_lay_prep<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(d_pts, (int)n, lp, px, py, lambda,
                                                               zmin, zmax, nlayers, nb);
        k_lay_chirp<<<dim3((unsigned)((nx + 255) / 256), nlayers), 256, 0, s>>>(
            cx, cdx, (int)nx, nlayers, px, lambda, zmin, zmax);
        k_lay_chirp<<<dim3((unsigned)((ny + 255) / 256), nlayers), 256, 0, s>>>(
            cy, cdy, (int)ny, nlayers, py, lambda, zmin, zmax);
    }
    OLX_TRY(check_launch("layered prep"));
    // Points go in equal chunks of at most KC_PTS, padded with zero factors to a whole stage.
    const bool split = precision == OLX_LAYERED_BF16X3;
    const int sp = split ? stage_pts<true>() : stage_pts<false>();
    const int64_t nchunk = (n + KC_PTS - 1) / KC_PTS;
    const int kc = (int)(((n + nchunk - 1) / nchunk + sp - 1) / sp * sp);
    const int ldk = (split ? 4 : 2) * kc, stages = kc / sp;
    const int chain = split ? CHAIN_SPLIT / sp : stages;
    // Partial planes for K slices take at most 2 GiB; without them (or if they do not
    // fit) the products accumulate in the hologram itself.
    const size_t np = (size_t)ny * (size_t)nx;
    const int smax = (int)std::max<size_t>(1, std::min<size_t>(64, ((size_t)2 << 30) / (sizeof(float2) * np)));
    // (4 us of another launch: 100 points into 64 x 64 24.6 us, 27.3 with it)
    const double merge = 4e-6 * 2.2e9;
    GemmPlan g = gemm_plan(ny, nx, stages, split, smax, merge);
    if (g.slices > 1 && spare(ctx, ctx->cgh_part, sizeof(float2) * np * (size_t)g.slices) != OLX_OK)
        g = gemm_plan(ny, nx, stages, split, 1, merge);
    // the asked-for 128-row tile keeps the plan's K slices, so its sums run in the same order
    if (flags & OLX_LAYERED_TILE128) g.wr = 2;
    float2* out = g.slices > 1 ? (float2*)ctx->cgh_part.p : (float2*)d_U;
    auto up = [](int64_t v, int64_t m) { return (v + m - 1) / m * m; };
    const size_t ybytes = sizeof(uint16_t) * (size_t)up(ny, 64 * g.wr) * ldk;
    const size_t xbytes = sizeof(uint16_t) * (size_t)up(nx, GTN) * ldk;
    OLX_TRY(ctx->lay_counts.reserve(ybytes + xbytes, ctx));
    uint32_t* Y = (uint32_t*)ctx->lay_counts.p;
    uint32_t* X = (uint32_t*)((char*)ctx->lay_counts.p + ybytes);

    // XCD tile swizzle: each XCD takes a contiguous run of
    // tiles, 4 tile rows at a time (OLX_LAYSWZ overrides; 0 = launch order).  At 4096^2 (1 M points,
    // 64 layers, f16): 109.3-109.6 ms against 111.1-111.2 ms in launch order (2, 8 rows:
    // 110.5-111.4 ms); the outputs are bitwise the same.
    static const char* swz_env = getenv("OLX_LAYSWZ");
    const int swz = swz_env ? atoi(swz_env) : 4;
    for (int64_t c = 0; c < nchunk; c++) {
        const int64_t j0 = c * kc;
        if (j0 >= n) break;
        const int kn = (int)std::min<int64_t>(kc, up(n - j0, sp)), st = kn / sp;
        const dim3 gy((unsigned)((kn + 255) / 256), (unsigned)((ny + GEN_RB - 1) / GEN_RB)),
            gx((unsigned)((kn + 255) / 256), (unsigned)((nx + GEN_RB - 1) / GEN_RB));
        {
            TimedLaunch tl(ctx, "layered_factors");
            auto gen = [&](auto t, auto SP) {
                using T = decltype(t);
                k_lay_gen<T, true, SP.value><<<gy, 256, 0, s>>>(lp, (int)j0, (int)n, kn, cy, cdy, (int)ny, Y, ldk / 2);
                k_lay_gen<T, false, SP.value><<<gx, 256, 0, s>>>(lp, (int)j0, (int)n, kn, cx, cdx, (int)nx, X, ldk / 2);
            };
            if (precision == OLX_LAYERED_F16) gen(_Float16(), std::false_type());
            else if (precision == OLX_LAYERED_BF16) gen(__bf16(), std::false_type());
            else gen(__bf16(), std::true_type());
        }
        OLX_TRY(check_launch("layered factors"));
        {
            TimedLaunch tl(ctx, "layered_gemm");
            const int acc = c > 0 || (acc0 && g.slices == 1);
            const int S = (st + g.kslice - 1) / g.kslice;
            if (precision == OLX_LAYERED_F16)
                cgemm<_Float16, false>(s, g.wr, S, Y, X, ldk, st, g.kslice, chain, out, np, ny, nx, acc, swz);
            else if (precision == OLX_LAYERED_BF16)
                cgemm<__bf16, false>(s, g.wr, S, Y, X, ldk, st, g.kslice, chain, out, np, ny, nx, acc, swz);
            else
                cgemm<__bf16, true>(s, g.wr, S, Y, X, ldk, st, g.kslice, chain, out, np, ny, nx, acc, swz);
        }
        OLX_TRY(check_launch("layered gemm"));
    }
    if (g.slices > 1) {
        const int64_t blocks = std::min<int64_t>(((int64_t)np + 255) / 256, 65536);
        k_lay_sum<<<(unsigned)blocks, 256, 0, s>>>(out, g.slices, (int64_t)np, (float2*)d_U, acc0 ? 1 : 0);
    }
    return check_launch("layered sum");
}

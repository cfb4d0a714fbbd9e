// olx_wrp.hip -- wavefront-recording-plane accumulation and the WRP method.
//
// WRPStep1 (include/golcgh.h:303-367 circle, :403-468 square) loops every point
// for every pixel.  Here points are binned instead:
//   1. per point: window radius W_j = |z_j - z_wrp| / sqrt(4 (p_lim/lambda)^2 - 1)
//      (square: D_j = sqrt(2) W_j) and the 16 x 16 pixel tiles its window touches;
//   2. lists of (cell, point) pairs, a cell being 8 x 8 tiles or more (at most 1024
//      cells), in ascending point index: each block of 512 points sets one bit a
//      pair in LDS masks, so that counts and ranks are popcounts and no global atomic
//      is needed; then a scan over the blocks and cells, and the fill;
//   3. one work-group per tile: walk its cell's list, keep the points whose window
//      touches the tile (order kept), stage their constants (position, window limit,
//      1/(2 dz lambda), 1/|dz|) in LDS, and accumulate exp(i pi rho^2/(lambda dz))/|dz|
//      for the pixels inside each window (one to four pixels of a column per thread).  Every tile sums its points in ascending
//      index order, sparse or dense, so the result does not depend on the launch.
// Lists per tile, counted and filled with one global atomic a (tile, point) pair and
// sorted again tile by tile, took 63 + 85 us beside the sum's 184 at 200,000 points into
// 4096^2 (1.8 million pairs): device-scope atomics run at about 28 a nanosecond.  Now 7 us
// of counting, 12 of scans and 10 of filling; the whole call 388 -> 188 us, and 200,000
// points into 256^2, whose tiles scanned the whole cloud, 3736 -> 705 us.
// This file is built without FMA contraction: dx*dx + dy*dy rounds each product,
// as the reference's host arithmetic does, so window membership is decided alike.
// Window tests and rho^2 use FP64 in the reference's expression order, so pixel
// membership is decided exactly as the reference does with PREC_T = double.
#include <climits>

#include "olx_common.hpp"

namespace olx {

constexpr int WT = 16;  // tile side (pixels)

__device__ __forceinline__ double wrp_radius(double z, double plane_z, double plim,
                                             double lambda, int square) {
    // WRPStep1Pre(_D), include/golcgh.h:298, :399-400
    const double W = 1.0 / sqrt(4.0 * (plim / lambda) * (plim / lambda) - 1.0) * fabs(z - plane_z);
    return square ? W * (double)1.41421353816986083984375 /* sqrtf(2.0f) */ : W;
}

// tile range [t0, t1] touched by a point's window along one axis
__device__ __forceinline__ void tile_span(double c, double R, double p, int n, int* t0, int* t1) {
    double lo = floor((c - R) / p) - 1.0, hi = ceil((c + R) / p) + 1.0;
    lo = fmax(lo, 0.0);
    hi = fmin(hi, (double)(n - 1));
    if (hi < lo) {
        *t0 = 1;
        *t1 = 0;
        return;
    }
    *t0 = (int)lo / WT;
    *t1 = (int)hi / WT;
}

__device__ __forceinline__ double window_extent(double Wd, int square) {
    return square ? 0.5 * Wd : Wd;
}

// ---------------------------------------------------------------- binning
constexpr int BIN_T = 512, BIN_W = BIN_T / 32;  // points a block, mask words a cell
constexpr int MAX_CELLS = 1024;                  // 64 KB of masks

struct WrpGrid {
    int ny, nx, tiles_x, tiles_y;
    int cl;                       // log2 of a cell's side in tiles
    int cells_x, ncell;
};

// cells of 8 x 8 tiles: a tile then tests about 8 candidates for a point it keeps, each a
// fraction of a per cent of the 256 pixels' sums; larger where there would be too many
static WrpGrid wrp_grid(int64_t ny, int64_t nx) {
    WrpGrid g;
    g.ny = (int)ny;
    g.nx = (int)nx;
    g.tiles_x = (int)((nx + WT - 1) / WT);
    g.tiles_y = (int)((ny + WT - 1) / WT);
    for (g.cl = 3;; g.cl++) {
        const int c = 1 << g.cl, cy = (g.tiles_y + c - 1) / c;
        g.cells_x = (g.tiles_x + c - 1) / c;
        g.ncell = g.cells_x * cy;
        if (g.ncell <= MAX_CELLS) return g;
    }
}

// the block's pairs as bits: mask[w ncell + cell] bit b is point 32 w + b of the block
__device__ __forceinline__ void wrp_masks(uint32_t* mask, ushort4 t, const WrpGrid& g) {
    for (int i = threadIdx.x; i < BIN_W * g.ncell; i += BIN_T) mask[i] = 0;
    __syncthreads();
    const int w = threadIdx.x >> 5;
    if (t.x <= t.y)
        for (int cy = t.z >> g.cl; cy <= t.w >> g.cl; cy++)
            for (int cx = t.x >> g.cl; cx <= t.y >> g.cl; cx++)
                atomicOr(&mask[w * g.ncell + cy * g.cells_x + cx], 1u << (threadIdx.x & 31));
    __syncthreads();
}

// tile spans of every point (x0, x1, y0, y1; x0 > x1: none), the pairs of each (block, cell)
// in cnt[block ncell + cell], and each block's (tile, point) pairs
__global__ void __launch_bounds__(BIN_T)
k_wrp_count(const olx_point* __restrict__ pts, int n, ushort4* __restrict__ spans, int* __restrict__ cnt,
            long long* __restrict__ pairs, WrpGrid g, double p, double lambda, double plane_z,
            double plim, int square) {
    __shared__ uint32_t mask[BIN_W * MAX_CELLS];
    __shared__ long long wsum[BIN_T / 64];
    const int j = blockIdx.x * BIN_T + threadIdx.x;
    ushort4 t = {1, 0, 1, 0};
    long long np = 0;
    if (j < n) {
        const olx_point q = pts[j];
        const double R = window_extent(wrp_radius(q.z, plane_z, plim, lambda, square), square);
        int x0, x1, y0, y1;
        tile_span(q.x, R, p, g.nx, &x0, &x1);
        tile_span(q.y, R, p, g.ny, &y0, &y1);
        if (x0 <= x1 && y0 <= y1) {
            t = {(unsigned short)x0, (unsigned short)x1, (unsigned short)y0, (unsigned short)y1};
            np = (long long)(x1 - x0 + 1) * (y1 - y0 + 1);
        }
        spans[j] = t;
    }
    wrp_masks(mask, t, g);
    for (int c = threadIdx.x; c < g.ncell; c += BIN_T) {
        int k = 0;
#pragma unroll
        for (int w = 0; w < BIN_W; w++) k += __popc(mask[w * g.ncell + c]);
        cnt[(size_t)blockIdx.x * g.ncell + c] = k;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) np += __shfl_down(np, off, 64);
    if (threadIdx.x % 64 == 0) wsum[threadIdx.x / 64] = np;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < BIN_T / 64; w++) np += wsum[w];
        pairs[blockIdx.x] = np;
    }
}

// exclusive scan of each cell's counts over the blocks, in place, and the cell's total: 64
// cells a work-group, the blocks in 16 runs
constexpr int CS_C = 64, CS_S = 16;
__global__ void __launch_bounds__(CS_C * CS_S)
k_wrp_cells(int* __restrict__ cnt, int nblk, int ncell, int* __restrict__ tot) {
    __shared__ int part[CS_S][CS_C];
    const int ci = threadIdx.x % CS_C, sg = threadIdx.x / CS_C, c = blockIdx.x * CS_C + ci;
    const int len = (nblk + CS_S - 1) / CS_S, b0 = min(sg * len, nblk), b1 = min(b0 + len, nblk);
    int v = 0;
    if (c < ncell)
#pragma unroll 8
        for (int b = b0; b < b1; b++) v += cnt[(size_t)b * ncell + c];
    part[sg][ci] = v;
    __syncthreads();
    if (c >= ncell) return;
    int run = 0;
    for (int k = 0; k < sg; k++) run += part[k][ci];
    if (sg == CS_S - 1) tot[c] = run + v;
#pragma unroll 8
    for (int b = b0; b < b1; b++) {
        const int x = cnt[(size_t)b * ncell + c];
        cnt[(size_t)b * ncell + c] = run;
        run += x;
    }
}

// the cells' list bases; base[ncell]: all entries, or -1 with more than 2^31 - 1 (tile, point) pairs, then those
// pairs and the entries of the fullest cell
__global__ void __launch_bounds__(MAX_CELLS)
k_wrp_bases(const int* __restrict__ tot, int ncell, const long long* __restrict__ pairs, int nblk,
            int* __restrict__ base) {
    __shared__ long long part[3][MAX_CELLS / 64];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int v = tid < ncell ? tot[tid] : 0;
    long long x = v, np = 0;
    int most = v;
    for (int b = tid; b < nblk; b += MAX_CELLS) np += pairs[b];
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const long long y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
        np += __shfl_xor(np, off, 64);
        most = max(most, __shfl_xor(most, off, 64));
    }
    if (lane == 63) part[0][wv] = x;
    if (lane == 0) {
        part[1][wv] = np;
        part[2][wv] = most;
    }
    __syncthreads();
    for (int k = 0; k < wv; k++) x += part[0][k];
    if (tid < ncell) base[tid] = (int)(x - v);
    if (tid == ncell - 1) {
        np = 0;
        for (int k = 0; k < MAX_CELLS / 64; k++) {
            np += part[1][k];
            most = max(most, (int)part[2][k]);
        }
        base[ncell] = np > INT_MAX ? -1 : (int)x;  // a cell's entries never outnumber its tiles'
        base[ncell + 1] = (int)min(np, (long long)INT_MAX);
        base[ncell + 2] = most;
    }
}

// list entries: the point, and its tile span within the cell in four bytes (x0, x1, y0, y1)
__global__ void __launch_bounds__(BIN_T)
k_wrp_fill(const ushort4* __restrict__ spans, int n, const int* __restrict__ cnt,
           const int* __restrict__ base, int2* __restrict__ list, WrpGrid g) {
    __shared__ uint32_t mask[BIN_W * MAX_CELLS];
    const int j = blockIdx.x * BIN_T + threadIdx.x;
    ushort4 t = {1, 0, 1, 0};
    if (j < n) t = spans[j];
    wrp_masks(mask, t, g);
    if (t.x > t.y) return;
    const int w = threadIdx.x >> 5, side = (1 << g.cl) - 1;
    const uint32_t below = (1u << (threadIdx.x & 31)) - 1u;
    for (int cy = t.z >> g.cl; cy <= t.w >> g.cl; cy++)
        for (int cx = t.x >> g.cl; cx <= t.y >> g.cl; cx++) {
            const int c = cy * g.cells_x + cx, ox = cx << g.cl, oy = cy << g.cl;
            int r = __popc(mask[w * g.ncell + c] & below);
            for (int k = 0; k < w; k++) r += __popc(mask[k * g.ncell + c]);
            const int x0 = max((int)t.x - ox, 0), x1 = min((int)t.y - ox, side);
            const int y0 = max((int)t.z - oy, 0), y1 = min((int)t.w - oy, side);
            list[base[c] + cnt[(size_t)blockIdx.x * g.ncell + c] + r] =
                make_int2(j, x0 | x1 << 8 | y0 << 16 | y1 << 24);
        }
}

struct WrpPt {     // per-point constants of one tile's list, staged in LDS
    double x, y;
    double lim;    // circle: W^2 (tmp < W^2); square: W (2 |dx| <= W)
    double rc;     // 1 / (2 dz lambda): phase in cycles = tmp * rc
    float inv;     // 1 / |dz|
    float pad;
};

__device__ __forceinline__ WrpPt wrp_stage(const olx_point& q, double lambda, double plane_z,
                                           double plim, int square) {
    WrpPt s;
    const double Wd = wrp_radius(q.z, plane_z, plim, lambda, square);
    const double dz = q.z - plane_z;
    s.x = q.x;
    s.y = q.y;
    s.lim = square ? Wd : Wd * Wd;
    s.rc = 1.0 / (2.0 * dz * lambda);
    s.inv = (float)(1.0 / fabs(dz));
    s.pad = 0.f;
    return s;
}

template <bool SQUARE>
__device__ __forceinline__ void wrp_pixel(const WrpPt& P, double dx, double dy, float& re,
                                          float& im) {
    const double tmp = dx * dx + dy * dy;
    const bool inside = SQUARE ? (fabs(dx) * 2 <= P.lim && fabs(dy) * 2 <= P.lim) : (tmp < P.lim);
    if (inside) {
        double cyc = tmp * P.rc;
        cyc -= rint(cyc);
        const float t = (float)cyc;
        re += __builtin_amdgcn_cosf(t) * P.inv;
        im += __builtin_amdgcn_sinf(t) * P.inv;
    }
}

// With XCD_CELLS cells or more, work-groups of one cell's tiles run on one XCD (dispatch is
// round-robin over 8), so its L2 holds the cell's list and points; fewer cells would load the
// XCDs unevenly, and there the tiles go in row order.  The list is walked NT entries a step, points
// that touch the tile collected by index, and summed once NT are there or the list ends.  A thread
// owns one column's rows t / 16 + RS r, which share dx and each staged point read from LDS.  Bound by
// FP64 and sine / cosine issue: 200,000 points into 4096 x 4096 take 450 million pixel sums.
constexpr int XCD_CELLS = 64;
template <bool SQUARE, int NT>
__global__ void __launch_bounds__(NT)
k_wrp_accum(const olx_point* __restrict__ pts, const int* __restrict__ base, const int2* __restrict__ list,
            float2* __restrict__ U, WrpGrid g, double p, double lambda, double plane_z, double plim) {
    __shared__ int ids[2 * NT];
    __shared__ WrpPt sp[NT];
    __shared__ int wcnt[NT / 64];
    int tx = blockIdx.x % g.tiles_x, ty = blockIdx.x / g.tiles_x;
    if (g.ncell >= XCD_CELLS) {
        const int b = blockIdx.x / 8, tin = b & ((1 << 2 * g.cl) - 1);
        const int c = (b >> 2 * g.cl) * 8 + blockIdx.x % 8;
        tx = (c % g.cells_x << g.cl) + (tin & ((1 << g.cl) - 1));
        ty = (c / g.cells_x << g.cl) + (tin >> g.cl);
        if (c >= g.ncell || tx >= g.tiles_x || ty >= g.tiles_y) return;
    }
    const int cell = (ty >> g.cl) * g.cells_x + (tx >> g.cl);
    const int lx = tx & ((1 << g.cl) - 1), ly = ty & ((1 << g.cl) - 1);
    constexpr int RT = WT * WT / NT, RS = WT / RT;  // rows a thread, and their distance
    const int w = tx * WT + threadIdx.x % WT, h0 = ty * WT + threadIdx.x / WT;
    const double xw = p * w;
    double yh[RT];
    float re[RT], im[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        yh[r] = p * (h0 + RS * r);
        re[r] = im[r] = 0.f;
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t end = (uint32_t)base[cell + 1];  // at most 2^31 - 1: unsigned, NT past it does not wrap
    int f = 0;  // points collected
    for (uint32_t i0 = (uint32_t)base[cell]; i0 < end; i0 += NT) {
        const uint32_t i = i0 + threadIdx.x;
        int2 e = make_int2(0, 0);
        bool take = false;
        if (i < end) {
            e = list[i];
            const uint32_t t = (uint32_t)e.y;
            take = lx >= (int)(t & 255) && lx <= (int)(t >> 8 & 255) && ly >= (int)(t >> 16 & 255) &&
                   ly <= (int)(t >> 24);
        }
        const unsigned long long mk = __ballot(take);
        if (lane == 0) wcnt[wv] = __popcll(mk);
        __syncthreads();
        int before = f;
#pragma unroll
        for (int k = 0; k < NT / 64; k++) {
            before += k < wv ? wcnt[k] : 0;
            f += wcnt[k];
        }
        if (take) ids[before + __popcll(mk & ((1ull << lane) - 1ull))] = e.x;
        __syncthreads();
        if (f < NT && i0 + NT < end) continue;  // f < 2 NT always
        for (int k0 = 0; k0 < f; k0 += NT) {
            const int m = min(NT, f - k0);
            if ((int)threadIdx.x < m)
                sp[threadIdx.x] = wrp_stage(pts[ids[k0 + threadIdx.x]], lambda, plane_z, plim, SQUARE);
            __syncthreads();
            for (int k = 0; k < m; k++) {
                const WrpPt P = sp[k];
                const double dx = xw - P.x;
#pragma unroll
                for (int r = 0; r < RT; r++) wrp_pixel<SQUARE>(P, dx, yh[r] - P.y, re[r], im[r]);
            }
            __syncthreads();
        }
        f = 0;
    }
#pragma unroll
    for (int r = 0; r < RT; r++)
        if (w < g.nx && h0 + RS * r < g.ny) U[(size_t)(h0 + RS * r) * g.nx + w] = make_float2(re[r], im[r]);
}

}  // namespace olx

using namespace olx;

extern "C" double olx_wrp_plane_z(int64_t ny, int64_t nx, double p, double lambda, double zmin,
                                  double p_limit, float s, int square) {
    float plane_z;
    if (s < 0) {
        if (square) {  // WRPMethod_D, include/golcgh.h:546-550
            const float D = (float)(nx * p * 0.05);
            const float d = (float)(std::sqrt(4 * std::pow((p_limit / lambda), 2) - 1) /
                                    std::sqrt(2) * D);
            plane_z = (float)(zmin - d);
        } else {  // WRPMethod, include/golcgh.h:567-571
            const float Wpow2 = (float)(nx * ny * p * p / M_PI * 1 / 1024.f);
            const float d = (float)std::sqrt((4 * std::pow((p / lambda), 2) - 1) * Wpow2);
            plane_z = (float)(zmin - d);
        }
    } else {
        plane_z = (float)(zmin * s);
    }
    return (double)plane_z;
}

extern "C" int olx_wrp_c64(olx_ctx* ctx, const olx_point* d_pts, int64_t n, void* d_U,
                           int64_t ny, int64_t nx, double p, double lambda, double plane_z,
                           double p_limit, uint32_t flags) {
    if (!ctx || !d_U) OLX_FAIL(OLX_EINVAL, "wrp: null argument");
    if (n < 0 || (n > 0 && !d_pts)) OLX_FAIL(OLX_EINVAL, "wrp: bad point array");
    if (n > INT32_MAX / 4) OLX_FAIL(OLX_EUNSUPPORTED, "wrp: too many points");
    if (ny <= 0 || nx <= 0 || ny > 65536 || nx > 65536) OLX_FAIL(OLX_EINVAL, "wrp: bad plane size");
    if (!(p > 0) || !(lambda > 0) || !(p_limit > 0.5 * lambda))
        OLX_FAIL(OLX_EINVAL, "wrp: need p > 0, lambda > 0 and p_limit > lambda/2");
    const int square = (flags & OLX_WRP_SQUARE) ? 1 : 0;
    const WrpGrid g = wrp_grid(ny, nx);
    const int nblk = (int)((n + BIN_T - 1) / BIN_T);
    // spans | pairs | counts | cell totals | bases
    const size_t ints = (size_t)nblk * g.ncell + 2 * g.ncell + 3;
    OLX_TRY(ctx->wrp_counts.reserve(sizeof(ushort4) * (size_t)n + sizeof(long long) * (size_t)nblk +
                                    sizeof(int) * ints, ctx));
    ushort4* spans = (ushort4*)ctx->wrp_counts.p;
    long long* pairs = (long long*)(spans + n);
    int* cnt = (int*)(pairs + nblk);
    int* tot = cnt + (size_t)nblk * g.ncell;
    int* base = tot + g.ncell;
    hipStream_t s = ctx->stream;
    {
        TimedLaunch tl(ctx, "wrp_bin");
        if (n > 0)
            k_wrp_count<<<nblk, BIN_T, 0, s>>>(d_pts, (int)n, spans, cnt, pairs, g, p, lambda, plane_z,
                                               p_limit, square);
        k_wrp_cells<<<(g.ncell + CS_C - 1) / CS_C, CS_C * CS_S, 0, s>>>(cnt, nblk, g.ncell, tot);
        k_wrp_bases<<<1, MAX_CELLS, 0, s>>>(tot, g.ncell, pairs, nblk, base);
    }
    OLX_TRY(check_launch("wrp count/scan"));
    int sums[3] = {0, 0, 0};  // list entries, (tile, point) pairs, entries of the fullest cell
    OLX_HIP(hipMemcpyAsync(sums, base + g.ncell, sizeof sums, hipMemcpyDeviceToHost, s));
    OLX_HIP(hipStreamSynchronize(s));
    const int total = sums[0];
    if (total < 0) OLX_FAIL(OLX_EUNSUPPORTED, "wrp: more than 2^31 (tile, point) pairs");
    OLX_TRY(ctx->wrp_lists.reserve(sizeof(int2) * (size_t)std::max(total, 1), ctx));
    int2* list = (int2*)ctx->wrp_lists.p;
    {
        TimedLaunch tl(ctx, "wrp_fill");
        if (n > 0) k_wrp_fill<<<nblk, BIN_T, 0, s>>>(spans, (int)n, cnt, base, list, g);
    }
    OLX_TRY(check_launch("wrp fill"));
    {
        TimedLaunch tl(ctx, "wrp_accum");
        const unsigned nt = g.ncell >= XCD_CELLS ? ((unsigned)(g.ncell + 7) / 8 * 8) << (2 * g.cl)
                                                 : (unsigned)(g.tiles_x * g.tiles_y);
        auto go = [&](auto SQ, auto NT) {
            k_wrp_accum<decltype(SQ)::value, decltype(NT)::value><<<nt, decltype(NT)::value, 0, s>>>(
                d_pts, base, list, (float2*)d_U, g, p, lambda, plane_z, p_limit);
        };
        const auto sq = [&](auto NT) {
            if (square) go(std::true_type(), NT);
            else go(std::false_type(), NT);
        };
        // Threads a tile: four pixels a thread (64) read each staged point least often, but
        // leave the chip's 1024 SIMDs short of waves on small planes.  64 / 128 / 256 threads, whole
        // call in us: 200,000 points into 4096 x 4096 (65536 tiles) 188 / 213, 2160 x 3840 182 / 196 / 287,
        // 2048 x 2048 (16384) 186 / 193 / 282, 1024 x 1024 (4096) 230 / 211 / 286, 20,000 into
        // 512 x 512 (1024) 93 / 74 / 72, 200,000 into 256 x 256 (256) 1722 / 1127 / 705.
        // Where a cell holds much of the cloud the fullest tiles' chains last longest, and more threads shorten
        // them: the tiles that such a load would fill count instead (in an even cloud a tile has a tenth to a
        // fortieth of its cell's entries).  200,000 points in 64 x 64 pixels of 4096^2, 64 / 256 threads: 21.1 / 9.0 ms, in
        // 100 x 100 of 8192^2 10.8 / 5.4.
        int64_t tiles = (int64_t)g.tiles_x * g.tiles_y;
        if (sums[2] > 256) tiles = std::min<int64_t>(tiles, 30 * (int64_t)sums[1] / sums[2]);
        if (tiles >= 16384) sq(std::integral_constant<int, 64>());
        else if (tiles >= 2048) sq(std::integral_constant<int, 128>());
        else sq(std::integral_constant<int, 256>());
    }
    return check_launch("wrp accumulate");
}

extern "C" int olx_wrp_method_c64(olx_ctx* ctx, const olx_point* d_pts, int64_t n, void* d_U,
                                  int64_t ny, int64_t nx, double p, double lambda, double zmin,
                                  double p_limit, float s, int mode, uint32_t flags,
                                  double* plane_z_out) {
    const int square = (flags & OLX_WRP_SQUARE) ? 1 : 0;
    const double plane_z = olx_wrp_plane_z(ny, nx, p, lambda, zmin, p_limit, s, square);
    if (plane_z_out) *plane_z_out = plane_z;
    OLX_TRY(olx_wrp_c64(ctx, d_pts, n, d_U, ny, nx, p, lambda, plane_z, p_limit, flags));
    // WRPStep2, include/golcgh.h:494-517 (AUTO falls back to ASM, not band-limited Fresnel)
    int m = mode;
    if (m == OLX_MODE_AUTO) {
        if (olx_asm_prop_check(ny, nx, p, p, lambda, plane_z) ||
            !olx_fresnel_prop_check(ny, nx, p, p, lambda, plane_z))
            m = OLX_MODE_ASM;
        else
            m = OLX_MODE_FRESNEL;
    }
    if (m == OLX_MODE_ASM) return olx_asm_c64(ctx, d_U, ny, nx, p, p, lambda, plane_z, 0);
    if (m == OLX_MODE_FRESNEL) return olx_fresnel_c64(ctx, d_U, ny, nx, p, p, lambda, plane_z, 0);
    OLX_FAIL(OLX_EINVAL, "wrp_method: unknown mode %d", mode);
}

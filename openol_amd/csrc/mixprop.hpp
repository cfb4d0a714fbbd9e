// mixprop.hpp -- the three passes of a padded complex64 propagation over n-point transforms of mixfft.hpp: A transforms the stored rows (one half of
// the bins a work-group), B transforms columns, multiplies by the transfer function and
// transforms back, C transforms rows back, scales and applies the post-chirp.
//
// What bounds them at 2160 x 3840 (Fresnel, 8.3 M pixels): A 68 us and C 80 us for 200 MB each
// (2.7 TB/s), B 185 us with 64 M vector instructions (104 us of issue), the rest waiting at the
// exchanges' barriers.  Before (2n-point transforms with their zeros, every stage and the transfer
// function an LDS round trip): 83 + 320 + 90 us, 174 M vector instructions in B.  1080 x 1920 ASM 135 -> 110 us,
// 500 x 735 93 -> 45, 300 x 400 70 -> 28, 1200 x 1600 167 -> 98, 3000 x 3000 500 -> 440, 4000 x 4000 1007 -> 855, 4320 x 7680
// 2495 -> 1663, 6000 x 6000 2907 -> 2143; of the 658 squares from 2 to 8192 three are slower (7436 by 4%).
// The first form of this file took the two halves one after the other with one work-group a CU: 773 us.
//
// The kernels of one QM (mixfft.hpp) are compiled in a file of their own: every radix is inlined
// in each of them, which takes the compiler a minute.
#pragma once
#include "mixfft.hpp"
#include "olx_common.hpp"
#include "prop_common.hpp"

namespace olx {

struct MxCols {  // column pass: the row plan's last stage (W's columns) and the LDS image
    int Rx, lrx;
    uint32_t mlrp;
    int image;
};
template <int QM>
void mx_rows_fwd(unsigned grid, const MxShape& sh, const float2* src, float2* W, const PropArgs& a,
                 const MxPlan<float2>* P, hipStream_t s);
template <int QM>
void mx_cols_conv(dim3 grid, const MxShape& sh, float2* W, const PropArgs& a, const MxPlan<float2>* P,
                  const MxCols& c, hipStream_t s);
template <int QM>
void mx_rows_inv(unsigned grid, const MxShape& sh, const float2* W, float2* dst, const PropArgs& a,
                 const MxPlan<float2>* P, hipStream_t s);

// Most threads of a work-group.  Six waves a SIMD (80 registers, a few spills on the way into the
// last stage) beat four (96): 2160 x 3840 Fresnel 338 against 394 us, since every wave waits for
// its exchanges and only other work-groups fill the gaps; at QM = 2 they would spill thousands.
constexpr int MX_NT = 1024;

#ifdef OLX_MIXPROP_QM
extern __shared__ __align__(16) char mx_lds[];

template <int QM>
__global__ void __launch_bounds__(MX_NT, (QM == 1 ? 6 : 4))
k_mx_rows_fwd(const float2* __restrict__ src, float2* __restrict__ W, PropArgs a,
              const MxPlan<float2>* __restrict__ P, int lognb) {
    const MxPos t = mx_pos<false>(lognb);
    const int par = blockIdx.y, nx = a.nx, R = P->f[P->nst - 1].R, lrp = mx_lrp(P->f[P->nst - 1].lr);
    const int row0 = xcd_remap(blockIdx.x, gridDim.x) << lognb, row = row0 + t.c;
    const float2 ay = (a.ay && row < a.rows) ? a.ay[row] : make_float2(1.f, 0.f);
    // rows past the last read zeros and store nothing
    const Rsrc sb = mx_rsrc(src + (size_t)row0 * a.ss, (int64_t)(a.rows - 1 - row0) * a.ss + nx);
    const Rsrc w2 = mx_rsrc(P->w2, nx);
    const uint32_t so = (uint32_t)(t.c * a.ss) * 8u;
    const uint32_t tile = (uint32_t)(a.rows * MX_CB) * 8u;
    const MxRowsOut<float2> st{mx_rsrc(W, 2ll * R * lrp * a.rows),
                     row < a.rows ? (uint32_t)(row * MX_CB) * 8u : 0x80000000u, tile,
                     (uint32_t)(lrp / MX_CB) * tile, par * R};
    mx_run<QM, false, false>((float2*)mx_lds, P, t,
        [&](int j, int r, int lr) {
            float2 x = bload(sb, so + j * 8u, r * lr * 8u);
            if (a.ax) x = cmul(x, cmul(a.ax[j + r * lr], ay));
            if (a.pre) x = cmul(x, a.pre[(size_t)(row % a.ny) * nx + j + r * lr]);
            if (par) x = cmul(x, bload(w2, j * 8u, r * lr * 8u));
            return x;
        }, st);
}

// the transfer function on a butterfly's bins 2 (j + r lr) + par
template <int MODE>
struct ColMul {
    const PropArgs& a;
    ColH ch;
    int par, My;
    Rsrc sy;
    template <int R>
    __device__ __forceinline__ void mul(int j, int lr, float2* v) const {
        if constexpr (MODE == K_TABLE) {
            float2 h[R];
#pragma unroll
            for (int r = 0; r < R; r++) h[r] = bload(sy, (2 * j + par) * 8u, r * lr * 16u);
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float2 x = cmul(ch.sx, h[r]);
                v[r] = cmul(v[r], a.adjoint ? cconj(x) : x);
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; r++) {
                v[r] = cmul(v[r], trans_h<MODE>(a, ch, 2 * (j + r * lr) + par, My));
                __builtin_amdgcn_sched_barrier(0);  // one value's FP64 temporaries at a time
            }
        }
    }
};
struct ColsOut : MxMeet<float2> {
    Rsrc wb;
    uint32_t wo;
    __device__ __forceinline__ void out(int j, int r, int lr, float2 v) const {
        if (!t.par) bstore(wb, wo + j * (MX_CB * 8u), r * lr * (MX_CB * 8u), sum(j, r, lr, v));
    }
};

template <int QM, int MODE>
__global__ void __launch_bounds__(MX_NT, (QM == 1 ? 6 : 4))
k_mx_cols_conv(float2* __restrict__ W, PropArgs a, const MxPlan<float2>* __restrict__ P, int lognb,
               MxCols k) {
    const MxPos t = mx_pos<true>(lognb);
    const int lrp = mx_lrp(k.lrx), Mx = 2 * a.nx, My = 2 * a.ny;
    const int col0 = xcd_remap(blockIdx.x, gridDim.x) << lognb, col = col0 + t.c;
    const int seg = mx_div(col, lrp, k.mlrp), jx = col - seg * lrp;  // seg = par Rx + r
    const int px = seg >= k.Rx, kx = jx + (seg - px * k.Rx) * k.lrx;
    // this field's rows of the tile
    const Rsrc wb = mx_rsrc(W + ((size_t)(col0 / MX_CB) * a.rows + (size_t)blockIdx.y * a.ny) * MX_CB,
                            (int64_t)a.ny * MX_CB);
    const Rsrc w2 = mx_rsrc(P->w2, a.ny);
    const uint32_t wo = (uint32_t)(col % MX_CB) * 8u;
    constexpr uint32_t ST = MX_CB * 8u;
    float2* lds = (float2*)mx_lds + t.par * k.image;
    mx_conv<QM>(lds, P, t,
        [&](int j, int r, int lr) {
            const float2 x = bload(wb, wo + j * ST, r * lr * ST);
            return t.par ? cmul(x, bload(w2, j * 8u, r * lr * 8u)) : x;
        },
        ColMul<MODE>{a, col_h<MODE>(a, jx < k.lrx ? 2 * kx + px : 0, Mx), t.par, My,
                     mx_rsrc(a.sy, MODE == K_TABLE ? My : 0)},
        ColsOut{{(float2*)mx_lds + k.image, w2, t}, wb, wo});
}

struct FieldOut : MxMeet<float2> {  // pass C: crop, scale, post-chirp, factor field, accumulate, 8-bit phase
    const PropArgs& a;
    Rsrc db;
    uint32_t dof;
    int row;
    bool post;
    float2 cy;
    __device__ __forceinline__ void out(int j, int r, int lr, float2 v) const {
        if (t.par) return;
        const int p = j + r * lr;
        float2 x = cscale(sum(j, r, lr, v), a.scale);
        if (post && abs(p - a.nx / 2) < a.cwl) x = cmul(x, cmul(a.cx[p], cy));
        if (a.post) x = cmul(x, a.post[(size_t)(row % a.ny) * a.nx + p]);
        if (a.accum) x = cadd(bload(db, dof + j * 8u, r * lr * 8u), x);
        bstore(db, dof + j * 8u, r * lr * 8u, x);
    }
};

template <int QM>
__global__ void __launch_bounds__(MX_NT, (QM == 1 ? 6 : 4))
k_mx_rows_inv(const float2* __restrict__ W, float2* __restrict__ dst, PropArgs a,
              const MxPlan<float2>* __restrict__ P, int lognb, int image) {
    const MxPos t = mx_pos<true>(lognb);
    const int nx = a.nx, R = P->b[0].R, lrp = mx_lrp(P->b[0].lr);
    const int row0 = xcd_remap(blockIdx.x, gridDim.x) << lognb, row = row0 + t.c;
    const bool post = a.cx != nullptr && abs(row - a.ny / 2) < a.chl;
    const float2 cy = post && row < a.rows ? a.cy[row] : make_float2(1.f, 0.f);
    const Rsrc wb = mx_rsrc(W, 2ll * R * lrp * a.rows);
    const Rsrc db = mx_rsrc(dst + (size_t)row0 * a.ds, (int64_t)(a.rows - 1 - row0) * a.ds + nx);
    const uint32_t tile = (uint32_t)(a.rows * MX_CB) * 8u, seg = (uint32_t)(lrp / MX_CB) * tile;
    const uint32_t wo = row < a.rows ? (uint32_t)(row * MX_CB) * 8u : 0x80000000u;
    mx_run<QM, true, true>((float2*)mx_lds + t.par * image, P, t,
        [&](int j, int r, int) { return bload(wb, wo + mx_col<float2>(j, tile), (uint32_t)(t.par * R + r) * seg); },
        FieldOut{{(float2*)mx_lds + image, mx_rsrc(P->w2, nx), t}, a, db,
                 row < a.rows ? (uint32_t)(t.c * a.ds) * 8u : 0x80000000u, row, post, cy});
    if (a.img8) {
        // the 8-bit phase of the rows just stored (each thread reads back what another wrote)
        __syncthreads();
        for (int c = 0; c < 1 << lognb && row0 + c < a.rows; c++)
            for (int p = threadIdx.x; p < nx; p += blockDim.x) {
                const size_t i = (size_t)(row0 + c) * a.ds + p;
                store_img8(a, i, dst[i]);
            }
    }
}

template <int QM>
void mx_rows_fwd(unsigned grid, const MxShape& sh, const float2* src, float2* W, const PropArgs& a,
                 const MxPlan<float2>* P, hipStream_t s) {
    k_mx_rows_fwd<QM><<<dim3(grid, 2), sh.nt, sh.lds, s>>>(src, W, a, P, sh.lognb);
}
template <int QM>
void mx_cols_conv(dim3 grid, const MxShape& sh, float2* W, const PropArgs& a, const MxPlan<float2>* P,
                  const MxCols& c, hipStream_t s) {
    const int nt = 2 * sh.nt;
    const size_t lds = 2 * sh.lds;
    if (a.mode == K_ASM) k_mx_cols_conv<QM, K_ASM><<<grid, nt, lds, s>>>(W, a, P, sh.lognb, c);
    else if (a.mode == K_ASHIFT) k_mx_cols_conv<QM, K_ASHIFT><<<grid, nt, lds, s>>>(W, a, P, sh.lognb, c);
    else if (a.mode == K_ASM32) k_mx_cols_conv<QM, K_ASM32><<<grid, nt, lds, s>>>(W, a, P, sh.lognb, c);
    else k_mx_cols_conv<QM, K_TABLE><<<grid, nt, lds, s>>>(W, a, P, sh.lognb, c);
}
template <int QM>
void mx_rows_inv(unsigned grid, const MxShape& sh, const float2* W, float2* dst, const PropArgs& a,
                 const MxPlan<float2>* P, hipStream_t s) {
    k_mx_rows_inv<QM><<<grid, 2 * sh.nt, 2 * sh.lds, s>>>(W, dst, a, P, sh.lognb, sh.image);
}
template void mx_rows_fwd<OLX_MIXPROP_QM>(unsigned, const MxShape&, const float2*, float2*, const PropArgs&,
                                          const MxPlan<float2>*, hipStream_t);
template void mx_cols_conv<OLX_MIXPROP_QM>(dim3, const MxShape&, float2*, const PropArgs&,
                                           const MxPlan<float2>*, const MxCols&, hipStream_t);
template void mx_rows_inv<OLX_MIXPROP_QM>(unsigned, const MxShape&, const float2*, float2*, const PropArgs&,
                                          const MxPlan<float2>*, hipStream_t);
#endif

}  // namespace olx

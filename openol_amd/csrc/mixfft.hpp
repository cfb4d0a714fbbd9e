// mixfft.hpp -- runtime-planned mixed-radix transforms in LDS, for float2 and double2, and the
// pieces of a padded propagation built on them (olx_prop_mr.hip, olx_prop64.hip).
//
// Lengths n whose prime factors are 2, 3, 5, 7, 11 and 13 run as a Stockham FFT: stage s of
// radix R with ns = product of the earlier radices takes butterfly j in [0, n/R) from
// x[j + r n/R], multiplies by W_{ns R}^{k r} (k = j mod ns), applies the R-point DFT and
// writes y[(j - k) R + k + r ns], natural order after the last stage.
//
// Zero padding is never transformed.  The 2n-point spectrum of an n-point field splits into
// its even and odd bins, each an n-point transform:
//   X[2k] = FFT_n(x)[k],   X[2k + 1] = FFT_n(x_j w^j)[k],   w = e^{-2 pi i / 2n},
// and the n kept values of the 2n-point inverse are IFFT(Xe)[j] + conj(w^j) IFFT(Xo)[j]
// (unnormalised).  A field centred in its padding and cropped at the same place is shifted by
// the same amount on the way in and out, which cancels, so the field is taken at offset 0.
// Every stage then works on values that are not zero.  A work-group's first waves take the even bins
// and its last the odd ones; they meet in LDS before the result is stored.
//
// What bounds these passes is the vector work between the LDS exchanges, then the exchanges'
// latency.  Hence: the first stage loads from global memory and the last one stores to it; a
// column pass's last forward stage keeps its values in registers, multiplies them by the
// transfer function and feeds the inverse transform, whose stages run in reversed order so that
// its first radix is the forward transform's last (m stages cost 2m - 2 exchanges); LDS
// addresses and twiddle addresses are linear in r, so an element costs one addition.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "buffer_access.hpp"
#include "fft_core.hpp"
#include "olx_common.hpp"

namespace olx {

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
template <class T> struct Cplx;
template <> struct Cplx<float> { using type = float2; };
template <> struct Cplx<double> { using type = double2; };
template <class C> using real_t = decltype(C::x);
template <class C>
__device__ __forceinline__ C mkc(real_t<C> x, real_t<C> y) {
    C c;
    c.x = x;
    c.y = y;
    return c;
}

// ------------------------------------------------------------------ DFTs in registers
constexpr double kMxPi = 3.141592653589793238462643383279502884;
constexpr double mx_sin(double x) {  // Taylor series after reduction to [-pi, pi]
    while (x > kMxPi) x -= 2 * kMxPi;
    while (x < -kMxPi) x += 2 * kMxPi;
    double term = x, sum = x;
    for (int i = 1; i < 40; i++) {
        term *= -x * x / ((2.0 * i) * (2.0 * i + 1));
        sum += term;
    }
    return sum;
}
constexpr double mx_cos(double x) { return mx_sin(x + kMxPi / 2); }
// cos / sin of 2 pi m / R, evaluated by the compiler: indexed by unrolled loop counters, every
// entry folds to an immediate
template <int R, class T>
struct MxRoots {
    T c[R], s[R];
    constexpr MxRoots() : c(), s() {
        for (int m = 0; m < R; m++) {
            c[m] = (T)mx_cos(2.0 * kMxPi * m / R);
            s[m] = (T)mx_sin(2.0 * kMxPi * m / R);
        }
    }
};
template <int R, class T>
__device__ constexpr MxRoots<R, T> kMxRoots{};

// multiply by W_R^m (forward e^{-2 pi i m / R}); m known after unrolling
template <int R, bool INV, class C>
__device__ __forceinline__ C mx_tw(int m, C a) {
    m %= R;
    if (m == 0) return a;
    if (4 * m == R) return INV ? mkc<C>(-a.y, a.x) : mkc<C>(a.y, -a.x);
    if (2 * m == R) return mkc<C>(-a.x, -a.y);
    if (4 * m == 3 * R) return INV ? mkc<C>(a.y, -a.x) : mkc<C>(-a.y, a.x);
    const auto c = kMxRoots<R, real_t<C>>.c[m];
    const auto s = INV ? kMxRoots<R, real_t<C>>.s[m] : -kMxRoots<R, real_t<C>>.s[m];
    return mkc<C>(a.x * c - a.y * s, a.x * s + a.y * c);
}

template <int R, bool INV, class C>
__device__ __forceinline__ void mx_dft(C* v);

// Good's prime-factor form for coprime A, B: n = B n1 + A n2, k = k1 mod A = k2 mod B, no
// twiddles (15 points: 178 operations against 266 by symmetric pairs)
template <int A, int B>
__host__ __device__ constexpr int mx_crt(int k1, int k2) {
    int k = k1;
    while (k % B != k2) k += A;
    return k;
}
template <int A, int B, bool INV, class C>
__device__ __forceinline__ void mx_pfa(C* v) {
    C t[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; n2++) {
#pragma unroll
        for (int n1 = 0; n1 < A; n1++) t[n2][n1] = v[(B * n1 + A * n2) % (A * B)];
        mx_dft<A, INV>(t[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; k1++) {
        C u[B];
#pragma unroll
        for (int n2 = 0; n2 < B; n2++) u[n2] = t[n2][k1];
        mx_dft<B, INV>(u);
#pragma unroll
        for (int k2 = 0; k2 < B; k2++) v[mx_crt<A, B>(k1, k2)] = u[k2];
    }
}

// R-point DFT, natural order in and out
template <int R, bool INV, class C>
__device__ __forceinline__ void mx_dft(C* v) {
    if constexpr (R == 2) {
        const C t = v[0];
        v[0] = cadd(t, v[1]);
        v[1] = csub(t, v[1]);
    } else if constexpr (R == 4) {
        const C t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
        const C t2 = cadd(v[1], v[3]), t3 = mx_tw<4, INV>(1, csub(v[1], v[3]));
        v[0] = cadd(t0, t2);
        v[2] = csub(t0, t2);
        v[1] = cadd(t1, t3);
        v[3] = csub(t1, t3);
    } else if constexpr (R == 8 || R == 16) {
        // n = Q n1 + n2, k = k1 + 4 k2
        constexpr int Q = R / 4;
        C b[Q][4];
#pragma unroll
        for (int n2 = 0; n2 < Q; n2++) {
#pragma unroll
            for (int n1 = 0; n1 < 4; n1++) b[n2][n1] = v[Q * n1 + n2];
            mx_dft<4, INV>(b[n2]);
#pragma unroll
            for (int k1 = 1; k1 < 4; k1++) b[n2][k1] = mx_tw<R, INV>(n2 * k1, b[n2][k1]);
        }
#pragma unroll
        for (int k1 = 0; k1 < 4; k1++) {
            C c[Q];
#pragma unroll
            for (int n2 = 0; n2 < Q; n2++) c[n2] = b[n2][k1];
            mx_dft<Q, INV>(c);
#pragma unroll
            for (int k2 = 0; k2 < Q; k2++) v[k1 + 4 * k2] = c[k2];
        }
    } else if constexpr (R == 6) {
        mx_pfa<2, 3, INV>(v);
    } else if constexpr (R == 10) {
        mx_pfa<2, 5, INV>(v);
    } else if constexpr (R == 12) {
        mx_pfa<3, 4, INV>(v);
    } else if constexpr (R == 14) {
        mx_pfa<2, 7, INV>(v);
    } else if constexpr (R == 15) {
        mx_pfa<3, 5, INV>(v);
    } else {
        // odd R: a_n = x_n + x_{R-n}, b_n = x_n - x_{R-n} (n = 1 .. H), then
        // y_k = A_k -/+ i B_k, y_{R-k} = A_k +/- i B_k with A_k = x_0 + sum a_n cos,
        // B_k = sum b_n sin (angles 2 pi n k / R; upper signs forward)
        constexpr int H = (R - 1) / 2;
        C a[H], b[H];
        C y0 = v[0];
#pragma unroll
        for (int n = 1; n <= H; n++) {
            a[n - 1] = cadd(v[n], v[R - n]);
            b[n - 1] = csub(v[n], v[R - n]);
            y0 = cadd(y0, a[n - 1]);
        }
        const C x0 = v[0];
        v[0] = y0;
#pragma unroll
        for (int k = 1; k <= H; k++) {
            C A = x0, B = mkc<C>(0, 0);
#pragma unroll
            for (int n = 1; n <= H; n++) {
                const auto c = kMxRoots<R, real_t<C>>.c[(n * k) % R];
                const auto s = kMxRoots<R, real_t<C>>.s[(n * k) % R];
                A = mkc<C>(fma(a[n - 1].x, c, A.x), fma(a[n - 1].y, c, A.y));
                B = mkc<C>(fma(b[n - 1].x, s, B.x), fma(b[n - 1].y, s, B.y));
            }
            const C up = mkc<C>(A.x + B.y, A.y - B.x), dn = mkc<C>(A.x - B.y, A.y + B.x);
            v[k] = INV ? dn : up;
            v[R - k] = INV ? up : dn;
        }
    }
}

// ------------------------------------------------------------------ plan
constexpr int MX_MAXST = 14;
struct MxStage {
    int R;         // radix
    int ns;        // product of the earlier radices
    int lr;        // n / R, butterflies of a transform
    uint32_t mns;  // fast-division magic of ns
    // LDS image before this stage: element p at p + (p / ns) rpad.  Every earlier product
    // divides n / R, so x[j + r lr] sits at j + (j / ns) rpad + r rstep, and this stage's
    // writes, into the next stage's image, at (j / ns) wblk + k + r ns.
    int rpad, rstep, wblk;
    int off;       // twiddles W_{ns R}^{k r} at tab[off + (r - 1) ns + k]: the lanes' k are contiguous
};
template <class C>
struct MxPlan {
    int n, nst, ntab;
    const C* w2;   // w^j = e^{-2 pi i j / 2n}, j in [0, n)
    const C* tab;  // stage twiddles
    MxStage f[MX_MAXST], b[MX_MAXST];  // the stages, and in reversed order for the inverse
};

// n / d for n, d < 2^16 (n d < 2^32): magic m = floor(2^32 / d) + 1
__host__ __device__ constexpr uint32_t mx_magic(int d) {
    return d <= 1 ? 0u : (uint32_t)((0x100000000ull / (uint64_t)d) + 1);
}
__device__ __forceinline__ int mx_div(int n, int d, uint32_t m) {
    return d == 1 ? n : (int)__umulhi((uint32_t)n, m);
}

// Butterflies a thread holds in a stage of radix R: about 16 values, and few butterflies (each takes address
// registers: 8 of radix 2 spilled).  QM 1 is the complex64 passes', 0 the complex128 ones' (the smaller counts
// keep their threads: 4% faster at 2100^2, 9% at 2450^2).  QM = 2 doubles them, for lengths whose two halves
// would need more than 1024 threads (all above 4096) or leave the CU emptier (mx_qm).
__host__ __device__ constexpr int mx_q(int R, int QM) {
    if (QM == 1) return R == 2 ? 6 : (R == 3 ? 4 : (R <= 5 ? 3 : (R <= 8 ? 2 : 1)));
    return (QM == 2 ? 2 : 1) * (R == 2 ? 4 : (R == 3 ? 3 : (R <= 8 ? 2 : 1)));
}

// A work-group's place in its transforms: nb = 2^lognb of them interleaved in LDS (element a of
// transform c at a nb + c) so that nb neighbouring rows or columns share their lines;
// thread tid owns transform c = tid mod nb and butterflies j0 + jstep q
struct MxPos {
    int c, lognb, j0, jstep, par;
    bool solo;  // a half is one wave: its exchanges need no work-group barrier
};
// With BOTH, the first half of the threads (whole waves) take the even bins and the others the odd
// ones, each in an LDS image of its own.
template <bool BOTH>
__device__ __forceinline__ MxPos mx_pos(int lognb) {
    const int nt = BOTH ? (int)blockDim.x / 2 : (int)blockDim.x;
    const int par = BOTH ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >= nt) : 0;
    const int tid = (int)threadIdx.x - par * nt;
    return MxPos{tid & ((1 << lognb) - 1), lognb, tid >> lognb, nt >> lognb, par, nt == 64};
}
// Between an exchange's accesses of different threads.  A wave's LDS accesses complete in order, so one
// wave on its own only has to keep the compiler from moving them.
__device__ __forceinline__ void mx_sync(const MxPos& t) {
    if (t.solo) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

template <int R, class C>
__device__ __forceinline__ void mx_read(const C* lds, const MxStage& S, const MxPos& t, int j, C* v) {
    const int a = j + mx_div(j, S.ns, S.mns) * S.rpad;
    const C* p = lds + (a << t.lognb) + t.c;
#pragma unroll
    for (int r = 0; r < R; r++) v[r] = p[(r * S.rstep) << t.lognb];
}
template <int R, class C>
__device__ __forceinline__ void mx_write(C* lds, const MxStage& S, const MxPos& t, int j, const C* v) {
    const int jq = mx_div(j, S.ns, S.mns), k = j - jq * S.ns;
    C* p = lds + ((jq * S.wblk + k) << t.lognb) + t.c;
#pragma unroll
    for (int r = 0; r < R; r++) p[(r * S.ns) << t.lognb] = v[r];
}
// a butterfly's twiddles, w[r - 1] = W_{ns R}^{k r}: loaded with its values, ahead of the barrier, so
// that their latency passes while the other waves arrive
template <int R, class C>
__device__ __forceinline__ void mx_twload(const MxStage& S, Rsrc tab, int j, C* w) {
    const int k = j - mx_div(j, S.ns, S.mns) * S.ns;
    const uint32_t vo = (uint32_t)(k * sizeof(C));
    const uint32_t so = (uint32_t)(S.off * sizeof(C)), st = (uint32_t)(S.ns * sizeof(C));
#pragma unroll
    for (int r = 1; r < R; r++) w[r - 1] = bloadc<C>(tab, vo, so + (r - 1) * st);
}
template <int R, bool INV, class C>
__device__ __forceinline__ void mx_twiddle(const C* w, C* v) {
#pragma unroll
    for (int r = 1; r < R; r++) v[r] = cmul(v[r], INV ? cconj(w[r - 1]) : w[r - 1]);
}

// the last stage's outputs: after a barrier where the two halves of the bins meet in LDS
template <int R, int QM, class C, class ST>
__device__ __forceinline__ void mx_out(const MxPos& t, int j0, int lr, const C (*v)[R], ST&& st) {
    if (st.meet) __syncthreads();
#pragma unroll
    for (int q = 0; q < mx_q(R, QM); q++) {
        const int j = j0 + t.jstep * q;
        if (j < lr) {
#pragma unroll
            for (int r = 0; r < R; r++) st.out(j, r, lr, v[q][r]);
        }
    }
}

// One stage.  ld(j, r) gives input j + r lr of the first stage, st takes output
// j + r lr of the last one.
// Both see r times a uniform stride beside a per-thread offset, so their addresses take one
// register each (buffer_access.hpp); a 64-bit address per value spilled hundreds.  The
// scheduling fences keep one butterfly's values live at a time.
template <int R, int QM, bool INV, class C, class LD, class ST>
__device__ __forceinline__ void mx_stage(C* lds, const MxStage& S, Rsrc tab, const MxPos& t, bool first,
                                         bool last, LD&& ld, ST&& st) {
    constexpr int Q = mx_q(R, QM);
    // twiddles ahead of the barrier, where there are registers: at QM = 2 up to 92 spilled, 18% of 6000^2
    constexpr bool AHEAD = sizeof(C) == 8 && QM == 1;
    int j0 = t.j0;
    // formed anew in each stage: hoisted out of the stage loop, the offsets of every radix's
    // butterflies spilled
    asm volatile("" : "+v"(j0));
    C v[Q][R], w[Q][R - 1];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int j = j0 + t.jstep * q;
        if (j < S.lr) {
            if (first) {
#pragma unroll
                for (int r = 0; r < R; r++) v[q][r] = ld(j, r, S.lr);
            } else {
                mx_read<R>(lds, S, t, j, v[q]);
                if (AHEAD) mx_twload<R>(S, tab, j, w[q]);
            }
        }
    }
    // before a first stage no wave reads the image any more: a preceding last stage's reads
    // all came before its own barrier
    if (!first) mx_sync(t);
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int j = j0 + t.jstep * q;
        if (j < S.lr) {
            if (!first) {
                if (!AHEAD) mx_twload<R>(S, tab, j, w[q]);
                mx_twiddle<R, INV>(w[q], v[q]);
            }
            mx_dft<R, INV>(v[q]);
            if (last) {
#pragma unroll
                for (int r = 0; r < R; r++) st.put(j, r, S.lr, v[q][r]);
            } else {
                mx_write<R>(lds, S, t, j, v[q]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if (!last) mx_sync(t);
    else mx_out<R, QM>(t, j0, S.lr, v, st);
}

// The last forward stage, the transfer function h(j, r) and the first inverse stage, in registers
template <int R, int QM, class C, class LD, class H, class ST>
__device__ __forceinline__ void mx_turn(C* lds, const MxStage& S, const MxStage& SB, Rsrc tab,
                                        const MxPos& t, bool only, LD&& ld, H&& h, ST&& st) {
    constexpr int Q = mx_q(R, QM);
    // twiddles ahead of the barrier, where there are registers: at QM = 2 up to 92 spilled, 18% of 6000^2
    constexpr bool AHEAD = sizeof(C) == 8 && QM == 1;
    int j0 = t.j0;
    // formed anew in each stage: hoisted out of the stage loop, the offsets of every radix's
    // butterflies spilled
    asm volatile("" : "+v"(j0));
    C v[Q][R], w[Q][R - 1];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int j = j0 + t.jstep * q;
        if (j < S.lr) {
            if (only) {
#pragma unroll
                for (int r = 0; r < R; r++) v[q][r] = ld(j, r, S.lr);
            } else {
                mx_read<R>(lds, S, t, j, v[q]);
                if (AHEAD) mx_twload<R>(S, tab, j, w[q]);
            }
        }
    }
    if (!only) mx_sync(t);
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int j = j0 + t.jstep * q;
        if (j < S.lr) {
            if (!only) {
                if (!AHEAD) mx_twload<R>(S, tab, j, w[q]);
                mx_twiddle<R, false>(w[q], v[q]);
            }
            mx_dft<R, false>(v[q]);
            h.template mul<R>(j, S.lr, v[q]);
            mx_dft<R, true>(v[q]);
            if (only) {
#pragma unroll
                for (int r = 0; r < R; r++) st.put(j, r, S.lr, v[q][r]);
            } else {
                mx_write<R>(lds, SB, t, j, v[q]);  // SB.ns = 1
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if (!only) mx_sync(t);
    else mx_out<R, QM>(t, j0, S.lr, v, st);
}

#define MX_RADIX_SWITCH(R_, ...)                          \
    switch (R_) {                                         \
        case 2: { constexpr int R = 2; __VA_ARGS__; } break;   \
        case 3: { constexpr int R = 3; __VA_ARGS__; } break;   \
        case 4: { constexpr int R = 4; __VA_ARGS__; } break;   \
        case 5: { constexpr int R = 5; __VA_ARGS__; } break;   \
        case 6: { constexpr int R = 6; __VA_ARGS__; } break;   \
        case 7: { constexpr int R = 7; __VA_ARGS__; } break;   \
        case 8: { constexpr int R = 8; __VA_ARGS__; } break;   \
        case 9: { constexpr int R = 9; __VA_ARGS__; } break;   \
        case 10: { constexpr int R = 10; __VA_ARGS__; } break; \
        case 11: { constexpr int R = 11; __VA_ARGS__; } break; \
        case 12: { constexpr int R = 12; __VA_ARGS__; } break; \
        case 13: { constexpr int R = 13; __VA_ARGS__; } break; \
        case 14: { constexpr int R = 14; __VA_ARGS__; } break; \
        case 15: { constexpr int R = 15; __VA_ARGS__; } break; \
        default: { constexpr int R = 16; __VA_ARGS__; } break; \
    }

// outputs of a stage that is not the last
struct MxNone {
    static constexpr bool meet = false;
    template <class C> __device__ void put(int, int, int, C) const {}
    template <class C> __device__ void out(int, int, int, C) const {}
};
template <class C>
__device__ __forceinline__ Rsrc mx_tab(const MxPlan<C>* __restrict__ P) {
    return make_rsrc(P->tab, (size_t)P->ntab * sizeof(C));
}
// n-point transform of the nb sequences, from ld to st; REV takes the stages in reversed order
template <int QM, bool INV, bool REV, class C, class LD, class ST>
__device__ __forceinline__ void mx_run(C* lds, const MxPlan<C>* __restrict__ P, const MxPos& t, LD&& ld,
                                       ST&& st) {
    const int m = P->nst;
    const Rsrc tab = mx_tab(P);
#pragma unroll 1
    for (int s = 0; s < m; s++) {
        const MxStage S = REV ? P->b[s] : P->f[s];
        MX_RADIX_SWITCH(S.R, mx_stage<R, QM, INV>(lds, S, tab, t, s == 0, s == m - 1, ld, st));
    }
}
// forward transform, h, inverse transform
template <int QM, class C, class LD, class H, class ST>
__device__ __forceinline__ void mx_conv(C* lds, const MxPlan<C>* __restrict__ P, const MxPos& t, LD&& ld,
                                        H&& h, ST&& st) {
    const int m = P->nst;
    const Rsrc tab = mx_tab(P);
    const MxNone no_st;
    const auto no_ld = [](int, int, int) { return C{}; };
#pragma unroll 1
    for (int s = 0; s < m - 1; s++) {
        const MxStage S = P->f[s];
        MX_RADIX_SWITCH(S.R, mx_stage<R, QM, false>(lds, S, tab, t, s == 0, false, ld, no_st));
    }
    {
        const MxStage S = P->f[m - 1], SB = P->b[0];
        MX_RADIX_SWITCH(S.R, mx_turn<R, QM>(lds, S, SB, tab, t, m == 1, ld, h, st));
    }
#pragma unroll 1
    for (int s = 1; s < m; s++) {
        const MxStage S = P->b[s];
        MX_RADIX_SWITCH(S.R, mx_stage<R, QM, true>(lds, S, tab, t, false, s == m - 1, no_ld, st));
    }
}

// ------------------------------------------------------------------ intermediate
// W: tiles of MX_CB columns of every row.  A row pass's thread holds bins j + r lr of a half (lr =
// n / R of its last stage), so column (par R + r) lrp + j, lrp = lr rounded up to whole tiles, makes its
// address linear in r.  The plan's last radix is one that pads little; padding columns are never
// written, and what the column pass makes of them is never read.  The column pass's nb columns of a row
// are contiguous, and a row pass writes MX_CB values of each of its rows side by side.
constexpr int MX_CB = 4;
__host__ __device__ inline int mx_lrp(int lr) { return (lr + MX_CB - 1) / MX_CB * MX_CB; }
// byte offset of column j (of r = 0, the first half) of a row, tile bytes apart, and the step of r
template <class C>
__device__ __forceinline__ uint32_t mx_col(int j, uint32_t tile) {
    return (uint32_t)(j / MX_CB) * tile + (uint32_t)(j % MX_CB) * (uint32_t)sizeof(C);
}

// descriptors of `count` values from p (none past the first 2 GiB; every access lies in them)
template <class C>
__device__ __forceinline__ Rsrc mx_rsrc(const C* p, int64_t count) {
    const int64_t b = count * (int64_t)sizeof(C);
    return make_rsrc(p, (size_t)(b < 0 ? 0 : (b > 0x7fffffff ? 0x7fffffff : b)));
}

// the odd half's results, times conj(w^p), wait in its LDS image (which no stage reads any more) for
// the even half to add
template <class C>
struct MxMeet {
    static constexpr bool meet = true;
    C* odd;
    Rsrc w2;
    MxPos t;
    __device__ __forceinline__ void put(int j, int r, int lr, C v) const {
        if (t.par) odd[((j + r * lr) << t.lognb) + t.c] = cmul(cconj(bloadc<C>(w2, j * (uint32_t)sizeof(C), r * lr * (uint32_t)sizeof(C))), v);
    }
    __device__ __forceinline__ C sum(int j, int r, int lr, C v) const {
        return cadd(v, odd[((j + r * lr) << t.lognb) + t.c]);
    }
};

template <class C>
struct MxRowsOut {  // pass A: a half's bins into W
    static constexpr bool meet = false;
    Rsrc wb;
    uint32_t wo, tile, seg;
    int first;  // par R
    __device__ __forceinline__ void put(int, int, int, C) const {}
    __device__ __forceinline__ void out(int j, int r, int, C v) const {
        bstorec(wb, wo + mx_col<C>(j, tile), (uint32_t)(first + r) * seg, v);
    }
};

// ------------------------------------------------------------------ host side
constexpr size_t MX_LDS = 160 * 1024;  // of a CU
struct MxShape {  // launch shape of a plan with 2^lognb transforms a work-group
    int lognb, nt;
    int qm;       // mx_q's QM
    int rlast;    // radix of the last stage
    int image;    // LDS values of the transforms (of one half of the bins)
    size_t lds;   // bytes
};
struct MxHost {
    int n = 0, nst = 0;
    MxStage f[MX_MAXST], b[MX_MAXST];
    int ntab = 0;
    int image = 0;  // LDS values of one transform, padding included
    int held[4] = {0, 0, 0, 0};  // transforms on a CU with 2^l a work-group (mx_fit; 0: it does not fit)
    MxShape shape[2];            // of the passes of one and of two halves a work-group
    std::string key;             // of the device plan in the context's tables
};

// relative cost of a point in a stage of radix R: the exchange and twiddles, and the DFT (radices
// below 5 occupy many threads for little work)
inline double mx_cost(int R) {
    static const double d[17] = {0, 0, 2, 4.7, 4, 7.2, 6.7, 9.4, 7, 11.5, 9.2, 13.5, 8.7, 15.7, 11.4, 11.9, 10.5};
    return (R < 5 ? 22.0 : 16.0) + d[R];
}
// cheapest radices (non-increasing) of n; false when n has a prime factor above 13
inline bool mx_radices(int n, int top, std::vector<int>& best, double* cost) {
    if (n == 1) {
        best.clear();
        *cost = 0;
        return true;
    }
    bool ok = false;
    *cost = 1e300;
    for (int r = top; r >= 2; r--) {
        if (n % r) continue;
        std::vector<int> rest;
        double c;
        if (!mx_radices(n / r, r, rest, &c) || c + mx_cost(r) >= *cost) continue;
        *cost = c + mx_cost(r);
        best.assign(1, r);
        best.insert(best.end(), rest.begin(), rest.end());
        ok = true;
    }
    return ok;
}
// threads for nb transforms: every stage's butterflies fit.  The complex64 passes take the larger counts of
// mx_q(R, 1) only where the smaller would need more than three waves a SIMD (1125^2 96 us with them, 88 without).
inline int mx_threads(const MxHost& P, int nb, int qm) {
    const auto need = [&](int m) {
        int nt = 64;
        for (int s = 0; s < P.nst; s++) {
            const int q = mx_q(P.f[s].R, m);
            nt = std::max(nt, ((P.f[s].lr + q - 1) / q * nb + 63) / 64 * 64);
        }
        return nt;
    };
    const int nt = need(qm == 1 ? 0 : qm);
    return qm == 1 && nt > 384 ? need(1) : nt;
}

// Bank conflicts of the writes of stage (R, ns) into the next image padded by `pad` a block:
// LDS serves 256 bytes a cycle (256 / eb lanes of eb bytes each).
inline int mx_conflicts(int n, int R, int ns, int pad, int nb, int eb) {
    const int lanes = std::min(32, 256 / eb), lr = n / R;
    int worst = 0;
    for (int g0 = 0; g0 < 64; g0 += lanes) {
        std::vector<int> hit(256 / eb, 0);
        int mx = 0;
        for (int l = g0; l < g0 + lanes; l++) {
            const int j = l / nb, c = l % nb;
            if (j >= lr) continue;
            const int a = ((j / ns) * (ns * R + pad) + j % ns) * nb + c;
            mx = std::max(mx, ++hit[a % (256 / eb)]);
        }
        worst += mx;
    }
    return worst;
}

inline bool mx_plan_host(int n, int eb, int nb, MxHost& P) {
    std::vector<int> rx;
    double c;
    if (!mx_radices(n, 16, rx, &c) || (int)rx.size() > MX_MAXST) return false;
    // the last radix: the one whose columns pad least (mx_lrp)
    for (size_t i = 0; i + 1 < rx.size(); i++)
        if (rx[i] * mx_lrp(n / rx[i]) < rx.back() * mx_lrp(n / rx.back())) std::swap(rx[i], rx.back());
    P.n = n;
    P.nst = (int)rx.size();
    P.image = n;
    P.ntab = 0;
    for (int dir = 0; dir < 2; dir++) {
        MxStage* st = dir ? P.b : P.f;
        if (dir) std::reverse(rx.begin(), rx.end());
        int ns = 1, pad = 0;
        for (int s = 0; s < P.nst; s++) {
            MxStage& S = st[s];
            S.R = rx[s];
            S.ns = ns;
            S.lr = n / S.R;
            S.mns = mx_magic(ns);
            S.rpad = pad;
            S.rstep = S.lr + pad * (S.lr / ns);
            S.off = P.ntab;
            if (s > 0) P.ntab += ns * (S.R - 1);
            int np = 0;
            if (s + 1 < P.nst) {
                int best = 1 << 30;
                // padding adds at most an eighth: the longest halves, 8192 values of 8 bytes or
                // 4096 of 16, then fit the LDS together
                for (int q = 0; q < 4 && 8 * q <= ns * S.R; q++) {
                    const int k = mx_conflicts(n, S.R, ns, q, nb, eb);
                    if (k < best) {
                        best = k;
                        np = q;
                    }
                }
                P.image = std::max(P.image, n + n / (ns * S.R) * np);
            }
            S.wblk = ns * S.R + np;
            pad = np;
            ns *= S.R;
        }
    }
    return true;
}

template <class C>
__global__ void k_mx_tables(C* __restrict__ w2, C* __restrict__ tab, MxPlan<C> plan, MxPlan<C>* __restrict__ dst) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e == 0) *dst = plan;
    double s, c;
    if (e < plan.n) {
        sincospi(-(double)e / (double)plan.n, &s, &c);
        w2[e] = mkc<C>((real_t<C>)c, (real_t<C>)s);
    }
    for (int d = 0; d < 2; d++)
        for (int q = 1; q < plan.nst; q++) {
            const MxStage& S = d ? plan.b[q] : plan.f[q];
            if (e < S.off || e >= S.off + S.ns * (S.R - 1)) continue;
            const int loc = e - S.off, r = loc / S.ns + 1, k = loc % S.ns;
            sincospi(-2.0 * (double)(k * r) / (double)(S.ns * S.R), &s, &c);
            tab[e] = mkc<C>((real_t<C>)c, (real_t<C>)s);
        }
}

// QM of the passes that hold their values in a thread's fewest registers
template <class C> constexpr int mx_base() { return sizeof(C) == 8 ? 1 : 0; }
// Work-groups of `halves` images on a CU, and their waves.  A SIMD holds 6 waves of the complex64 passes (4 at
// QM = 2), 3 of the complex128 ones (4 above 512 threads, in fewer registers), and a work-group's waves go
// round the four SIMDs, so 6 of them take two places on each.
struct MxHold {
    int groups, waves;
};
template <class C>
inline MxHold mx_hold(const MxHost& H, int lognb, int qm, int halves) {
    const int w = halves * mx_threads(H, 1 << lognb, qm) / 64;
    const int per = sizeof(C) == 16 ? (w <= 8 ? 3 : 4) : (qm == 2 ? 4 : 6);
    const size_t lds = halves * sizeof(C) * ((size_t)H.image << lognb);
    const int groups = std::min(w < 4 ? 4 * per / w : per / ((w + 3) / 4), (int)(MX_LDS / lds));
    return MxHold{groups, groups * w};
}

// QM of a pass of `halves` images a work-group: 2 where 1 needs too many threads, and where it puts more
// work-groups on a CU with no fewer waves, since the one waits for its exchanges while the others run
// (14 waves alone / 8 and 8: 3718^2 1092 / 940 us, 4000^2 1097 / 869, 4160^2 1240 / 1011, 3432^2 824 / 686).
template <class C>
inline int mx_qm(const MxHost& H, int lognb, int maxnt, int halves) {
    if (halves * mx_threads(H, 1 << lognb, mx_base<C>()) > maxnt) return 2;
    if (sizeof(C) != 8 || lognb > 0) return mx_base<C>();
    const MxHold a = mx_hold<C>(H, 0, 1, halves), b = mx_hold<C>(H, 0, 2, halves);
    return b.groups > a.groups && b.waves >= a.waves ? 2 : 1;
}
// Launch shape.  A work-group alone on its CU takes all the threads it can (6000^2 2475 -> 2180 us, 5280^2 2069 ->
// 1804, 6804^2 3613 -> 3160 against the fewest that hold its butterflies); the complex64 passes' waves are whole
// rounds of the four SIMDs (10 -> 12 waves: 2420^2 395 -> 369 us, 2600^2 445 -> 395, 3528^2 712 -> 617).
template <class C>
inline MxShape mx_shape(const MxHost& H, int lognb, int maxnt, int halves) {
    MxShape s;
    s.lognb = lognb;
    s.qm = mx_qm<C>(H, lognb, maxnt, halves);
    s.nt = mx_threads(H, 1 << lognb, s.qm);
    if (s.qm == 2 && mx_hold<C>(H, lognb, 2, halves).groups == 1) s.nt = std::max(s.nt, maxnt / halves);
    const int w = halves * s.nt / 64;
    if (sizeof(C) == 8 && w > 4) s.nt = (w + 3) / 4 * 256 / halves;
    s.rlast = H.f[H.nst - 1].R;
    s.image = H.image << lognb;
    s.lds = sizeof(C) * (size_t)s.image;
    return s;
}

// the host side of a plan, kept in the context (the search of a length's radices, and the launch shapes, would
// otherwise be spent on every call)
template <class C>
inline const MxHost* mx_host(olx_ctx* ctx, int n, int lognb, int maxnt) {
    auto& slot = ctx->mx_hosts[((uint64_t)n << 16) | (uint64_t)(sizeof(C) << 4) | (uint64_t)lognb];
    if (!slot) {
        auto H = std::make_shared<MxHost>();
        if (!mx_plan_host(n, (int)sizeof(C), 1 << lognb, *H)) return nullptr;
        for (int l = 0; lognb == 0 && l < 4; l++) {
            const MxHost* G = l ? mx_host<C>(ctx, n, l, maxnt) : H.get();
            if (2 * mx_threads(*G, 1 << l, mx_base<C>()) > maxnt || 2 * sizeof(C) * ((size_t)G->image << l) > MX_LDS) break;
            H->held[l] = mx_hold<C>(*G, l, mx_base<C>(), 2).groups << l;
        }
        for (int h = 1; h <= 2; h++) H->shape[h - 1] = mx_shape<C>(*H, lognb, maxnt, h);
        char key[64];
        snprintf(key, sizeof key, "mx%d|%d|%d", (int)sizeof(C), n, lognb);
        H->key = key;
        slot = H;
    }
    return (const MxHost*)slot.get();
}

// Transforms (2^lognb, lognb <= hi) of a work-group: the number that keeps the most of a pass's `total`
// transforms on a CU, the fewest where several do.  Measured: 2160-point columns 345 us with one, 313 with two;
// 1500 (complex128) 323 and 222; 1080 197 and 245; 156-point rows 63 with one, 52 with four.
template <class C>
inline int mx_fit(olx_ctx* ctx, int n, int64_t total, int hi, int maxnt) {
    const MxHost* H = mx_host<C>(ctx, n, 0, maxnt);
    int best = 0;
    int64_t most = 0;
    for (int l = 0; H && l <= hi && H->held[l]; l++) {
        const int64_t held = std::min<int64_t>(H->held[l], (total + 255) / 256);
        if (held > most) {
            most = held;
            best = l;
        }
    }
    return best;
}

// the device-resident plan of n-point transforms, 2^lognb a work-group (built on first use)
template <class C>
inline int mx_plan(olx_ctx* ctx, int n, int lognb, int maxnt, const MxPlan<C>** out, MxShape* shape) {
    const MxHost* H = mx_host<C>(ctx, n, lognb, maxnt);
    if (!H) OLX_FAIL(OLX_EUNSUPPORTED, "transform length %d: prime factors must be 2, 3, 5, 7, 11, 13", n);
    *shape = H->shape[1];
    bool fresh = false;
    int rc = OLX_OK;
    const size_t nw = (size_t)n + (size_t)(n & 1), nt = (size_t)H->ntab + (size_t)(H->ntab & 1);
    const size_t bytes = sizeof(C) * (nw + nt) + sizeof(MxPlan<C>);
    char* mem = (char*)table(ctx, H->key, (bytes + sizeof(float2) - 1) / sizeof(float2), &fresh, &rc);
    if (!mem) return rc;
    C* w2 = (C*)mem;
    C* tab = w2 + nw;
    MxPlan<C>* d = (MxPlan<C>*)(tab + nt);
    if (fresh) {
        MxPlan<C> P;
        memset(&P, 0, sizeof P);
        P.n = n;
        P.nst = H->nst;
        P.ntab = H->ntab;
        P.w2 = w2;
        P.tab = tab;
        memcpy(P.f, H->f, sizeof(MxStage) * H->nst);
        memcpy(P.b, H->b, sizeof(MxStage) * H->nst);
        const int total = std::max(n, H->ntab);
        k_mx_tables<C><<<(total + 255) / 256, 256, 0, ctx->stream>>>(w2, tab, P, d);
        OLX_TRY(check_launch("mixed-radix plan"));
    }
    *out = d;
    return OLX_OK;
}

}  // namespace olx

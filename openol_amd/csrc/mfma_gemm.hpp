// mfma_gemm.hpp -- the complex GEMM of the point-cloud holograms on MFMA (gfx950),
// shared by the layered CGH (olx_layered.hip) and the direct Fresnel CGH
// (olx_cgh_mfma.hip).
//
//   U[h][w] = sum_j Y_j(h) X_j(w)    as two real GEMMs over interleaved columns:
//   Re U = A Br^T, Im U = A Bi^T,  A = [Re Y, Im Y], Br = [Re X, -Im X], and Bi formed
//   from Br in registers (a half swap and one sign bit).
//
// Factors are 16-bit (FP16 or BF16), products accumulate in FP32.  A SPLIT product
// carries each factor as hi + lo (two 16-bit values) and forms hi hi + lo hi + hi lo.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "olx_common.hpp"

namespace olx {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef float f16v_t __attribute__((ext_vector_type(16)));

constexpr int KS = 64;          // halves of a factor row per LDS stage
constexpr int ROWB = KS * 2;    // bytes per LDS row
constexpr int GTN = 128;        // work-group tile columns
constexpr int GEMM_CUS = 256;   // compute units a launch should fill

// Factor rows.  Plain: 2 halves per point, point j at halves 2 j, 2 j + 1 (a stage is 32
// points).  SPLIT: 4 halves per point, in groups of 16 points: 32 halves of hi then the
// same 32 of lo (a stage is one group), so both forms stage 128 bytes a row alike.
template <bool SPLIT>
constexpr int stage_pts() { return SPLIT ? 16 : 32; }
// 32-bit word of point j's hi value in its factor row (the lo value is 16 words on)
template <bool SPLIT>
__host__ __device__ constexpr int fac_word(int j) { return SPLIT ? (j / 16) * 32 + j % 16 : j; }

template <typename T>
__device__ inline uint32_t pack2(float a, float b, float* ra, float* rb);
template <>
__device__ inline uint32_t pack2<_Float16>(float a, float b, float* ra, float* rb) {
    const _Float16 x = (_Float16)a, y = (_Float16)b;
    *ra = (float)x;
    *rb = (float)y;
    return (uint32_t)__builtin_bit_cast(uint16_t, x) | ((uint32_t)__builtin_bit_cast(uint16_t, y) << 16);
}
template <>
__device__ inline uint32_t pack2<__bf16>(float a, float b, float* ra, float* rb) {
    const __bf16 x = (__bf16)a, y = (__bf16)b;
    *ra = (float)x;
    *rb = (float)y;
    return (uint32_t)__builtin_bit_cast(uint16_t, x) | ((uint32_t)__builtin_bit_cast(uint16_t, y) << 16);
}

// Bi operand from Br: per dword (lo = Re X, hi = -Im X) -> (lo = Im X, hi = Re X)
__device__ inline uint32_t bi_of_br(uint32_t w) {
    const uint32_t sw = (w >> 16) | (w << 16);  // (lo = -Im X, hi = Re X)
    return sw ^ 0x00008000u;                    // negate the low half
}

template <typename T>
__device__ inline f16v_t mfma(const uint4& a, const uint4& b, f16v_t c);
template <>
__device__ inline f16v_t mfma<_Float16>(const uint4& a, const uint4& b, f16v_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a),
                                                  __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
}
template <>
__device__ inline f16v_t mfma<__bf16>(const uint4& a, const uint4& b, f16v_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8_t, a),
                                                   __builtin_bit_cast(bf8_t, b), c, 0, 0, 0);
}

// Work-group tile: 64 WR x 128 outputs by 2 WR waves in a WR x 2 grid, each owning 64 x 64
// (8 MFMAs per 16-wide K step and product).  WR = 4 (8 waves, two per SIMD) moves the
// fewest factor bytes per output; WR = 2 halves the tile where whole 256-row tiles would
// leave compute units idle (gemm_plan).
// Stages go from global memory straight into LDS (global_load_lds_dwordx4: lane l of
// a wave writes 16 bytes at the wave's LDS base + 16 l), so no registers hold them.
// LDS rows are 64 halves (128 B) without padding; the 16-byte chunk c of row r sits
// in slot c ^ ((r >> 1) & 7).  A ds_read_b128 serves 16 lanes (16 rows, one chunk)
// from the 64 banks at a time: rows of one parity take 8 distinct slots in one half
// of a 256-byte bank line and rows of the other parity the other half, so no two
// lanes of a group share a bank.  Three stages (144 KiB for WR = 4): loads
// run two stages ahead of the MFMAs.  Each K step's fragments are read while the
// previous step's MFMAs run, and its Bi operand is formed between them.  An output's K
// order depends on neither the tile nor the grid, so every tile gives identical results.
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Work-group barrier without the release fence of __syncthreads(), which would wait
// for every outstanding global load (the direct loads of the next stage included).
// Callers wait for the loads that must have landed with s_waitcnt first; the asm
// statements keep the compiler from moving memory accesses across the barrier.
__device__ __forceinline__ void stage_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// fragment of 16-byte chunk pair kk from the swizzled stage (sa, sb): lane holds row (lane % 32),
// chunk 2 kk + lane / 32, found at byte soff = (lane % 32) * ROWB + 16 (chunk ^ ((lane >> 1) & 7))
// (row bases are multiples of 32, so (row >> 1) & 7 = ((lane % 32) >> 1) & 7)
__device__ __forceinline__ void lay_lfrag(const char* sa, const char* sb, int soff, int wr, int wc,
                                          uint4 (&fa)[2], uint4 (&fb)[2]) {
#pragma unroll
    for (int i = 0; i < 2; i++) fa[i] = *(const uint4*)(sa + (wr * 64 + i * 32) * ROWB + soff);
#pragma unroll
    for (int j = 0; j < 2; j++) fb[j] = *(const uint4*)(sb + (wc * 64 + j * 32) * ROWB + soff);
}

__device__ __forceinline__ void lay_bi(const uint4 (&fb)[2], uint4 (&bi)[2]) {
#pragma unroll
    for (int j = 0; j < 2; j++)
        bi[j] = make_uint4(bi_of_br(fb[j].x), bi_of_br(fb[j].y), bi_of_br(fb[j].z), bi_of_br(fb[j].w));
}

template <typename T>
__device__ __forceinline__ void lay_mfma8(const uint4 (&fa)[2], const uint4 (&fb)[2],
                                          const uint4 (&bi)[2], f16v_t (&accr)[2][2],
                                          f16v_t (&acci)[2][2]) {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            accr[i][j] = mfma<T>(fa[i], fb[j], accr[i][j]);
            acci[i][j] = mfma<T>(fa[i], bi[j], acci[i][j]);
        }
}

// The 8 MFMAs of one K step from (fa, fb, bi).  The Bi operand of the next step (whose
// fragments were read at the start of this one) is formed during the second
// half, each MFMA followed by an equal share of its 16 VALU operations, so the VALU
// work issues while the matrix unit is busy instead of in front of the next step.
template <typename T>
__device__ __forceinline__ void lay_step(const uint4 (&fa)[2], const uint4 (&fb)[2],
                                         const uint4 (&bi)[2], const uint4 (&fbn)[2],
                                         uint4 (&bin)[2], f16v_t (&accr)[2][2],
                                         f16v_t (&acci)[2][2]) {
    lay_mfma8<T>(fa, fb, bi, accr, acci);
    lay_bi(fbn, bin);
    // half of the MFMAs alone (the next fragments are still arriving), then
    // (MFMA, VALU ...) pairs carrying the 16 VALU operations
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
    }
}

// One K step's fragments of a SPLIT product: hi and lo of A and Br
struct SFrag {
    uint4 ah[2], al[2], bh[2], bl[2];
};
__device__ __forceinline__ void lay_sfrag(const char* sa, const char* sb, int shi, int slo, int wr,
                                          int wc, SFrag& f) {
    lay_lfrag(sa, sb, shi, wr, wc, f.ah, f.bh);
    lay_lfrag(sa, sb, slo, wr, wc, f.al, f.bl);
}
// The 24 MFMAs of one SPLIT K step: hi hi alone (the next step's fragments arrive), lo hi
// while Bi's lo part is formed, hi lo while the next step's Bi hi part is formed.
template <typename T>
__device__ __forceinline__ void lay_step_split(const SFrag& f, const uint4 (&ih)[2], const SFrag& fn,
                                               uint4 (&ihn)[2], f16v_t (&accr)[2][2],
                                               f16v_t (&acci)[2][2]) {
    uint4 il[2];
    lay_mfma8<T>(f.ah, f.bh, ih, accr, acci);
    lay_mfma8<T>(f.al, f.bh, ih, accr, acci);
    lay_bi(f.bl, il);
    lay_mfma8<T>(f.ah, f.bl, il, accr, acci);
    lay_bi(fn.bh, ihn);
    __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
#pragma unroll
    for (int q = 0; q < 16; q++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
    }
}

// direct loads of one stage (K columns k0 .. k0 + 63) into (da, db): the instruction for
// 8-row group g writes bytes g*1024 .. +1023; lane l fills row r = 8g + l/8, slot l%8
// with global chunk (l%8) ^ ((r >> 1) & 7) = (l%8) ^ (4 (g & 1) + l/16) -- g = wave + 2 WR q
// keeps the parity of the wave index (loff is that lane's byte offset, in 32 bits so that the
// rest of the address stays uniform, in scalar registers)
template <typename T, int WR>
__device__ __forceinline__ void lay_dload(const T* gA, const T* gB, size_t ldk, size_t k0,
                                          uint32_t loff, int wave, char* da, char* db) {
    constexpr int WAVES = 2 * WR;
#pragma unroll
    for (int q = 0; q < 64 * WR / 8 / WAVES; q++) {
        const int g = wave + WAVES * q;
        __builtin_amdgcn_global_load_lds((const void*)((const char*)(gA + (size_t)(8 * g) * ldk + k0) + loff),
                                         (lds_ptr_t)(da + g * 8 * ROWB), 16, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < GTN / 8 / WAVES; q++) {
        const int g = wave + WAVES * q;
        __builtin_amdgcn_global_load_lds((const void*)((const char*)(gB + (size_t)(8 * g) * ldk + k0) + loff),
                                         (lds_ptr_t)(db + g * 8 * ROWB), 16, 0, 0);
    }
}

// s_waitcnt immediates (expcnt and, except in the last, lgkmcnt left open): all of this
// wave's loads landed, or all but the newest stage's (loads complete in issue order);
// the last also waits for all of this wave's LDS reads
constexpr int WAIT_VM0 = 0x0F70;
// direct loads per wave and stage
template <int WR> constexpr int stage_loads() { return (64 * WR + GTN) / 8 / (2 * WR); }
template <int WR> constexpr int wait_vm_stage() { return 0x0F70 | stage_loads<WR>(); }
template <int WR> constexpr int wait_vm_stage_lgkm0() { return 0x0070 | stage_loads<WR>(); }
static_assert(stage_loads<4>() == 6 && stage_loads<2>() == 8, "vmcnt fits 4 bits");

// fragments and Bi operands carried from stage to stage: two K steps' worth, used in turn
template <bool SPLIT>
struct GemmRegs {
    uint4 fa0[2], fb0[2], fa1[2], fb1[2], bi0[2], bi1[2];
};
template <>
struct GemmRegs<true> {
    SFrag f0, f1;
    uint4 ih0[2], ih1[2];
};

// One stage: read (sa, sb), load stage st + 2 into (da, db) -- the buffers of stage
// st - 1, whose reads all completed before that stage's barrier -- and finish with
// stage st + 1 landed in (na, nb) and its first fragments and Bi operand in the first
// set of r.  The barrier sits before the last step's MFMAs.  The six LDS pointers are restrict:
// after inlining, the reads carry alias scopes that tell them apart from the direct
// loads in flight, so the compiler waits for those loads only where they are read.
// Nothing is conditional (branches would merge the compiler's wait bookkeeping into
// full waits): past the end, the last stage is loaded again into a buffer that is not
// read any more, and the fragments read are not used.
template <typename T, int WR, bool SPLIT>
__device__ __forceinline__ void lay_stage(
    const T* gA, const T* gB, size_t ldk, uint32_t loff, int wave, int wr, int wc, const int (&soff)[4],
    int st, int nsteps, const char* __restrict__ sa, const char* __restrict__ sb,
    const char* __restrict__ na, const char* __restrict__ nb, char* __restrict__ da,
    char* __restrict__ db, GemmRegs<SPLIT>& r, f16v_t (&accr)[2][2], f16v_t (&acci)[2][2]) {
    lay_dload<T, WR>(gA, gB, ldk, (size_t)min(st + 2, nsteps - 1) * KS, loff, wave, da, db);
    // sched_barrier(0) fences: each step's fragment reads for the next step are issued
    // before its MFMAs, which cover their latency
    if constexpr (SPLIT) {
        lay_sfrag(sa, sb, soff[1], soff[3], wr, wc, r.f1);
        __builtin_amdgcn_sched_barrier(0);
        lay_step_split<T>(r.f0, r.ih0, r.f1, r.ih1, accr, acci);
        __builtin_amdgcn_sched_barrier(0);
    } else {
        lay_lfrag(sa, sb, soff[1], wr, wc, r.fa1, r.fb1);
        __builtin_amdgcn_sched_barrier(0);
        lay_step<T>(r.fa0, r.fb0, r.bi0, r.fb1, r.bi1, accr, acci);
        __builtin_amdgcn_sched_barrier(0);
        lay_lfrag(sa, sb, soff[2], wr, wc, r.fa0, r.fb0);
        __builtin_amdgcn_sched_barrier(0);
        lay_step<T>(r.fa1, r.fb1, r.bi1, r.fb0, r.bi0, accr, acci);
        __builtin_amdgcn_sched_barrier(0);
        lay_lfrag(sa, sb, soff[3], wr, wc, r.fa1, r.fb1);
        __builtin_amdgcn_sched_barrier(0);
        lay_step<T>(r.fa0, r.fb0, r.bi0, r.fb1, r.bi1, accr, acci);
        __builtin_amdgcn_sched_barrier(0);
    }
    // The last step's operands are in registers: once this wave's reads of the stage
    // are complete and stage st + 1 has landed, the barrier can come before the last
    // step's MFMAs, which then cover the next stage's first reads (after the barrier
    // the other waves may start loading into this stage's buffers).
    __builtin_amdgcn_s_waitcnt(wait_vm_stage_lgkm0<WR>());
    stage_barrier();
    if constexpr (SPLIT) {
        lay_sfrag(na, nb, soff[0], soff[2], wr, wc, r.f0);
        __builtin_amdgcn_sched_barrier(0);
        lay_step_split<T>(r.f1, r.ih1, r.f0, r.ih0, accr, acci);
    } else {
        lay_lfrag(na, nb, soff[0], wr, wc, r.fa0, r.fb0);
        __builtin_amdgcn_sched_barrier(0);
        lay_step<T>(r.fa1, r.fb1, r.bi1, r.fb0, r.bi0, accr, acci);
    }
    __builtin_amdgcn_sched_barrier(0);
}

// U (+)= A (Br, Bi)^T over `stages` stages of the factor rows (ldk halves apart).
// blockIdx.z takes kslice stages of them and writes the plane U + z plane (plane: values).
// An FP32 accumulator holds at most `chain` stages: longer slices add to U chain by chain,
// so that the roundings happen at the magnitude of a part of the sum.  With flip = 1 they are subtracted
// where chain and slice together are odd, for factors that are negated there: the matrix unit rounds its
// sums down, not to the nearest, and what that adds to every term, 4e-10 of it and more, then cancels
// (20,000 points into 200 x 200: 3.3e-7 of the field in the mean, 1e-9 so).  (Chains in launches of
// their own measured 60 us apiece at 2160 x 3840: a tail of idle compute units each.)
// The factor matrices hold whole tiles (rows past ny / nx padded, any content: they
// only reach outputs past the hologram's edge, which are not stored).
template <typename T, int WR, bool SPLIT>
__global__ void __launch_bounds__(128 * WR, 1)
k_cgemm(const T* __restrict__ A, const T* __restrict__ Br, int ldk, int stages, int kslice, int chain,
        float2* __restrict__ U, size_t plane, int ny, int nx, int accumulate, int swz, int flip) {
    constexpr int GTM = 64 * WR;
    __shared__ __align__(16) char sA0[GTM * ROWB], sA1[GTM * ROWB], sA2[GTM * ROWB];
    __shared__ __align__(16) char sB0[GTN * ROWB], sB1[GTN * ROWB], sB2[GTN * ROWB];
    char *a0 = sA0, *a1 = sA1, *a2 = sA2, *b0 = sB0, *b1 = sB1, *b2 = sB2;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave >> 1, wc = wave & 1;
    int bx = blockIdx.x, by = blockIdx.y;
    if (swz > 0) {
        // work-groups are dealt to the 8 XCDs in turn: give each XCD a contiguous run of
        // tiles, taken swz tile rows at a time, so that the tiles running together on one
        // XCD share few A rows and B columns in its L2
        const int gx = gridDim.x, G = gx * gridDim.y;
        const int id = blockIdx.y * gx + blockIdx.x;
        const int t = (id % 8) * (G / 8) + id / 8;
        const int grp = t / (swz * gx), in = t % (swz * gx);
        by = grp * swz + in % swz;
        bx = in / swz;
    }
    const int h0 = by * GTM, w0 = bx * GTN;
    const int st0 = blockIdx.z * kslice, st1 = min(st0 + kslice, stages);
    U += (size_t)blockIdx.z * plane;
    const uint32_t loff = (uint32_t)(lane >> 3) * (uint32_t)ldk * 2u +
                          (uint32_t)(((lane & 7) ^ (4 * (wave & 1) + (lane >> 4))) * 16);
    int soff[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++)
        soff[kk] = (lane & 31) * ROWB + (((2 * kk + (lane >> 5)) ^ ((lane >> 1) & 7)) * 16);
    int odd = flip & blockIdx.z;
    for (int cs = st0; cs < st1; cs += chain, odd ^= flip) {
        const int nsteps = min(chain, st1 - cs);
        const T* gA = A + (size_t)h0 * ldk + (size_t)cs * KS;
        const T* gB = Br + (size_t)w0 * ldk + (size_t)cs * KS;
        GemmRegs<SPLIT> r;
        f16v_t accr[2][2], acci[2][2];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) accr[i][j][v] = acci[i][j][v] = 0.f;

        static_assert(KS == 64, "four 16-wide chunk pairs of 8 16-byte chunks per stage");
        lay_dload<T, WR>(gA, gB, (size_t)ldk, 0, loff, wave, a0, b0);
        lay_dload<T, WR>(gA, gB, (size_t)ldk, (size_t)min(1, nsteps - 1) * KS, loff, wave, a1, b1);
        __builtin_amdgcn_s_waitcnt(wait_vm_stage<WR>());
        stage_barrier();
        if constexpr (SPLIT) {
            lay_sfrag(a0, b0, soff[0], soff[2], wr, wc, r.f0);
            lay_bi(r.f0.bh, r.ih0);
        } else {
            lay_lfrag(a0, b0, soff[0], wr, wc, r.fa0, r.fb0);
            lay_bi(r.fb0, r.bi0);
        }
        int st = 0;
        for (; st + 3 <= nsteps; st += 3) {
            lay_stage<T, WR, SPLIT>(gA, gB, ldk, loff, wave, wr, wc, soff, st, nsteps, a0, b0, a1, b1, a2, b2,
                                    r, accr, acci);
            lay_stage<T, WR, SPLIT>(gA, gB, ldk, loff, wave, wr, wc, soff, st + 1, nsteps, a1, b1, a2, b2, a0,
                                    b0, r, accr, acci);
            lay_stage<T, WR, SPLIT>(gA, gB, ldk, loff, wave, wr, wc, soff, st + 2, nsteps, a2, b2, a0, b0, a1,
                                    b1, r, accr, acci);
        }
        if (st < nsteps)
            lay_stage<T, WR, SPLIT>(gA, gB, ldk, loff, wave, wr, wc, soff, st, nsteps, a0, b0, a1, b1, a2, b2,
                                    r, accr, acci);
        if (st + 1 < nsteps)
            lay_stage<T, WR, SPLIT>(gA, gB, ldk, loff, wave, wr, wc, soff, st + 1, nsteps, a1, b1, a2, b2, a0,
                                    b0, r, accr, acci);
        // no direct load may still be writing LDS when the work-group ends
        __builtin_amdgcn_s_waitcnt(WAIT_VM0);
        // epilogue: lane holds column w = l % 32 and rows 8 (v/4) + 4 (l/32) + v % 4.  Its
        // addresses are formed here: hoisted out of the chain loop they spilled 60 registers.
        int hb = h0, wb = w0, ln = lane;
        const float sg = odd ? -1.f : 1.f;
        asm volatile("" : "+s"(hb), "+s"(wb), "+v"(ln));
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int h = hb + wr * 64 + i * 32 + 8 * (v >> 2) + 4 * (ln >> 5) + (v & 3);
                    const int w = wb + wc * 64 + j * 32 + (ln & 31);
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
        accumulate = 1;
        stage_barrier();  // the next chain's loads reuse the stages other waves have read
    }
}

// Tile height and K slices of a product.  A launch runs ceil(tiles slices / CUs) rounds of
// one work-group per CU; a round of the 128-row tile costs about 0.55 of a 256-row one's
// (half the MFMAs, two thirds of the factor bytes).  Slices shorten the rounds of a
// hologram with few tiles (300 x 400 has 8), at the price of a partial plane each, written
// here and read by the pass that adds them.  Measured: layered split BF16, 2160 x 3840, 270 tiles of
// 256 rows in two rounds 60.0 ms, 510 of 128 rows in two 34.1 ms (with the split product in one
// launch); 20,000 points into 800 x 900 2.00 -> 0.43 ms.
struct GemmPlan {
    int wr, slices, kslice;
};
// merge: cycles of the launch that adds the planes, where one slice needs none
inline GemmPlan gemm_plan(int64_t ny, int64_t nx, int stages, bool split, int max_slices, double merge) {
    const auto up = [](int64_t v, int64_t m) { return (v + m - 1) / m; };
    // cycles of a stage of the 256-row tile (MFMA issue), and of one plane's store and load
    const double stage = split ? 3072.0 : 2048.0;
    const double plane = (double)ny * (double)nx * 16.0 / 5.0e12 * 2.2e9;
    GemmPlan best{4, 1, stages};
    double bc = 1e300;
    for (int wr : {4, 2}) {
        const int64_t tiles = up(ny, 64 * wr) * up(nx, GTN);
        for (int S = 1; S <= max_slices && S <= stages; S++) {
            const int ks = (int)up(stages, S);
            if ((int)up(stages, ks) != S) continue;
            const double rounds = (double)up(tiles * S, GEMM_CUS);
            const double c = rounds * (ks + 4) * stage * (wr == 4 ? 1.0 : 0.55) + (S > 1 ? S * plane + merge : 0.0);
            if (c < bc) {
                bc = c;
                best = GemmPlan{wr, S, ks};
            }
        }
    }
    return best;
}

// launches one product over `stages` stages
template <typename T, bool SPLIT>
inline void cgemm(hipStream_t s, int wr, int slices, const void* A, const void* B, int ldk, int stages,
                  int kslice, int chain, float2* U, size_t plane, int64_t ny, int64_t nx, int acc, int swz, int flip = 0) {
    const unsigned gy = (unsigned)((ny + 64 * wr - 1) / (64 * wr)), gx = (unsigned)((nx + GTN - 1) / GTN);
    const dim3 grid(gx, gy, (unsigned)slices);
    // the swizzle needs a tile count divisible by the 8 XCDs and whole groups of rows
    if (swz > 0 && ((gx * gy) % 8 != 0 || gy % swz != 0)) swz = 0;
    if (wr == 4)
        k_cgemm<T, 4, SPLIT><<<grid, 512, 0, s>>>((const T*)A, (const T*)B, ldk, stages, kslice, chain, U, plane,
                                                  (int)ny, (int)nx, acc, swz, flip);
    else
        k_cgemm<T, 2, SPLIT><<<grid, 256, 0, s>>>((const T*)A, (const T*)B, ldk, stages, kslice, chain, U, plane,
                                                  (int)ny, (int)nx, acc, swz, flip);
}

}  // namespace olx

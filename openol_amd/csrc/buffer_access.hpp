// buffer_access.hpp -- raw buffer loads and stores of the propagation passes.
#pragma once
#include <hip/hip_runtime.h>

namespace olx {

// Global accesses of the propagation passes are raw buffer operations: a per-thread
// 32-bit byte offset in one VGPR, the per-value part (uniform) in an SGPR (but see the
// 16-byte stores).  The descriptor carries the buffer's size, so an access past the end reads zero and a
// store past the end is dropped instead of touching other memory.
struct Rsrc {
    __amdgpu_buffer_rsrc_t r;
};
__device__ __forceinline__ Rsrc make_rsrc(const void* p, size_t bytes) {
    // raw buffer, stride 0, gfx9 data format word
    return Rsrc{__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000)};
}
__device__ __forceinline__ float2 bload(Rsrc b, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(b.r, voff, soff, 0));
}
__device__ __forceinline__ void bstore(Rsrc b, uint32_t voff, uint32_t soff, float2 v) {
    using V = decltype(__builtin_amdgcn_raw_buffer_load_b64(b.r, 0, 0, 0));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V, v), b.r, voff, soff, 0);
}
__device__ __forceinline__ float bloadf(Rsrc b, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b.r, voff, soff, 0));
}
__device__ __forceinline__ void bstoref(Rsrc b, uint32_t voff, uint32_t soff, float v) {
    using V = decltype(__builtin_amdgcn_raw_buffer_load_b32(b.r, 0, 0, 0));
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(V, v), b.r, voff, soff, 0);
}
// two adjacent complex values in one 16-byte access
__device__ __forceinline__ void bload2(Rsrc b, uint32_t voff, uint32_t soff, float2& x, float2& y) {
    const float4 q = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(b.r, voff, soff, 0));
    x = make_float2(q.x, q.y);
    y = make_float2(q.z, q.w);
}
// A store of 16 bytes reads its data registers for some cycles after it is issued, and a vector
// instruction that writes one of them right behind it is seen by the store.  The compiler keeps
// such a write back only where the store has no scalar offset; with one, a value's lowest 32 bits
// were now and then the next store's index (800 x 1701 in complex128: some pixels of every call
// off by 1e-9 to 1e-6).  So either the whole offset stands in the vector register (the complex128
// passes: no time lost), or two wait states that read the data follow the store (the two-column
// passes, which the additions slow by 6 % at 8192 x 8192).
__device__ __forceinline__ void bstore2(Rsrc b, uint32_t voff, uint32_t soff, float2 x, float2 y) {
    using V = decltype(__builtin_amdgcn_raw_buffer_load_b128(b.r, 0, 0, 0));
    const V v = __builtin_bit_cast(V, make_float4(x.x, x.y, y.x, y.y));
    __builtin_amdgcn_raw_buffer_store_b128(v, b.r, voff, soff, 0);
    asm volatile("s_nop 1" ::"v"(v));
}
// one value of either complex type
template <class C>
__device__ __forceinline__ C bloadc(Rsrc b, uint32_t voff, uint32_t soff) {
    if constexpr (sizeof(C) == 8) return __builtin_bit_cast(C, __builtin_amdgcn_raw_buffer_load_b64(b.r, voff, soff, 0));
    else return __builtin_bit_cast(C, __builtin_amdgcn_raw_buffer_load_b128(b.r, voff, soff, 0));
}
template <class C>
__device__ __forceinline__ void bstorec(Rsrc b, uint32_t voff, uint32_t soff, C v) {
    if constexpr (sizeof(C) == 8) {
        using V = decltype(__builtin_amdgcn_raw_buffer_load_b64(b.r, 0, 0, 0));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V, v), b.r, voff, soff, 0);
    } else {
        using V = decltype(__builtin_amdgcn_raw_buffer_load_b128(b.r, 0, 0, 0));
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(V, v), b.r, voff + soff, 0, 0);
    }
}

}  // namespace olx

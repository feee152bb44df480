// Four consecutive cells of a row (a quad) as 16-byte values, for the kernels whose lanes own quads.
#pragma once

#include "fw_internal.h"

namespace fw {

struct alignas(16) F4 {
    float x, y, z, w;
    __device__ float& operator[](int i) { return (&x)[i]; }
    __device__ float operator[](int i) const { return (&x)[i]; }
};
struct alignas(16) I4 {
    int x, y, z, w;
    __device__ int operator[](int i) const { return (&x)[i]; }
};

// Vector access at a 32-bit element index: the array base stays in scalar registers and each
// lane supplies a 32-bit byte offset (grids here have fewer than 2^30 cells per array, checked
// on the host), which saves a 64-bit address per access.
__device__ __forceinline__ const char* at_(const void* base, uint32_t i) { return reinterpret_cast<const char*>(base) + (i << 2); }
__device__ __forceinline__ F4 ld4(const float* base, uint32_t i) { return *reinterpret_cast<const F4*>(at_(base, i)); }
__device__ __forceinline__ I4 ldi4(const int32_t* base, uint32_t i) { return *reinterpret_cast<const I4*>(at_(base, i)); }
__device__ __forceinline__ float ld1(const float* base, uint32_t i) { return *reinterpret_cast<const float*>(at_(base, i)); }
// four 16-bit codes at element index i (i % 4 == 0: 8-byte aligned)
__device__ __forceinline__ uint2 ldc4(const uint16_t* base, uint32_t i) {
    return *reinterpret_cast<const uint2*>(reinterpret_cast<const char*>(base) + (i << 1));
}

__device__ __forceinline__ void st4(float* base, uint32_t i, const F4& v) {
    *reinterpret_cast<F4*>(reinterpret_cast<char*>(base) + (i << 2)) = v;
}
// non-temporal 16-byte access for the memory variables (read and written once per step)
typedef float f4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ F4 ld4nt(const float* base, uint32_t i) {
    const f4v v = __builtin_nontemporal_load(reinterpret_cast<const f4v*>(at_(base, i)));
    return F4{v.x, v.y, v.z, v.w};
}
__device__ __forceinline__ void st4nt(float* base, uint32_t i, const F4& v) {
    const f4v w = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(w, reinterpret_cast<f4v*>(reinterpret_cast<char*>(base) + (i << 2)));
}

// Whether all the quads of this wavefront's active lanes (`cw`: a lane's four codes) have one code
// that is not the escape; `code` is it then.
__device__ __forceinline__ bool wave_code(uint2 cw, uint32_t* code) {
    const uint32_t c0 = __builtin_amdgcn_readfirstlane(cw.x);
    *code = c0 & 0xffffu;
    return (c0 >> 16) == *code && *code != kCodeEscape && __all(cw.x == c0 && cw.y == c0);
}

}  // namespace fw

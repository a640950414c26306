// The matrix-core operations and the SwiGLU shared by the grouped GEMMs (device code).
#pragma once

#include "common.hpp"

namespace nomas {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// A lane's 16-byte operand fragment (one row, 64 bytes of k per stage split
// over the 4 lane groups) feeds kSub MFMAs: one 16x16x32 for 16-bit types,
// four 16x16x4 for f32 (MFMA t takes element t; lane group g then holds
// k = 4 g + t of the stage, the same for both operands).
template <typename T> struct Mfma;
template <> struct Mfma<__bf16> {
    typedef bf16x8_t V;
    static constexpr int kSub = 1;
    static __device__ __forceinline__ f32x4_t run(V a, V b, f32x4_t c, int) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma<_Float16> {
    typedef f16x8_t V;
    static constexpr int kSub = 1;
    static __device__ __forceinline__ f32x4_t run(V a, V b, f32x4_t c, int) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma<float> {
    typedef f32x4_t V;
    static constexpr int kSub = 4;
    static __device__ __forceinline__ f32x4_t run(V a, V b, f32x4_t c, int t) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[t], c, 0, 0, 0);
    }
};

enum { kGateUp = 0, kDown = 1 };  // the two GEMMs of an expert

// silu(g) * u.  For 16-bit outputs the hardware reciprocal (1 ulp) and
// exponential add a few f32 ulps, far below the output's own rounding.
template <typename T>
__device__ __forceinline__ float swiglu(float g, float u) {
    if constexpr (sizeof(T) == 2) return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
    else return g / (1.0f + expf(-g)) * u;
}

}  // namespace nomas

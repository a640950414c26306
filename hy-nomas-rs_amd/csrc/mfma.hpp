// The matrix-core operations and the SwiGLU shared by the grouped GEMMs (device code).
#pragma once

#include "kernels.hpp"

namespace nomas {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// One 16x16x32 MFMA on the lane's 16-byte fragments of 16-bit types (one row,
// 64 bytes of k split over the 4 lane groups).  For f32, V holds 4 values.
template <typename T> struct Mfma;
template <> struct Mfma<__bf16> {
    typedef bf16x8_t V;
    static __device__ __forceinline__ f32x4_t run(V a, V b, f32x4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma<_Float16> {
    typedef f16x8_t V;
    static __device__ __forceinline__ f32x4_t run(V a, V b, f32x4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma<float> {
    typedef f32x4_t V;
};
// v_mfma_f32_16x16x4_f32: element t of the fragments, k = 4 (lane group) + t.
__device__ __forceinline__ f32x4_t mfma_f32(float a, float b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// f32 products on the bf16 matrix cores: each f32 value is the exact sum of
// three bf16 planes (the value rounded to bf16, the remainder rounded, the
// rest: 8 + 8 + 8 significant bits), and a product of two values is the six
// plane products down to 2^-16 of the largest, added smallest first into the
// f32 accumulator.  Left out are the second plane of one value times the third of the
// other, twice: each below 2^-8 x 2^-17 of the values' powers of two, so at most 2^-24
// of the product (half a unit of its last place; on N(0, 1) pairs 2^-27.4 in the
// mean square), and what is left has six roundings per 32 products.  The bf16
// MFMA does a plane product in 1/16 of the time of the f32 MFMAs.  Weights stay
// f32 in memory and are split by the GEMM; activations (x_perm, h) are split
// once, by the kernels that write them (kernels.hpp).
// The matrix cores flush planes below bf16's smallest normal, 2^-126: a value
// below 2^-107 would lose bits (of weights of 2^-115 the product kept 16).  So
// both operands are taken times 2^24, where the last bit of every f32 value
// is a normal bf16: activations when they are split, weights once at upload (but
// not a layer that holds a weight of 2^103 or more).  The sums are scaled back
// by the epilogue, exactly (partial sums overflow from 2^80 on instead of 2^128).
// Sums that come out infinite or NaN are made again with f32 MFMAs by the GEMMs:
// those, and products with a value that has no planes (2^103 and more, infinite,
// NaN: the mark below) or with a weight that rounds past bf16's largest.
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
constexpr int kPlanes = kActPlanes;
constexpr int kProducts = 6;
constexpr float kPlaneMax = 0x1p127f;  // of a value times kPlaneScale
constexpr uint32_t kRawMark = 0x7f80;  // plane 1 (infinite) of a value stored as its raw halves in planes 0 and 2
__host__ __device__ constexpr int product_a(int p) { return p == 0 ? 0 : p == 1 ? 2 : p == 2 ? 1 : p == 3 ? 0 : p == 4 ? 1 : 0; }
__host__ __device__ constexpr int product_b(int p) { return p == 0 ? 2 : p == 1 ? 0 : p == 2 ? 1 : p == 3 ? 1 : p == 4 ? 0 : 0; }

// Two f32 to bf16 (round to nearest even), the first in the low half.
__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// The planes of a lane's 8 values, one pair of values at a time in four steps
// of at most 3 instructions (to be spread between MFMAs).
struct SplitState {
    float r0, r1, s0, s1;
};
template <int STEP>
__device__ __forceinline__ void split_step(float x0, float x1, int d, u32x4_t (&pl)[kPlanes], SplitState& t) {
#pragma clang fp contract(off)
    if constexpr (STEP == 0) {
        const uint32_t p = cvt_pk_bf16(x0, x1);
        pl[0][d] = p;
        t.s0 = __uint_as_float(p << 16);
        t.s1 = __uint_as_float(p & 0xffff0000u);
    } else if constexpr (STEP == 1) {
        t.r0 = x0 - t.s0;
        t.r1 = x1 - t.s1;
        pl[1][d] = cvt_pk_bf16(t.r0, t.r1);
    } else if constexpr (STEP == 2) {
        const uint32_t p = pl[1][d];
        t.s0 = __uint_as_float(p << 16);
        t.s1 = __uint_as_float(p & 0xffff0000u);
        t.r0 -= t.s0;
    } else {
        t.r1 -= t.s1;
        pl[2][d] = cvt_pk_bf16(t.r0, t.r1);
    }
}
__device__ __forceinline__ void split_all(const f32x4_t& a, const f32x4_t& b, u32x4_t (&pl)[kPlanes]) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const float x0 = d < 2 ? a[2 * d] : b[2 * d - 4], x1 = d < 2 ? a[2 * d + 1] : b[2 * d - 3];
        SplitState t;
        split_step<0>(x0, x1, d, pl, t);
        split_step<1>(x0, x1, d, pl, t);
        split_step<2>(x0, x1, d, pl, t);
        split_step<3>(x0, x1, d, pl, t);
    }
}
// The planes of any two values times kPlaneScale, or the values themselves
// where they are too large.
__device__ __forceinline__ void split_exact(float x0, float x1, uint32_t (&pl)[kPlanes]) {
#pragma clang fp contract(off)  // the remainders are of the f32 value, not of the product it may come from
    const float s0 = x0 * kPlaneScale, s1 = x1 * kPlaneScale;
    pl[0] = cvt_pk_bf16(s0, s1);
    const float r0 = s0 - __uint_as_float(pl[0] << 16), r1 = s1 - __uint_as_float(pl[0] & 0xffff0000u);
    pl[1] = cvt_pk_bf16(r0, r1);
    pl[2] = cvt_pk_bf16(r0 - __uint_as_float(pl[1] << 16), r1 - __uint_as_float(pl[1] & 0xffff0000u));
    const bool ok0 = __builtin_fabsf(s0) < kPlaneMax, ok1 = __builtin_fabsf(s1) < kPlaneMax;
    if (!(ok0 && ok1)) {
        const uint32_t b0 = __float_as_uint(x0), b1 = __float_as_uint(x1);
        const uint32_t m = (ok0 ? 0 : 0xffffu) | (ok1 ? 0 : 0xffff0000u);
        pl[0] = (pl[0] & ~m) | ((b0 >> 16 | (b1 & 0xffff0000u)) & m);
        pl[1] = (pl[1] & ~m) | ((kRawMark | kRawMark << 16) & m);
        pl[2] = (pl[2] & ~m) | (((b0 & 0xffffu) | b1 << 16) & m);
    }
}
// ... of 4 or 8 values; plane p's bf16s in order in pl[p]
template <int N>
__device__ __forceinline__ void split_exact_n(const float* v, uint32_t (&pl)[kPlanes][N / 2]) {
#pragma unroll
    for (int d = 0; d < N / 2; ++d) {
        uint32_t q[kPlanes];
        split_exact(v[2 * d], v[2 * d + 1], q);
#pragma unroll
        for (int p = 0; p < kPlanes; ++p) pl[p][d] = q[p];
    }
}
// A value from its planes: the low (0) or high (1) half of each plane's word.
__device__ __forceinline__ float unsplit1(uint32_t p0, uint32_t p1, uint32_t p2, int half) {
    auto bits = [&](uint32_t p) { return half ? p & 0xffff0000u : p << 16; };
    auto v = [&](uint32_t p) { return __uint_as_float(bits(p)); };
    if (bits(p1) == kRawMark << 16) return __uint_as_float(bits(p0) | bits(p2) >> 16);
    return (v(p0) + (v(p1) + v(p2))) * (1.0f / kPlaneScale);
}
// Value s (0-7) of a lane's fragment.
__device__ __forceinline__ float unsplit(const u32x4_t (&pl)[kPlanes], int s) {
    return unsplit1(pl[0][s / 2], pl[1][s / 2], pl[2][s / 2], s % 2);
}
__device__ __forceinline__ f32x4_t mfma_plane(const u32x4_t& a, const u32x4_t& b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
// NaN if any of the values so far was infinite or NaN, else 0.
__device__ __forceinline__ float not_finite(const f32x4_t& v, float t) {
#pragma unroll
    for (int s = 0; s < 4; ++s) t = __builtin_fmaf(v[s], 0.0f, t);
    return t;
}
// Which values are taken from the f32 MFMAs: in the down GEMM each sum that is
// not finite, in gate/up both sums of a hidden unit where one is not (h alone
// does not say which).  Both GEMM kernels keep all other values as they are, so
// that a row's bits do not depend on the kernel.
__device__ __forceinline__ void keep_finite(f32x4_t& v, const f32x4_t& again) {
#pragma unroll
    for (int s = 0; s < 4; ++s) v[s] = __builtin_isfinite(v[s]) ? v[s] : again[s];
}
__device__ __forceinline__ bool unit_finite(float g, float u) {
    return __builtin_isfinite(g) && __builtin_isfinite(u);
}

enum { kGateUp = 0, kDown = 1 };  // the two GEMMs of an expert

// silu(g) * u.  For 16-bit outputs the hardware reciprocal (1 ulp) and
// exponential add a few f32 ulps, far below the output's own rounding.
template <typename T>
__device__ __forceinline__ float swiglu(float g, float u) {
    if constexpr (sizeof(T) == 2) return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
    else return g / (1.0f + expf(-g)) * u;
}

// Where hidden units hc..hc+3 (hc % 4 == 0) of row r are in the first plane of an f32 h.
__device__ __forceinline__ unsigned char* hidden_at(void* h, int64_t a_cap, int r, int hc) {
    return static_cast<unsigned char*>(h) + ((int64_t)(hc / 32 * kPlanes) * a_cap + r) * kKBlockBytes +
           hc / 4 % 4 * 16 + hc / 16 % 2 * 8;
}
// ... and their values.
__device__ __forceinline__ void load_hidden(void* h, int64_t a_cap, int r, int hc, float (&v)[4]) {
    const unsigned char* src = hidden_at(h, a_cap, r, hc);
    uint2 p[kPlanes];
#pragma unroll
    for (int t = 0; t < kPlanes; ++t) p[t] = *reinterpret_cast<const uint2*>(src + t * a_cap * kKBlockBytes);
#pragma unroll
    for (int s = 0; s < 4; ++s)
        v[s] = s < 2 ? unsplit1(p[0].x, p[1].x, p[2].x, s % 2) : unsplit1(p[0].y, p[1].y, p[2].y, s % 2);
}
// Hidden units hc..hc+3 (hc % 4 == 0) of row r into h, K-blocked (f32: planes).
template <typename T>
__device__ __forceinline__ void store_hidden(void* h, int64_t a_cap, int r, int hc, const float (&v)[4]) {
    unsigned char* dst;
    if constexpr (sizeof(T) == 4) {
        uint32_t pl[kPlanes][2];
        split_exact_n<4>(v, pl);
        dst = hidden_at(h, a_cap, r, hc);
#pragma unroll
        for (int p = 0; p < kPlanes; ++p)
            *reinterpret_cast<uint2*>(dst + p * a_cap * kKBlockBytes) = make_uint2(pl[p][0], pl[p][1]);
    } else {
        constexpr int KB = kblock_elems<T>();
        T t[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            // rounded to f32 and then to T, as gemm_mfma does (the compiler made one
            // operation with a single rounding of the last product and the f16)
            float f = v[s];
            asm("" : "+v"(f));
            t[s] = Elt<T>::from_f32(f);
        }
        uint2 raw;
        __builtin_memcpy(&raw, t, sizeof(raw));
        dst = static_cast<unsigned char*>(h) + ((int64_t)(hc / KB) * a_cap + r) * kKBlockBytes + hc % KB * 2;
        *reinterpret_cast<uint2*>(dst) = raw;
    }
}

}  // namespace nomas

// MFMA wrappers for the 16-bit element types of gfx950 and the vector types they take.
//
// Operand layouts of a wavefront (lane = 16 * g + r, r < 16, g < 4):
//   k32: D[16x16] += A[16x32] * B[32x16]; lane holds row r of A / column r of B, elements
//        k = 8g .. 8g+7 (16 bytes); D: lane holds column r, rows 4g .. 4g+3.
//   k16: the same with 16-deep operands, elements k = 4g .. 4g+3 (8 bytes).
#pragma once

#include "hsa_common.h"

namespace hsa {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));

template <typename T> struct Mma;

template <> struct Mma<BF16> {
    static constexpr uint16_t kOne = 0x3f80, kInf = 0x7f80;
    static __device__ __forceinline__ f32x4 k32(u32x4_t a, u32x4_t b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 k16(u32x2_t a, u32x2_t b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4_t, a),
                                                         __builtin_bit_cast(s16x4_t, b), c, 0, 0, 0);
    }
    // round-to-nearest-even pair
    static __device__ __forceinline__ uint32_t pack(float a, float b) {
        f32x2 v = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
    }
    // the inputs are exactly representable: keep the high halves
    static __device__ __forceinline__ uint32_t pack_exact(float a, float b) {
        return (__float_as_uint(a) >> 16) | (__float_as_uint(b) & 0xffff0000u);
    }
};

template <> struct Mma<F16> {
    static constexpr uint16_t kOne = 0x3c00, kInf = 0x7c00;
    static __device__ __forceinline__ f32x4 k32(u32x4_t a, u32x4_t b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                      __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 k16(u32x2_t a, u32x2_t b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4_t, a),
                                                     __builtin_bit_cast(f16x4_t, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack(float a, float b) {
        f32x2 v = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
    }
    static __device__ __forceinline__ uint32_t pack_exact(float a, float b) { return pack(a, b); }
};

// The largest magnitude (as bits) among 16-bit values: infinities and NaN are those from Mma<T>::kInf on.
struct LargestBits {
    u16x2_t m = {0, 0};
    __device__ __forceinline__ void add(u32x4_t v) {
#pragma unroll
        for (int w = 0; w < 4; ++w) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2_t, v[w] & 0x7fff7fffu));
    }
    template <typename T> __device__ __forceinline__ bool finite() const { return m[0] < Mma<T>::kInf && m[1] < Mma<T>::kInf; }
};

// k16 with the B operand in fp32 (b[i]: row 4g + i of column r): products and sums in fp32, on four
// v_mfma_f32_16x16x4_f32 whose steps take the same element of every lane's four (any order of the
// contraction will do).  Eight times the matrix-core cycles of k16.
template <typename T>
__device__ __forceinline__ f32x4 k16_f32(u32x2_t a, const float (&b)[4], f32x4 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(to_float<T>((uint16_t)(a[i >> 1] >> (16 * (i & 1)))), b[i], c, 0, 0, 0);
    return c;
}

// weights as the B operand of k16, rounded to the element type
template <typename T> struct RoundedWeights {
    u32x2_t h;
    __device__ __forceinline__ void set(const float (&b)[4]) { h = u32x2_t{Mma<T>::pack(b[0], b[1]), Mma<T>::pack(b[2], b[3])}; }
    __device__ __forceinline__ f32x4 product(u32x2_t a, f32x4 c) const { return Mma<T>::k16(a, h, c); }
};

// in fp32
template <typename T> struct Fp32Weights {
    float f[4];
    __device__ __forceinline__ void set(const float (&b)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = b[i];
    }
    __device__ __forceinline__ f32x4 product(u32x2_t a, f32x4 c) const { return k16_f32<T>(a, f, c); }
};

// The same bits on the 16-bit matrix instructions: b as a sum of 16-bit numbers, each the rounded rest of the ones
// before it (the rests are exact in fp32).  bf16: three numbers, all 24 bits of b.  fp16: two, an error of at
// most 2^-23 |b| for 2^-2 <= |b| <= 2^15, of at most 2^-25 below.  The first two go into one 32-deep
// product against the A operand taken twice; the third takes a 32-deep product as well, because a k16
// result as the very next k32's accumulator gave wrong sums here: one shape per chain of products.
template <typename T> struct SplitWeights;
template <> struct SplitWeights<BF16> {
    u32x4_t hm, lo;
    __device__ __forceinline__ void set(const float (&b)[4]) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint32_t h = Mma<BF16>::pack(b[2 * p], b[2 * p + 1]);
            const float r0 = b[2 * p] - __uint_as_float(h << 16), r1 = b[2 * p + 1] - __uint_as_float(h & 0xffff0000u);
            const uint32_t m = Mma<BF16>::pack(r0, r1);
            hm[p] = h;
            hm[2 + p] = m;
            lo[2 + p] = 0;
            lo[p] = Mma<BF16>::pack(r0 - __uint_as_float(m << 16), r1 - __uint_as_float(m & 0xffff0000u));
        }
    }
    __device__ __forceinline__ f32x4 product(u32x2_t a, f32x4 c) const {
        const u32x4_t twice = {a[0], a[1], a[0], a[1]};
        return Mma<BF16>::k32(twice, hm, Mma<BF16>::k32(twice, lo, c));
    }
};
template <> struct SplitWeights<F16> {
    u32x4_t hm;
    __device__ __forceinline__ void set(const float (&b)[4]) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint32_t h = Mma<F16>::pack(b[2 * p], b[2 * p + 1]);
            const f16x2_t f = __builtin_bit_cast(f16x2_t, h);
            hm[p] = h;
            hm[2 + p] = Mma<F16>::pack(b[2 * p] - (float)f[0], b[2 * p + 1] - (float)f[1]);
        }
    }
    __device__ __forceinline__ f32x4 product(u32x2_t a, f32x4 c) const {
        return Mma<F16>::k32(u32x4_t{a[0], a[1], a[0], a[1]}, hm, c);
    }
};

}  // namespace hsa

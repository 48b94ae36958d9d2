// fp32 products on gfx950's bf16 matrix cores: an fp32 operand is split into
// three bf16 planes, x = h + m + l (h = bf16(x), m = bf16(x - h), l = the rest,
// exact: 3 x 8 significant bits), and a product x y is the six plane products
// h h + (h m + m h) + (m m + h l + l h), each exact, summed in the MFMA's fp32
// accumulators. The dropped m l, l m, l l reach 2^-24 of the product at the
// worst (x = y = 1 + 2^-8 - 2^-17), one rounding of fp32, and 2^-27.5 in the root
// mean square. gfx950 runs 16 bf16 MFMAs in the time of one fp32 MFMA of the
// same size, so six of them take 2.7 times less matrix time; an operand that is
// bf16 to begin with is its own h plane, and its products with a split one take
// three. Below 2^-110 the planes end at bf16's smallest step and miss up to
// 2^-134 of x. A non-finite operand gives non-finite results, but an infinity
// may come out as NaN (inf - inf in the split), and so may a magnitude above
// 3.389e38, which bf16 rounds to infinity.
#pragma once

#include "tt_common.h"

namespace {

// The three bf16 planes of eight fp32 values.
struct Planes {
    bf16x8 h, m, l;
};

// Two fp32 values rounded to bf16 (low half: a), and r - that value.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}
__device__ __forceinline__ void sub_bf16(uint32_t p, float& a, float& b) {
    a -= __uint_as_float(p << 16);
    b -= __uint_as_float(p & 0xffff0000u);
}

// Splitting eight fp32 values, in eight slices of five or six instructions.
struct Split8 {
    static constexpr int SLICES = 8;
    float r[8];
    uint32_t h[4], m[4], l[4];
    template <int I>
    __device__ __forceinline__ void slice() {
        constexpr int j = I & 3;
        if constexpr (I < 4) {
            h[j] = pack_bf16(r[2 * j], r[2 * j + 1]);
            sub_bf16(h[j], r[2 * j], r[2 * j + 1]);
        } else if constexpr (I < SLICES) {
            m[j] = pack_bf16(r[2 * j], r[2 * j + 1]);
            sub_bf16(m[j], r[2 * j], r[2 * j + 1]);
            l[j] = pack_bf16(r[2 * j], r[2 * j + 1]);
        }
    }
    __device__ __forceinline__ void all() {
        static_for<SLICES>([&](auto i) { slice<decltype(i)::value>(); });
    }
    static __device__ __forceinline__ bf16x8 vec(const uint32_t (&x)[4]) {
        return __builtin_bit_cast(bf16x8, (u32x4){x[0], x[1], x[2], x[3]});
    }
    __device__ __forceinline__ Planes planes() const { return {vec(h), vec(m), vec(l)}; }
};
__device__ __forceinline__ Split8 split_begin(const f32x4& a, const f32x4& b) {
    return {{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}, {}, {}, {}};
}
// Accumulator rows r0 .. r0 + 7 (the next product's operand).
__device__ __forceinline__ Split8 split_begin(const f32x16& s, int r0) {
    return {{s[r0], s[r0 + 1], s[r0 + 2], s[r0 + 3], s[r0 + 4], s[r0 + 5], s[r0 + 6], s[r0 + 7]}, {}, {}, {}};
}

}  // namespace

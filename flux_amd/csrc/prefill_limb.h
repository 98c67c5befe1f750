// Float32 products on the bf16 matrix cores.
//
// A float32 value is the exact sum of three bf16 limbs (8 + 8 + 8 significant bits, each
// rounded to nearest from what the limbs before it leave), so a product of two values is nine
// limb products.  The six largest are kept: the dropped three are at most 2^-23 of the product
// (a second times a third limb, twice), and 5.7e-9 of a sum of random ones.  Each limb product is
// exact in float32 and v_mfma_f32_32x32x16_bf16 sums sixteen of them per instruction, against
// two per v_mfma_f32_32x32x2_f32, so the accumulator is rounded less often and, with the small
// products in an accumulator of their own, the result is closer to the exact sum (normal data,
// K = 576: 1.4e-7 against 4.3e-7 relative; 1536: 2.3e-7 against 7.0e-7; 4096: 4.0e-7 against
// 1.15e-6).  Six of these instructions take 192 cycles for sixteen K values, eight of the
// float32 ones 512.
//
// That holds from 2^-110 to the largest bf16.  Limbs cannot carry infinities (inf - inf) nor
// magnitudes above (kLimbMax), bf16 has no bits below 2^-133 for the low limbs of smaller values
// (kLimbMin), and overflowing limb products need not agree in sign: kernels find out whether any
// of these shows in what they computed, and then compute it with the float32 instruction.
#pragma once

#include "prefill_common.h"

namespace flux {
namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
// float4 loads from rows that are only 4-byte aligned (one instruction all the same).
typedef f32x4 f32x4_u __attribute__((aligned(4)));

constexpr int kLimbs = 3;
constexpr float kLimbMax = 3.3895313892515355e38f;  // largest finite bf16 (0x7f7f)
constexpr float kLimbMin = 0x1p-110f;               // and the least magnitude whose limbs add up to it

// The limbs of eight values, as MFMA operands.
struct Limbs8 {
    u32x4 limb[kLimbs];
};

__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// Splits a pair into its three packed limbs.
__device__ __forceinline__ void split_pair(float a, float b, unsigned& l0, unsigned& l1, unsigned& l2) {
    l0 = pack_bf16(a, b);
    a -= __uint_as_float(l0 << 16);
    b -= __uint_as_float(l0 & 0xffff0000u);
    l1 = pack_bf16(a, b);
    a -= __uint_as_float(l1 << 16);
    b -= __uint_as_float(l1 & 0xffff0000u);
    l2 = pack_bf16(a, b);
}

__device__ __forceinline__ Limbs8 split8(const f32x4& lo, const f32x4& hi) {
    Limbs8 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = i < 2 ? lo[2 * i] : hi[2 * i - 4];
        const float b = i < 2 ? lo[2 * i + 1] : hi[2 * i - 3];
        unsigned l0, l1, l2;
        split_pair(a, b, l0, l1, l2);
        r.limb[0][i] = l0;
        r.limb[1][i] = l1;
        r.limb[2][i] = l2;
    }
    return r;
}

// running = max(running, |a|, |b|); NaN inputs are ignored.
__device__ __forceinline__ void track_max(float& running, float a, float b) {
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(running) : "v"(a), "v"(b));
}

// Orders magnitudes as integers (an addition and a minimum, against two comparisons), zero last.
__device__ __forceinline__ unsigned magnitude_key(float v) { return 2 * __float_as_uint(v) - 1; }

// Whether the limbs of a value may not add up to it (they are then within 2^-134 of it).
__device__ __forceinline__ bool limbs_drop(float v) { return v != 0.0f && fabsf(v) < kLimbMin; }

__device__ __forceinline__ f32x16 mfma_bf16(const u32x4& a, const u32x4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

constexpr int kLimbProducts = 6;

}  // namespace
}  // namespace flux

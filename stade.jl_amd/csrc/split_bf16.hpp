// fp32 products on the bf16 matrix cores, without loss: an fp32 value is written as h + m + l,
// three bf16 values that hold its 24 bits exactly (h = bf16(a), m = bf16(a - h), l = a - h - m;
// both subtractions are exact), and a product of two such values is the sum of six bf16
// products accumulated in fp32, small ones first: l h + h l + m m + m h + h m + h h.  A bf16
// product is exact in fp32, and the three products left out (m l, l m, l l) are together at
// most 2^-24 of h h: less than the rounding of one fp32 accumulation.
//
// What the split cannot hold: an element with 0 < |a| < 2^-110, whose l part falls below bf16's
// smallest subnormal (`tiny` below notices it, from 2^-109 on), and an element that is not
// finite or whose nearest bf16 is infinite (it leaves a NaN in every sum it takes part in, as
// h - h does).  The kernels notice both per block and then form the block's output with fp32
// matrix instructions.
#pragma once

#include <hip/hip_runtime.h>

namespace stade {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    uint32_t r;  // (one instruction; from two scalar conversions the compiler makes three)
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float bf16_lo(uint32_t v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t v) { return __builtin_bit_cast(float, v & 0xffff0000u); }

// the smallest 2 |h| - 1 (as bits, so zero counts as the largest) of the elements seen: below
// kTinyBits an element is nonzero and under 2^-109, where its l part may not be exact
constexpr unsigned short kTinyBits = ((127 - 109) << 8) - 1;

__device__ __forceinline__ u16x2 twice_less_one(uint32_t h) {
    u16x2 r;
    asm("v_pk_mad_u16 %0, %1, 2, -1 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h));
    return r;
}

__device__ __forceinline__ void split8(const float (&v)[8], u32x4 (&c)[3], u16x2& tiny) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t h = pack_bf16(v[2 * q], v[2 * q + 1]);
        const float r0 = v[2 * q] - bf16_lo(h), r1 = v[2 * q + 1] - bf16_hi(h);
        const uint32_t m = pack_bf16(r0, r1);
        c[0][q] = h;
        c[1][q] = m;
        c[2][q] = pack_bf16(r0 - bf16_lo(m), r1 - bf16_hi(m));
        tiny = __builtin_elementwise_min(tiny, twice_less_one(h));
    }
}

// whether an element seen is too small for the split
__device__ __forceinline__ bool any_tiny(u16x2 tiny) { return tiny.x < kTinyBits || tiny.y < kTinyBits; }

// the six products' parts (of the first and the second operand), in the order they are added
constexpr int kSplitA[6] = {2, 0, 1, 1, 0, 0}, kSplitB[6] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ floatx16 mfma_bf16(bf16x8 a, bf16x8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

}  // namespace stade

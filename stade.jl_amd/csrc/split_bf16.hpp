// fp32 products on the bf16 matrix cores, without loss: an fp32 value is written as h + m + l,
// three bf16 values that hold its 24 bits exactly (h = bf16(a), m = bf16(a - h), l = a - h - m;
// both subtractions are exact), and a product of two such values is the sum of six bf16
// products accumulated in fp32, small ones first: l h + h l + m m + m h + h m + h h.  A bf16
// product is exact in fp32, and the three products left out (m l, l m, l l) are together at
// most 2^-24 of h h: less than the rounding of one fp32 accumulation.
//
// What the split cannot hold: a nonzero element whose last bits lie below bf16's smallest
// subnormal, 2^-133 (from |a| < 2^-110 on, where h and m leave a rest that is no bf16 value; from
// |a| < 2^-134 on nothing of it is left in the parts), and an element that is not finite or
// whose nearest bf16 is infinite (it leaves a NaN in every sum it takes part in, as h - h does).
// The rest a - h - m is exact in fp32, and it is a bf16 value if and only if the low half of
// its bits is zero, subnormals included (bf16 has fp32's exponents): `lost` gathers those
// halves, one instruction a pair.  (A test of the size of h instead takes two, sends exact
// small values such as 2^-120 away as well, and sees a zero in an element below 2^-134.)  The
// kernels look at both per block and then form the block's output with fp32 matrix instructions.
#pragma once

#include <hip/hip_runtime.h>

namespace stade {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    uint32_t r;  // (one instruction; from two scalar conversions the compiler makes three)
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float bf16_lo(uint32_t v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t v) { return __builtin_bit_cast(float, v & 0xffff0000u); }

__device__ __forceinline__ void split8(const float (&v)[8], u32x4 (&c)[3], uint32_t& lost) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t h = pack_bf16(v[2 * q], v[2 * q + 1]);
        const float r0 = v[2 * q] - bf16_lo(h), r1 = v[2 * q + 1] - bf16_hi(h);
        const uint32_t m = pack_bf16(r0, r1);
        c[0][q] = h;
        c[1][q] = m;
        const float t0 = r0 - bf16_lo(m), t1 = r1 - bf16_hi(m);
        c[2][q] = pack_bf16(t0, t1);
        lost |= __builtin_bit_cast(uint32_t, t0) | __builtin_bit_cast(uint32_t, t1);
    }
}

// whether an element seen has bits that its parts do not hold
__device__ __forceinline__ bool any_lost(uint32_t lost) { return (lost & 0xffffu) != 0; }

// the six products' parts (of the first and the second operand), in the order they are added
constexpr int kSplitA[6] = {2, 0, 1, 1, 0, 0}, kSplitB[6] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ floatx16 mfma_bf16(bf16x8 a, bf16x8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

}  // namespace stade

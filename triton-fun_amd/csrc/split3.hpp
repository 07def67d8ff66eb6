// float32 products on the 16-bit matrix instructions.
//
// The published splitting of Henry, Tang and Heinecke ("Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", 2019): a float32 value is the sum of three bfloat16 values, its rounding and the roundings of the two remainders (8 + 8 + 8 bits of
// significand; bfloat16 has float32's exponents, so nothing has to be scaled).  Of the nine products of two such sums the six
// largest are taken, the smallest first; the three left out are below 2^-24 of the product.  The 16-bit instructions run at
// sixteen times the float32 ones' rate, so six of them cost three eighths of one float32 product, and they add sixteen products
// with one rounding where the float32 ones round after each: against float64, 32 x 32 results over 64 / 128 / 512 N(0, 1) products
// are off by 1.1e-7 / 1.6e-7 / 3.4e-7 of their norm (float32 instructions: 1.4e-7 / 2.1e-7 / 4.1e-7).
// What the parts cannot hold:
//   * an infinity, a NaN or a value above bfloat16's largest (3.39e38) turns its remainders into NaN, and with them every result it
//     enters, which is then taken again in float32 arithmetic;
//   * bfloat16 ends at 2^-133 (the matrix instructions take and give subnormal values as they are), so a value below 2^-110 loses what
//     it has below that.  The backward multiplies what it splits in the loop by kSplitLift, which puts the last bit of any float32 value
//     there; results that overflow for it are taken again in float32 arithmetic.  The forward, whose probabilities are at most 2^8, takes a row again
//     where an output is below 2^-104: a small column of V, or one that only keys of small probability have.  A row's own operand (Q; K and
//     V in dK + dV) is not lifted, and the row is taken again where all that a lane has of it is small (out_of_split's lower line) or some
//     of it so large (its upper line) that the other factor's lost bits show.  What is left: single values below 2^-110 among larger
//     ones of a row, where the other factor is above 2^80, and, in the forward, a column of V with nothing above 2^-134, which comes out as zero.
#pragma once
#include "tile_copy.hpp"

namespace splat {

struct Split3 {
    Frag<bf16> p[3];
};

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));

// One step of a pair's split: its next part, and what is left of it.  (Shifts and subtractions: the two-term dot product that
// would take a remainder in one instruction runs on the matrix pipe and holds up the products there.)
__device__ __forceinline__ bf16x2 split_step(float& r0, float& r1, bool last) {
    const f32x2 r = {r0, r1};
    const bf16x2 h = __builtin_convertvector(r, bf16x2);
    if (!last) {
        const uint32_t u = __builtin_bit_cast(uint32_t, h);
        r0 -= __builtin_bit_cast(float, u << 16);
        r1 -= __builtin_bit_cast(float, u & 0xffff0000u);
    }
    return h;
}
__device__ __forceinline__ void put_pair(Frag<bf16>& f, int i, bf16x2 h) { f.v[2 * i] = h[0], f.v[2 * i + 1] = h[1]; }

__device__ __forceinline__ Split3 split3(const f32x8& x) {
    Split3 s;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float r0 = x[2 * i], r1 = x[2 * i + 1];
#pragma unroll
        for (int k = 0; k < 3; ++k) put_pair(s.p[k], i, split_step(r0, r1, k == 2));
    }
    return s;
}

constexpr float kSplitLift = 0x1p16f;

// Whether the largest magnitude of some values is outside what products of split operands keep float32's precision for.
__device__ __forceinline__ bool out_of_split(float most) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(most));  // found here, not where the answer is wanted: the values need not be kept until then
#endif
    return (most > 0.f && most < 0x1p-96f) || most > 0x1p80f;
}

// The six products of a split operand pair, in the order they are added: A's parts one after the other, the smallest first, so that
// the registers of a part that is done with can take the next fragment's.
constexpr int kSplitA[6] = {2, 1, 1, 0, 0, 0}, kSplitB[6] = {0, 1, 0, 2, 1, 0};
constexpr int kSplitLast[3] = {5, 2, 0};  // the last product that part k of A takes part in

}  // namespace splat

// Pieces of the fused float32 backward kernels: 16x16 tiles of scores on the float32 matrix instruction.
//
// Operand layouts of acc[16x16] += A[16x4] * B[4x16] (v_mfma_f32_16x16x4_f32): lane (n = lane % 16, g = lane / 16) feeds row n
// of A and column n of B at contraction slot g, and holds rows 4g .. 4g + 3 of column n of the result.  Which index of the
// contraction a slot stands for is free as long as A and B agree:
//   * products over d take d = 16t + 4g + j in instruction 4t + j, so that one 16-byte read of a row feeds four instructions;
//   * products over positions take position 4g + j in instruction j: register j of a score tile is then the B operand as it
//     stands, without any exchange between lanes;
//   * of the output of those, row m of tile dt stands for d = 4m + dt (+ 64h), so that one 16-byte read of a row of the other
//     operand feeds four tiles, and a lane's 16 results of one row are 16 consecutive columns.
#pragma once
#include "rows16.hpp"

namespace splat {

constexpr int f32_tile(int d) { return d == 64 ? 32 : 16; }  // positions per tile: 8 KB an operand

__device__ __forceinline__ void mma4(f32x4& acc, float a, float b) { acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0); }

__device__ __forceinline__ f32x4 lds_load_f32x4(uint32_t addr) { return __builtin_bit_cast(f32x4, lds_load128(addr)); }

}  // namespace splat

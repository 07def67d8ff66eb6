// K / V tile geometry, LDS swizzles and the asynchronous global -> LDS tile copy shared by the tiled kernels.
#pragma once
#include "acsr_plan.hpp"

namespace splat {

template <typename T, int D, bool KT, int BN = kBN>
struct TileGeom {
    static constexpr int ES = sizeof(T);
    static constexpr int EPC = 16 / ES;                       // elements per 16-byte chunk
    static constexpr int K_ROWB = KT ? BN * ES : D * ES;      // bytes per LDS row of the K tile (no padding)
    static constexpr int K_ROWS = KT ? D : BN;
    static constexpr int V_ROWB = D * ES;
    static constexpr int K_BYTES = K_ROWB * K_ROWS;
    static constexpr int V_BYTES = V_ROWB * BN;
    static constexpr int STAGE = K_BYTES + V_BYTES;
};

// XOR swizzle of the 16-byte chunk index of a row-major LDS tile with ROWB-byte rows, chosen so that 16
// lanes reading the same logical chunk of 16 consecutive rows hit 16 different bank groups.
template <int ROWB>
__device__ __forceinline__ constexpr int swz(int row) {
    constexpr int CPR = ROWB / 16;
    constexpr int CH = CPR < 16 ? CPR : 16;
    constexpr int RPB = ROWB >= 256 ? 1 : 256 / ROWB;
    return (row / RPB) & (CH - 1);
}
template <int ROWB, bool SWZ>
__device__ __forceinline__ int lds_off(int row, int byte_col) {
    if constexpr (SWZ)
        return row * ROWB + ((((byte_col >> 4) ^ swz<ROWB>(row)) << 4) | (byte_col & 15));
    else
        return row * ROWB + byte_col;
}

// Swizzle of the 64-byte block index for tiles read with the transposing read, whose 64 lanes touch 8
// consecutive rows x 64 bytes: 4 consecutive rows must fall into the 4 different 64-byte quadrants of the
// 256-byte bank space (what a row pitch of 256+64 bytes would give, which the 1 KiB LDS-DMA blocks rule out).
template <int ROWB>
__device__ __forceinline__ constexpr int swz64(int row) {
    return ROWB >= 256 ? (row & 3) : ((row >> 1) & 1);
}
// The same for transposing reads 16 columns (32 bytes) wide, whose 64 lanes touch 16 rows: four groups of 4 consecutive rows, 4
// apart (rows = positions) or 8 apart (rows = d); the 32-byte blocks of any 8 of them that come together fill the 256-byte
// bank space.
template <int ROWB>
__device__ __forceinline__ constexpr int swz32(int row) {
    static_assert(ROWB == 64 || ROWB == 128 || ROWB == 256, "row pitch");
    return ROWB == 256 ? (row & 7) : ROWB == 128 ? (((row >> 1) & 1) | (((row >> 3) & 1) << 1)) : ((row >> 3) & 1);
}
// Swizzle for tiles that are read both ways: the 64-byte block index is rotated as for the transposing read, and the
// chunk inside the block by the next two row bits, so that the 16 rows a row-wise 16-byte read touches at once land on
// 16 different chunk positions of the 256-byte bank space (rows 16 apart share their pattern; rows 8 apart differ in
// the second bit of the chunk position).  The map is its own inverse.
template <int ROWB>
__device__ __forceinline__ constexpr int dual_chunk(int row, int c) {
    return (((c >> 2) ^ swz64<ROWB>(row)) << 2) | ((c & 3) ^ ((row >> 2) & 3));
}
// Swizzle of the 16-byte chunk index for tiles that are read row-wise, 16 rows at the same chunk, and by the narrow transposing
// reads: the 16 rows of either half get 16 different chunk positions of the 256-byte bank space, and any 8 consecutive of them
// different 32-byte blocks.
template <int ROWB>
__device__ __forceinline__ constexpr int swz_both16(int row) {
    static_assert(ROWB == 128 || ROWB == 256, "row pitch");
    return ROWB == 256 ? ((row & 7) << 1) | ((row >> 3) & 1) : ((row >> 1) & 3) << 1 | ((row >> 3) & 1);
}
// logical 16-byte chunk held at physical chunk position pc of `row`; MODE 0: none, 1: chunk XOR (b128 row reads),
// 2: 64-byte block XOR (transposing reads), 3: both kinds of read (dual_chunk), 4: 32-byte block XOR (narrow transposing reads)
template <int ROWB, int MODE>
__device__ __forceinline__ int logical_chunk(int row, int pc) {
    if constexpr (MODE == 1) return pc ^ swz<ROWB>(row);
    if constexpr (MODE == 2) return (((pc >> 2) ^ swz64<ROWB>(row)) << 2) | (pc & 3);
    if constexpr (MODE == 3) return dual_chunk<ROWB>(row, pc);
    if constexpr (MODE == 4) return (((pc >> 1) ^ swz32<ROWB>(row)) << 1) | (pc & 1);
    return pc;
}

typedef __attribute__((address_space(1))) const void gptr_t;
typedef __attribute__((address_space(3))) void lptr_t;

// One wavefront-wide 1 KiB copy global -> LDS without passing through registers: lane i's 16 bytes land at
// lds_block + 16*i (lds_block must be wavefront-uniform).
//
// The copies are written as inline asm on purpose.  The compiler orders every LDS read behind every copy instruction it
// knows of (it cannot tell which LDS bytes a copy writes) and, while one is outstanding, turns all its counted waits
// into waits for everything; that would stall each tile on the copies of the next one.  Copies it does not see are
// ordered by the kernels themselves: wait_loads<N>() for this wavefront's copies, then a barrier, before any wavefront
// reads the stage.  The waits the compiler emits for loads it does know stay safe: loads complete in order, so extra
// copies in flight only make such a wait cover more than it needs to.
__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}
// per-lane 64-bit source address
__device__ __forceinline__ void dma16(const void* src, char* lds_block) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(lds_address(lds_block)), "v"(src)
                 : "memory", "m0");
}
// wavefront-uniform 64-bit base + per-lane 32-bit byte offset
__device__ __forceinline__ void dma16_uniform(const void* base, uint32_t lane_off, char* lds_block) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_address(lds_block)), "v"(lane_off), "s"(base)
                 : "memory", "m0");
}
// One wavefront-wide 256-byte copy: lane i's 4 bytes from its own address land at lds_block + 4*i.
__device__ __forceinline__ void dma4(const void* src, char* lds_block) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
                 :
                 : "s"(lds_address(lds_block)), "v"(src)
                 : "memory", "m0");
}

// Copy a ROWS x ROWB-byte tile into LDS; row r comes from row_ptr(r) (16-byte aligned, ROWB readable bytes).
// Each wavefront issues ROWS*ROWB/4096 instructions of 1 KiB.
template <typename T, int ROWB, int ROWS, int SWZ, typename RowPtr>
__device__ __forceinline__ void dma_tile(char* tile, int wave, int lane, RowPtr row_ptr) {
    constexpr int NI = ROWS * ROWB / 1024;  // wavefront instructions per tile
    constexpr int CPR = ROWB / 16;          // chunks per row
    static_assert(NI % 4 == 0 && (1024 % ROWB == 0 || ROWB % 1024 == 0), "tile shape");
#pragma unroll
    for (int i = 0; i < NI / 4; ++i) {
        const int q = wave + 4 * i;
        const int flat = q * 64 + lane;  // chunk position in the tile
        const int row = flat / CPR, pc = flat % CPR;
        const int c = logical_chunk<ROWB, SWZ>(row, pc);
        dma16(reinterpret_cast<const char*>(row_ptr(row)) + c * 16, tile + q * 1024);
    }
}

typedef __attribute__((address_space(3))) const u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) const float lds_f32;

__device__ __forceinline__ u32x4 lds_load128(uint32_t addr) { return *reinterpret_cast<lds_u32x4*>((uintptr_t)addr); }
__device__ __forceinline__ s16x4 lds_load_tr16(uint32_t addr) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>((uintptr_t)addr));
}
__device__ __forceinline__ void lds_store128(uint32_t addr, u32x4 x) {
    *reinterpret_cast<__attribute__((address_space(3))) u32x4*>((uintptr_t)addr) = x;
}
__device__ __forceinline__ float lds_load_f32(uint32_t addr) { return *reinterpret_cast<lds_f32*>((uintptr_t)addr); }

// Wait until at most N of this wavefront's global loads (LDS-DMA copies included) are outstanding.
template <int N>
__device__ __forceinline__ void wait_loads() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

}  // namespace splat

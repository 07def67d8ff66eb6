// Pieces of the kernels whose wavefronts own 16 rows (attention_f32.hip, attention_bwd_f32.hip, attention_bwd_f32_keys.hip,
// attention_rows16.hip, operators_f32.hip, sddmm_rows16.hip): reductions over the lanes of a row, the walk of half a row block over its tiles, and the rows'
// windows.  Lane (n = lane % 16, g = lane / 16) holds row n's scores at positions 4g .. 4g + 3 of every subtile of 16.
#pragma once
#include "attn_tile.hpp"

namespace splat {

constexpr int kHalfRows = 64;  // rows of a workgroup: 4 wavefronts of 16, half a row block of the plan

// f over the four lanes n, n + 16, n + 32, n + 48 of a column; all four get the result
template <typename F>
__device__ __forceinline__ float over_groups(float x, F f) {
    const auto a = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
    const uint32_t a0 = a[0], a1 = a[1];
    x = f(__builtin_bit_cast(float, a0), __builtin_bit_cast(float, a1));
    const auto b = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
    const uint32_t b0 = b[0], b1 = b[1];
    return f(__builtin_bit_cast(float, b0), __builtin_bit_cast(float, b1));
}

// f over the 16 lanes of a group (rotations inside a row of 16 lanes)
template <typename F>
__device__ __forceinline__ int over_rows16(int x, F f) {
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, true));
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x124, 0xf, 0xf, true));
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x122, 0xf, 0xf, true));
    return f(x, __builtin_amdgcn_update_dpp(0, x, 0x121, 0xf, 0xf, true));
}

// The extent of a wavefront's 16 rows in tile positions, as wave_span, from lanes that hold the window of row n = lane % 16
__device__ __forceinline__ WaveSpan span_of_rows16(const RowWin& w, bool uniform) {
    const bool empty = w.cnt <= 0;
    auto lo = [](int a, int b) { return min(a, b); };
    auto hi = [](int a, int b) { return max(a, b); };
    WaveSpan s;
    s.lo_min = __builtin_amdgcn_readfirstlane(over_rows16(empty ? 0x3fffffff : w.lo, lo));
    s.lo_max = __builtin_amdgcn_readfirstlane(over_rows16(empty ? 0x3fffffff : w.lo, hi));
    s.hi_min = __builtin_amdgcn_readfirstlane(over_rows16(empty ? -0x3fffffff : w.lo + w.cnt, lo));
    s.hi_max = __builtin_amdgcn_readfirstlane(over_rows16(empty ? -0x3fffffff : w.lo + w.cnt, hi));
    if (!uniform) s.lo_max = 0x3fffffff;
    return s;
}

// acc[16x16] += A[16x4] . B[4x16] in float32; lane (n, g) holds value g of row n (A), of column n (B), rows 4g .. 4g + 3 of column n (acc)
__device__ __forceinline__ void mma4(f32x4& acc, float a, float b) { acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0); }

// Position of a walk over tiles of BN positions: the segment, its plan, the next tile and the end of the segment's range.
struct HalfWalk {
    int seg, tile, end;
    SegPlan pl;
};

// Segment sg of row block rb in the plan table, cut down to the tiles that the given half of the block's rows sees
template <int BN>
__device__ __forceinline__ HalfWalk half_walk(const PlanRec* pt, int n_rb, int n_seg, int rb, int half, int sg) {
    HalfWalk w;
    w.seg = sg;
    const PlanRec r = plan_uniform_load(pt + plan_seg_at(n_seg, rb, sg));
    w.pl.c0 = r.x, w.pl.cs = r.y, w.pl.n_tiles = r.z, w.pl.uniform = r.w;
    const PlanRec s0 = plan_uniform_load(pt + plan_span_at(n_rb, n_seg, rb, sg, 2 * half));
    const PlanRec s1 = plan_uniform_load(pt + plan_span_at(n_rb, n_seg, rb, sg, 2 * half + 1));
    w.tile = max(min(s0.x, s1.x), 0) / BN;
    w.end = max(min((max(max(s0.w, s1.w), 0) + BN - 1) / BN, r.z * (kBN / BN)), w.tile);
    return w;
}

// The window of one row in the walk of the current segment, the periodic part of its live positions, and the extent of the
// wavefront's 16 rows: subtiles before lo_min / from hi_max on hold nothing for it, from lo_max to hi_min they need no mask.
struct RowState {
    RowWin win;
    int first, dec;  // dec: by how much `first` falls per tile
    uint64_t pat;
    int lo_min, lo_max, hi_min, hi_max;

    template <int BN>
    __device__ __forceinline__ void enter(const RowWin& w, int phase, bool uniform, int tile0) {
        win = w;
        first = 0, dec = 0, pat = ~0ull;
        if (!uniform) {
            dec = BN % w.lin;
            first = phase - (tile0 * BN) % w.lin;
            if (first < 0) first += w.lin;
            pat = 0;
            for (int q = 0; q < 64; q += w.lin) pat |= 1ull << q;
        }
        const bool empty = w.cnt <= 0;
        auto lo = [](int a, int b) { return min(a, b); };
        auto hi = [](int a, int b) { return max(a, b); };
        lo_min = __builtin_amdgcn_readfirstlane(over_rows16(empty ? 0x3fffffff : w.lo, lo));
        lo_max = __builtin_amdgcn_readfirstlane(over_rows16(empty ? 0x3fffffff : w.lo, hi));
        hi_min = __builtin_amdgcn_readfirstlane(over_rows16(empty ? -0x3fffffff : w.lo + w.cnt, lo));
        hi_max = __builtin_amdgcn_readfirstlane(over_rows16(empty ? -0x3fffffff : w.lo + w.cnt, hi));
        if (!uniform) lo_max = 0x3fffffff;  // never without a mask
    }
    __device__ __forceinline__ void next_tile() {
        const int f = first - dec;
        first = f < 0 ? f + win.lin : f;
    }
    // the scores of a tile (register j of subtile u: position j0 + 16u + 4g + j), `masked` where the row has no entry
    template <int SUB>
    __device__ __forceinline__ void mask_tile(f32x4 (&s)[SUB], int j0, int g, bool uniform, float masked = kNegBigA) const {
        if (uniform) {  // every position of the span
            const int at = j0 + 4 * g - win.lo;
#pragma unroll
            for (int u = 0; u < SUB; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) s[u][j] = (unsigned)(at + 16 * u + j) < (unsigned)win.cnt ? s[u][j] : masked;
        } else {
            asm volatile("");  // (keeps the bit masks below out of the paths that do not need them)
            const uint64_t bits = row_live_bits(win, j0, first, pat) >> (4 * g);
#pragma unroll
            for (int u = 0; u < SUB; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) s[u][j] = keep_or_mask(s[u][j], ((int)((uint32_t)(bits >> (16 * u)) << (31 - j))) >> 31, masked);
        }
    }
};

}  // namespace splat

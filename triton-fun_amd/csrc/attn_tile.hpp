// Pieces of the fused attention kernels (forward and backward) that work on one tile of scores.
#pragma once
#include "tile_copy.hpp"

namespace splat {

constexpr float kNegBigA = -1.0e30f;

struct AttnParams {
    const void* q;
    const void* k;
    const void* v;
    void* o;
    int64_t q_sb, q_sh, q_sl;
    int64_t k_sb, k_sh, k_sd, k_sl;
    int64_t v_sb, v_sh, v_sl;
    int64_t o_sb, o_sh, o_sl;
    int B, H, L;
    float scale_log2e;
    int n_seg;
    SegPtrs seg[SPLAT_MAX_SEGMENTS];
    int n_row_blocks;
    int total;
    int row_stride;
    const PlanRec* plan;  // plan table of this mask (PLANNED kernels), variant already selected
    float* lse;           // optional [B*H, L]: log of every row's sum of exponentials (natural log, scaled scores)
    int live_percent;     // host only: share of the walked positions that some row sees, 0 where the caller did not say
    Divisor by_blocks, by_h;  // workgroups per head and H, filled in by the launch
    bool keys_anywhere;   // host only: K^T with the keys contiguous whose rows are not whole 16-byte pieces
};

constexpr float kRescaleThreshold = 8.0f;  // in log2 units: exponentials stay below 2^8 before the reference moves

// the float32 forward (attention_f32.hip); p.n_row_blocks and p.total are filled in by the launch
int launch_attn_f32(const AttnParams& p, int d, bool kt, hipStream_t st);
// the 16-bit forward for launches of few row blocks (attention_rows16.hip)
template <typename T>
int launch_attn_rows16(const AttnParams& p, int d, bool kt, hipStream_t st);

// Live positions of one row in the tile that starts at position j0, one bit per position (bit b = position j0 + b):
// the row's span [lo, lo + cnt) intersected with its periodic pattern.  `first` is the smallest offset >= 0 in the tile
// whose position is congruent to the row's first one modulo its step (0 for unit step) and `pat` has a bit at every
// multiple of the step below 64.
__device__ __forceinline__ uint64_t row_live_bits(const RowWin& w, int j0, int first, uint64_t pat) {
    const int a = w.lo - j0, b = a + w.cnt;  // live range [a, b) in tile offsets
    const uint64_t lo_m = a <= 0 ? ~0ull : (a >= 64 ? 0ull : ~0ull << a);
    const uint64_t hi_m = b >= 64 ? ~0ull : (b <= 0 ? 0ull : (1ull << b) - 1ull);
    const uint64_t per = first < 64 ? pat << first : 0ull;
    return lo_m & hi_m & per;
}

// x where keep is -1, the masked score -1e30 where keep is 0 (one bit-field insert)
__device__ __forceinline__ float keep_or_mask(float x, int keep, float masked = kNegBigA) {
    const uint32_t xb = __builtin_bit_cast(uint32_t, x), nb = __builtin_bit_cast(uint32_t, masked);
    return __builtin_bit_cast(float, (xb & (uint32_t)keep) | (nb & ~(uint32_t)keep));
}

// Accumulator register j of a 32-key half of a tile holds the half's position 8*(j/4) + 4*g + j%4; `bits`, the half's part
// of `live` (see row_live_bits) moved down by 4*g, says whether the score is kept.
__device__ __forceinline__ void mask_half(f32x16& s, uint32_t bits) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int c = 8 * (j >> 2) + (j & 3);
        s[j] = keep_or_mask(s[j], ((int)(bits << (31 - c))) >> 31);
    }
}

}  // namespace splat

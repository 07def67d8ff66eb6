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
// the float32 forward whose wavefronts share the keys of 16 or 32 rows (attention_shared_f32.hip)
int launch_attn_shared_f32(const AttnParams& p, int d, bool kt, int rows, hipStream_t st);
// the 16-bit forward of 16 rows a wavefront (attention_rows16.hip)
template <typename T>
int launch_attn_rows16(const AttnParams& p, int d, bool kt, hipStream_t st);
// the 16-bit forward whose wavefronts share the keys of 32 rows (attention_shared.hip)
template <typename T>
int launch_attn_shared(const AttnParams& p, int d, bool kt, int waves, hipStream_t st);

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

// Keys c .. c + 7 of a row of K^T that may start anywhere (L >= 8).  Behind the row's last key there are zeros, or, in a piece that begins
// there, some of its last keys: positions that no row sees, whose scores are masked.
template <typename T>
__device__ __forceinline__ u32x4 keys_piece(const T* row, int c, int L) {
    const int over = min(max(c + 8 - L, 0), 8);  // how many of them do not exist: the row's last whole piece, moved down
    u32x4 x;
    __builtin_memcpy(&x, row + min(c, L - 8), 16);
    if (over > 0) {
        const uint64_t lo = (uint64_t)x[1] << 32 | x[0], hi = (uint64_t)x[3] << 32 | x[2];
        const int s = 16 * (over & 3);
        const uint64_t a = over >= 4 ? hi : lo, b = over >= 4 ? 0 : hi;
        const uint64_t l = s == 0 ? a : (a >> s) | (b << (64 - s)), h = b >> s;
        x = u32x4{(uint32_t)l, (uint32_t)(l >> 32), (uint32_t)h, (uint32_t)(h >> 32)};
    }
    return x;
}

// Exponentials of one tile of scores against the rows' references (mb = reference * c2), as MFMA B fragments; returns
// the lane's sum.
template <int NT, typename T>
__device__ __forceinline__ float exp_tile(const f32x16 (&s)[NT], Frag<T> (&pf)[NT][2], float mb, float c2) {
    float rs = 0.f;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float pv = fast_exp2(fmaf(s[nt][j], c2, -mb));
            rs += pv;
            pf[nt][j >> 3].v[j & 7] = (T)pv;
        }
    return rs;
}

// Fold one tile of 32*NT keys of (masked) scores of one 32-row tile into the running softmax state and emit the
// exponentials.  One lane owns one query row (half of its positions).  Returns whether every row of the wavefront
// has a real reference afterwards.
template <int NT, typename T, int DT>
__device__ __forceinline__ bool softmax_tile(f32x16 (&s)[NT], Frag<T> (&pf)[NT][2], float& m_ref, float& l_run,
                                             f32x16 (&o)[DT], float c2) {
    float mx = s[0][0];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int j = 0; j < 16; ++j) mx = fmaxf(mx, s[nt][j]);
    mx = with_lane_xor<32, 64>(mx, [](float a, float b) { return fmaxf(a, b); });  // the other half of the row lives in lane ^ 32
    // move the reference only when some row's maximum has outrun it by the threshold (always on the first
    // live tile); rows that do not move keep alpha = 1
    if (__any((mx - m_ref) * c2 > kRescaleThreshold)) {
        const float m_new = ((mx - m_ref) * c2 > kRescaleThreshold) ? mx : m_ref;
        const float alpha = fast_exp2((m_ref - m_new) * c2);
        const bool had_data = __any(m_ref > 0.5f * kNegBigA);  // otherwise O and l are still all zero
        m_ref = m_new;
        if (had_data) {
            l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int j = 0; j < 16; ++j) o[dt][j] *= alpha;
        }
    }
    // Masked scores are -1e30: their exponential underflows to exactly 0 as long as the reference is a real
    // score.  A row that has seen no live score yet keeps the -1e30 reference; give it offset 0 so that its
    // (all masked) entries still map to 0 instead of exp2(0).
    const bool real = m_ref > 0.5f * kNegBigA;
    l_run += exp_tile<NT, T>(s, pf, real ? m_ref * c2 : 0.f, c2);
    return !__any(!real);
}

}  // namespace splat

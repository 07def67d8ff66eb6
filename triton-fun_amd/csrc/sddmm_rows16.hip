// SDDMM on ACSR of 16-bit operands in launches of few row blocks, and of short rows in larger ones, inner dimension up to 128.
//
// Such a launch is one chain of latencies a workgroup, row maps -> plan -> tile -> products -> stores, and what shortens it is
// little work a workgroup: 64 rows of one (batch, head) in 4 wavefronts of 16, tiles of 64 positions requested a tile ahead through
// registers, two stages, one barrier a tile, and a row block's tiles shared out over workgroups until there are two a CU (four: 10.4
// for 9.1 us at 16 heads of 1024 rows, 300 slots, d = 32).  K stored along the keys is turned on its way into LDS, lanes = keys, wherever its
// rows start and whatever the step.  The kernels that took these launches, bfloat16, heads of 1024 rows, us: rows of K, 4 heads, 129 slots, d = 128
// (sddmm_lines.hip) 8.9 -> 6.6; 8 heads, 300 slots (sddmm.hip) d = 32 16.7 -> 7.5, d = 128 14.1 -> 8.6; K along the keys (sddmm.hip), 8 heads,
// 33 slots, d = 80 15.7 -> 6.3, 32 heads 16.5 -> 8.0; where K was turned by a launch of its own first, 16 heads of 1000 rows, 129 slots,
// d = 64, the three operators 26.5 -> 20.5.  An SpMM of this shape was slower than spmm_tile.hip's at every size (1.04 to 1.26).
#include <algorithm>

#include "rows16.hpp"
#include "sddmm_params.hpp"

namespace splat {

namespace {

constexpr int kTile = 64;
static_assert(kPlanBM == 2 * kHalfRows && kBN == kTile, "half a row block of the plan per workgroup, its tiles");

template <typename T>
struct Vec4 {
    typedef T type __attribute__((ext_vector_type(4)));
};

}  // namespace

// S^T = K Q^T: a lane owns one row and holds four consecutive positions of every 16.  KS: 32-value steps of the contraction.  SM: the softmax of
// its rows that a wavefront takes at the end (sddmm_params.hpp).
template <typename T, int KS, bool KT, int SM>
__global__ __launch_bounds__(256, 4) void sddmm_rows16_kernel(const SddmmParams p) {
    constexpr int ROWB = KS == 1 ? 64 : KS == 2 ? 128 : 256;  // bytes of an LDS row: a power of two, for the swizzle
    constexpr int STAGE = kTile * ROWB, CPR = 4 * KS, NP = kTile * CPR / 256;
    typedef typename Vec4<T>::type vec4;

    __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];
    __shared__ SegPlan s_plan[SPLAT_MAX_SEGMENTS];
    __shared__ PlanScratch<kHalfRows> s_ps;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;

    load_args(p.total, p.key_split, p.by_split.m, p.by_split.shift, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.n_row_blocks, p.H, p.row_stride, p.L,
              p.n_keys, p.d, p.T, p.n_seg, p.plan, p.q, p.q_sb, p.q_sh, p.q_sl, p.k, p.k_sb, p.k_sh, p.k_sd, p.k_sl, p.out);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int block = quotient(logical, p.by_split), share = logical - block * p.key_split;
    const int per_head = 2 * p.n_row_blocks;  // halves of the plan's row blocks
    const int bh = quotient(block, p.by_blocks);
    const int at_block = per_head - 1 - (block - bh * per_head);
    const int rb = at_block >> 1, half = at_block & 1;
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride, L = p.L, d = p.d;
    const int r0 = block_first_row(rb, kPlanBM, rs) + rs * half * kHalfRows;
    if (r0 >= L) return;

    const T* kb = (const T*)p.k + b * p.k_sb + h * p.k_sh;
    const int row_in = min(r0 + rs * (wave * 16 + n), L - 1);
    const u32x4 zero = {0u, 0u, 0u, 0u};

    Frag<T> q[KS];
    {
        const T* qr = (const T*)p.q + b * p.q_sb + h * p.q_sh + (int64_t)row_in * p.q_sl;
#pragma unroll
        for (int t = 0; t < KS; ++t) {
            q[t].v = __builtin_bit_cast(typename Frag<T>::vec, zero);
            if (32 * t + 8 * g < d) q[t] = global_frag<T>(qr + 32 * t + 8 * g);
        }
    }
    if (!p.plan) plan_segments<kHalfRows, kTile>(p.seg, p.n_seg, r0, rs, L, true, s_plan, &s_ps, tid);

    const uint32_t base = lds_address(smem);
    int pc_row[NP], pc_c[NP];
    uint32_t pc_to[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int f = tid + 256 * i;
        pc_row[i] = KT ? f % kTile : f / CPR;
        pc_c[i] = KT ? f / kTile : f % CPR;
        pc_to[i] = base + lds_off<ROWB, true>(pc_row[i], pc_c[i] * 16);
    }
    uint32_t k_addr[KS];
#pragma unroll
    for (int t = 0; t < KS; ++t) k_addr[t] = base + lds_off<ROWB, true>(n, (4 * t + g) * 16);

    T* const out_row = (T*)p.out + ((int64_t)bh * L + row_in) * p.T;
    // (one rounding as in sddmm_lines.hip, which takes the launches without a plan table: the same bits)
    const float exp_mul = p.scale * 1.4426950408889634f, exp_sub = p.row_lse ? p.row_lse[(int64_t)bh * L + row_in] * 1.4426950408889634f : 0.f;

    uint32_t stage = 0;
    for (int sg = 0; sg < p.n_seg; ++sg) {
        HalfWalk walk;
        RowWin win;
        if (p.plan) {
            const PlanRec rec = p.plan[plan_row_at(p.n_row_blocks, p.n_seg, rb, sg, half * kHalfRows + wave * 16 + n)];
            walk = half_walk<kTile>(p.plan, p.n_row_blocks, p.n_seg, rb, half, sg);
            // (the table knows the mask alone: a row's slots are bounded by the buffer's here, as load_row_map does)
            const int64_t most = walk.pl.uniform ? (int64_t)p.seg[sg].max_cnt : (int64_t)rec.z * (p.seg[sg].max_cnt - 1) + 1;
            win.lo = rec.x, win.cnt = (int)min((int64_t)rec.y, most), win.lin = rec.z;
        } else {
            walk.pl.c0 = __builtin_amdgcn_readfirstlane(s_plan[sg].c0);
            walk.pl.cs = __builtin_amdgcn_readfirstlane(s_plan[sg].cs);
            walk.pl.n_tiles = __builtin_amdgcn_readfirstlane(s_plan[sg].n_tiles);
            walk.pl.uniform = __builtin_amdgcn_readfirstlane(s_plan[sg].uniform);
            walk.tile = 0, walk.end = walk.pl.n_tiles;
            win = make_row_win(cached_row_map<kHalfRows>(&s_ps, sg, wave * 16 + n), walk.pl);
        }
        const SegPlan pl = walk.pl;
        const int tiles = walk.end - walk.tile;
        const int first = walk.tile + quotient(tiles * share, p.by_split), end = walk.tile + quotient(tiles * (share + 1), p.by_split);
        if (first >= end) continue;

        u32x4 raw[NP];
        auto load_tile = [&](int tile) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int key = min(max(pl.c0 + pl.cs * (tile * kTile + pc_row[i]), 0), p.n_keys - 1);
                raw[i] = zero;
                if (8 * pc_c[i] < d) {
                    if constexpr (KT) {
                        const T* src = kb + (int64_t)(8 * pc_c[i]) * p.k_sd + (int64_t)key * p.k_sl;
                        Frag<T> f;
#pragma unroll
                        for (int e = 0; e < 8; ++e) f.v[e] = src[e * p.k_sd];
                        raw[i] = __builtin_bit_cast(u32x4, f.v);
                    } else {
                        raw[i] = *reinterpret_cast<const u32x4*>(kb + (int64_t)key * p.k_sl + 8 * pc_c[i]);
                    }
                }
            }
        };
        load_tile(first);
        const WaveSpan span = span_of_rows16(win, pl.uniform != 0);
        T* const dst = out_row + p.seg[sg].slot_offset;

        for (int tile = first; tile < end; ++tile) {
            const int j0 = tile * kTile;
#pragma unroll
            for (int i = 0; i < NP; ++i) lds_store128(pc_to[i] + stage, raw[i]);
            lds_barrier();  // the tile is there, and everybody is done with the one before it, whose stage comes next
            if (tile + 1 < end) load_tile(tile + 1);
#pragma unroll
            for (int u = 0; u < kTile / 16; ++u) {
                const int ju = j0 + 16 * u;
                if (ju + 16 <= span.lo_min || ju >= span.hi_max) continue;
                f32x4 s = {0.f, 0.f, 0.f, 0.f};
                Frag<T> kf[KS];
#pragma unroll
                for (int t = 0; t < KS; ++t)
                    kf[t].v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128(k_addr[t] + stage + 16 * u * ROWB));
#pragma unroll
                for (int t = 0; t < KS; ++t) mma16(s, kf[t], q[t]);
                if (p.row_lse) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) s[j] = fast_exp2(fmaf(s[j], exp_mul, -exp_sub));
                } else {
                    s *= p.scale;
                }
                vec4 x;
#pragma unroll
                for (int j = 0; j < 4; ++j) x[j] = rounded<T>(s[j]);
                const int at = ju + 4 * g - win.lo;  // of the lane's first position, from the row's first
                if (ju >= span.lo_max && ju + 16 <= span.hi_min) {
                    __builtin_memcpy(dst + at, &x, 8);  // any alignment
                } else if (pl.uniform) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if ((unsigned)(at + j) < (unsigned)win.cnt) dst[at + j] = x[j];
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (win_live(win, ju + 4 * g + j)) dst[win_slot(win, ju + 4 * g + j)] = x[j];
                }
            }
            stage ^= STAGE;
        }
    }
    if constexpr (SM != kNoSoftmax) softmax_own_rows<T, SM, false>(p, bh, r0 + rs * 16 * wave, rs);
}

int launch_sddmm_rows16(const SddmmParams& p0, int in_dtype, bool kt, hipStream_t st) {
    if (p0.out_dtype != in_dtype || p0.d % 8 != 0 || p0.d > 128 || !p0.q_vec || (!kt && !p0.k_vec)) return 0;
    SddmmParams p = p0;
    p.n_row_blocks = count_row_blocks(p.L, kPlanBM, p.row_stride);
    const int64_t blocks = 2 * (int64_t)p.B * p.H * p.n_row_blocks;
    // The lines, as shares of the other kernels' time.  K along the keys, which the general kernel reads badly: 0.34 to 0.85 up to 512 blocks,
    // at 1024 0.66 to 0.89 for d = 80 and rows of 33 to 129 slots, 0.82 to 1.20 for d = 128 or 300 slots.
    // Rows of K of up to 256 slots with the plan table, masks of 33 to 129 slots: d <= 96 0.62 to 1.04 up to 640 blocks, 0.83 to 1.21 at 1024;
    // d = 128 0.60 to 0.91 up to 256, 0.84 to 1.07 from 384 to 640.  Without the table the prologue is longer, and once more for every segment:
    // d <= 96 0.42 to 0.98 at 256 blocks, 0.84 to 1.08 at 512, d = 128 0.65 to 1.01 at 128, 0.89 to 1.03 at 256; two segments 0.90 to 0.99 at
    // half of that, 1.01 to 1.06 there.  (sddmm_lines.hip, which takes the others, adds in the same order: the table changes no bit.)
    // Longer rows: the others are the general kernel's up to 511, which adds in another order, so the line is one for both.  With the table and
    // without, one segment of up to 400 slots 0.34 to 1.11 up to 512 blocks, two of up to 700 0.28 to 1.06; beyond, 0.35 to 1.00 up to 256
    // (320 to 512: 0.73 to 1.42) but for one segment at d = 64, 0.55 to 0.85 up to 128, 0.84 to 1.20 at 192 and 256.
    const bool d64 = p.d > 32 && p.d <= 64, wide = p.d > 96;
    const int long_rows = p.T <= (p.n_seg > 1 ? 700 : 400) ? 512 : d64 && p.n_seg == 1 ? 128 : 256;
    const int rows = p.T > 256 ? long_rows : p.plan ? (wide ? 256 : 640) : (wide ? 128 : 256) / p.n_seg;
    const int most = kt ? (p.d > 64 && p.d <= 96 && p.T <= 256 ? 1024 : 512) : rows;
    // And with the table, launches that fill the chip, rows of K: rows of at most 40 slots at 0.70 to 0.95 (one of 40 launches 1.03) up to 16384
    // blocks; longer ones that are no whole 64-byte pieces, which the line-wise kernel stores in most, from where that has more than its one
    // round of workgroups (at 1024 blocks 0.83 to 1.10) to 4096: d <= 32 0.57 to 0.95, d = 64 from 129 slots on 0.63 to 0.99, d = 80 to 128 up
    // to 240 slots 0.55 to 0.96 (whole pieces, 128 slots, 1.05 to 1.32; 251 slots at d = 128 1.06 to 1.12).
    const bool ragged = p.T % 32 != 0 && p.T <= (p.d > 64 ? 240 : 255) && (p.d <= 32 || p.d > 64 || p.T >= 120);
    const bool fills = !kt && p.plan && (p.T <= 40 ? blocks <= 16384 : ragged && blocks > 1024 && blocks <= 4096);
    if (blocks > most && !fills) return 0;
    p.key_split = (int)std::min<int64_t>((p.T + kTile - 1) / kTile + 2, std::max<int64_t>(1, 512 / blocks));
    // Whole rows where their softmax follows here: at 256 blocks 0.80 to 0.97 of the three launches' time (33 to 256 slots, d = 64 and 128)
    // against those with two workgroups a block; at 192 0.92 to 1.14, and below, where more share a block, up to 1.25.
    if (blocks >= 256 && own_rows_fit(p)) p.key_split = 1;
    if (p.key_split != 1 || !own_rows_fit(p)) p.probs = nullptr;
    p.total = (int)(blocks * p.key_split);
    p.by_split = divisor(p.key_split), p.by_blocks = divisor(2 * p.n_row_blocks), p.by_h = divisor(p.H);
    const int grid = ((p.total + 7) / 8) * 8;
    auto go = [&](auto t, auto kt_c) {
        using T = decltype(t);
        constexpr bool KT = decltype(kt_c)::value;
        by_split_of<kSoftmax32, kSoftmax512>(p, [&](auto sm) {
            constexpr int SM = decltype(sm)::value;
            if (p.d <= 32) sddmm_rows16_kernel<T, 1, KT, SM><<<grid, 256, 0, st>>>(p);
            else if (p.d <= 64) sddmm_rows16_kernel<T, 2, KT, SM><<<grid, 256, 0, st>>>(p);
            else if (p.d <= 96) sddmm_rows16_kernel<T, 3, KT, SM><<<grid, 256, 0, st>>>(p);
            else sddmm_rows16_kernel<T, 4, KT, SM><<<grid, 256, 0, st>>>(p);
        });
    };
    auto by_type = [&](auto kt_c) { return in_dtype == SPLAT_BF16 ? go(bf16{}, kt_c) : go(f16{}, kt_c); };
    if (kt) by_type(std::true_type{});
    else by_type(std::false_type{});
    return p.probs ? 2 : 1;
}

}  // namespace splat

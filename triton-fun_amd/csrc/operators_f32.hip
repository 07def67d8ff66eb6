// SDDMM and SpMM on ACSR in float32, inner dimension and output columns up to 128.
//
// A workgroup of 4 wavefronts owns 64 rows of one (batch, head), a wavefront 16 of them, and walks their key positions in tiles of
// 32: the float32 matrix instructions of 16 rows skip more of the masked positions than those of 32, half the rows a
// workgroup put twice as many of them on the chip, and 8 to 35 KiB of LDS and under 128 registers let four share a CU.  Float32 launches are
// small (a tenth of the 16-bit rate makes large ones rare), so what bounds them is the chain row maps -> plan -> tile ->
// products of a workgroup and how many of these chains are in flight.  A tile is requested a tile ahead, through registers, and written
// to one of two stages, one barrier a tile.
// The three operators against the kernels of 128 rows a workgroup and tiles of 64 that took these launches before (sddmm.hip, spmm.hip, which
// keep the longer rows and 16-bit outputs): 2 heads of 2048 rows, blocks of 64, d = 80 58 -> 22 us; 2 heads of 3001 rows, 501 slots, d = 96
// 135 -> 60; 16 heads of 2048, 256 slots, d = 64 87 -> 61, 128 heads 465 -> 361; 64 heads of 2048, 129 slots, d = 128 267 -> 185; where the
// matrix instructions bound both (64 heads of 4096, blocks of 512) 586 -> 577.  Over 900 launches of 1 to 128 heads of 200 to 2048 rows, 9 to
// 513 slots, d = 16 to 128, causal, windowed, strided and blocked masks: SDDMM 0.26 to 1.24 of the time, 0.58 in the mean, SpMM 0.20 to 1.06,
// 0.45.  Large launches of longer rows at d <= 64 are at the upper end; where SDDMM leaves them stands at its launcher.  SpMM keeps them: of 192 to
// 1024 slots and 512 to 2048 row blocks of d = 16 to 128 0.51 to 1.18, 16 of 864 above 1.02, all of blocked masks at d = 32 and 64.
#include <algorithm>

#include "rows16.hpp"
#include "sddmm_params.hpp"
#include "spmm_params.hpp"

namespace splat {

namespace {

constexpr int kRows = 64, kTile = 32;

// values 4c .. 4c + 3 of a row of n values, zeros past its end; `vec`: the row starts on a 16-byte boundary
__device__ __forceinline__ f32x4 row_piece(const float* row, int c, int n, bool vec) {
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
    if (vec && 4 * c + 4 <= n) {
        x = *reinterpret_cast<const f32x4*>(row + 4 * c);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (4 * c + e < n) x[e] = row[4 * c + e];
    }
    return x;
}

}  // namespace

// out[bh, r, s] = scale * q[r] . k[column of slot s], or the probability exp(that - lse[r]).  S^T = K Q^T: a lane owns one row and
// holds four consecutive positions of every 16.  KQ: 16-value steps of the contraction.  KT: K stored along the keys; it is turned on its
// way into LDS, lanes = keys, wherever its rows start.  SM: the softmax of its rows that a wavefront takes at the end (sddmm_params.hpp).
template <int KQ, bool KT, int SM>
__global__ __launch_bounds__(256, 4) void sddmm_f32_kernel(const SddmmParams p) {
    constexpr int ROWB = KQ <= 2 ? 128 : KQ <= 4 ? 256 : 512;  // bytes of an LDS row: a power of two, for the swizzle
    constexpr int STAGE = kTile * ROWB, CPR = 4 * KQ, NP = kTile * CPR / 256;

    __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];
    __shared__ SegPlan s_plan[SPLAT_MAX_SEGMENTS];
    __shared__ PlanScratch<kRows> s_ps;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;

    load_args(p.total, p.key_split, p.by_split.m, p.by_split.shift, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.n_row_blocks, p.H, p.row_stride, p.L,
              p.n_keys, p.d, p.T, p.n_seg, p.plan, p.q, p.q_sb, p.q_sh, p.q_sl, p.k, p.k_sb, p.k_sh, p.k_sd, p.k_sl, p.out);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int block = quotient(logical, p.by_split), share = logical - block * p.key_split;
    const int bh = quotient(block, p.by_blocks);
    const int rb = p.n_row_blocks - 1 - (block - bh * p.n_row_blocks);
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride, L = p.L, d = p.d;
    const int r0 = block_first_row(rb, kRows, rs);

    const float* kb = (const float*)p.k + b * p.k_sb + h * p.k_sh;
    const int my_row = r0 + rs * (wave * 16 + n);
    const int row_in = min(my_row, L - 1);

    f32x4 q[KQ];
    {
        const float* qr = (const float*)p.q + b * p.q_sb + h * p.q_sh + (int64_t)row_in * p.q_sl;
#pragma unroll
        for (int t = 0; t < KQ; ++t) q[t] = row_piece(qr, 4 * t + g, d, p.q_vec);
    }
    plan_segments<kRows, kTile>(p.seg, p.n_seg, r0, rs, L, true, s_plan, &s_ps, tid);

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
    uint32_t k_addr[KQ];
#pragma unroll
    for (int t = 0; t < KQ; ++t) k_addr[t] = base + lds_off<ROWB, true>(n, (4 * t + g) * 16);

    float* const out_row = (float*)p.out + ((int64_t)bh * L + row_in) * p.T;
    const float lse = p.row_lse ? p.row_lse[(int64_t)bh * L + row_in] : 0.f;

    uint32_t stage = 0;
    for (int sg = 0; sg < p.n_seg; ++sg) {
        SegPlan pl = s_plan[sg];
        pl.c0 = __builtin_amdgcn_readfirstlane(pl.c0);
        pl.cs = __builtin_amdgcn_readfirstlane(pl.cs);
        pl.n_tiles = __builtin_amdgcn_readfirstlane(pl.n_tiles);
        pl.uniform = __builtin_amdgcn_readfirstlane(pl.uniform);
        const int first = quotient(pl.n_tiles * share, p.by_split);
        const int end = quotient(pl.n_tiles * (share + 1), p.by_split);
        if (first >= end) continue;

        f32x4 raw[NP];
        auto load_tile = [&](int tile) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int key = min(max(pl.c0 + pl.cs * (tile * kTile + pc_row[i]), 0), p.n_keys - 1);
                if constexpr (KT) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int at = 4 * pc_c[i] + e;
                        raw[i][e] = kb[(int64_t)min(at, d - 1) * p.k_sd + key];
                        if (at >= d) raw[i][e] = 0.f;
                    }
                } else {
                    raw[i] = row_piece(kb + (int64_t)key * p.k_sl, pc_c[i], d, p.k_vec);
                }
            }
        };
        load_tile(first);
        const RowWin win = make_row_win(cached_row_map<kRows>(&s_ps, sg, wave * 16 + n), pl);
        const WaveSpan span = span_of_rows16(win, pl.uniform != 0);
        float* const dst = out_row + p.seg[sg].slot_offset;

        for (int tile = first; tile < end; ++tile) {
            const int j0 = tile * kTile;
#pragma unroll
            for (int i = 0; i < NP; ++i) lds_store128(pc_to[i] + stage, __builtin_bit_cast(u32x4, raw[i]));
            lds_barrier();  // the tile is there, and everybody is done with the one before it, whose stage comes next
            if (tile + 1 < end) load_tile(tile + 1);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int ju = j0 + 16 * u;
                if (ju + 16 <= span.lo_min || ju >= span.hi_max) continue;
                f32x4 kf[KQ];
#pragma unroll
                for (int t = 0; t < KQ; ++t) kf[t] = __builtin_bit_cast(f32x4, lds_load128(k_addr[t] + stage + 16 * u * ROWB));
                f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int t = 0; t < KQ; ++t)
#pragma unroll
                    for (int j = 0; j < 4; ++j) mma4(s, kf[t][j], q[t][j]);
                s *= p.scale;
                if (p.row_lse) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) s[j] = fast_exp2((s[j] - lse) * 1.4426950408889634f);
                }
                const int at = ju + 4 * g - win.lo;  // of the lane's first position, from the row's first
                if (ju >= span.lo_max && ju + 16 <= span.hi_min) {
                    __builtin_memcpy(dst + at, &s, 16);  // any alignment
                } else if (pl.uniform) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if ((unsigned)(at + j) < (unsigned)win.cnt) dst[at + j] = s[j];
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (win_live(win, ju + 4 * g + j)) dst[win_slot(win, ju + 4 * g + j)] = s[j];
                }
            }
            stage ^= STAGE;
        }
    }
    if constexpr (SM != kNoSoftmax) softmax_own_rows<float, SM, false>(p, bh, r0 + rs * 16 * wave, rs);
}

// out[bh, r, :] = sum over the live slots s of p[bh, r, s] * v[column of s, :].  O^T = V^T P^T: a lane reads its row's entries at 8 consecutive
// positions straight from the compressed row, zeros where the row has none, and holds four consecutive columns of every 16.
// NT: 16-column tiles of the output that a workgroup takes.
template <int NT>
__global__ __launch_bounds__(256, 4) void spmm_f32_kernel(const SpmmParams p) {
    // 16 bytes of padding: rows 8 apart, which the lanes of one read touch, fall into different halves of the banks
    constexpr int ROWB = NT * 64 + 16, STAGE = kTile * ROWB, CPR = 4 * NT, NP = kTile * CPR / 256;

    __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];
    __shared__ SegPlan s_plan[SPLAT_MAX_SEGMENTS];
    __shared__ PlanScratch<kRows> s_ps;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;

    load_args(p.total, p.by_chunks.m, p.by_chunks.shift, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.n_row_blocks, p.H, p.row_stride, p.L,
              p.n_keys, p.n_out, p.T, p.n_seg, p.plan, p.v, p.v_sb, p.v_sh, p.v_sl, p.p);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int block = quotient(logical, p.by_chunks), col0 = (logical - block * p.n_col_chunks) * (16 * NT);
    const int bh = quotient(block, p.by_blocks);
    const int rb = p.n_row_blocks - 1 - (block - bh * p.n_row_blocks);
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride, L = p.L;
    const int r0 = block_first_row(rb, kRows, rs);

    const float* vb = (const float*)p.v + b * p.v_sb + h * p.v_sh;
    const int my_row = r0 + rs * (wave * 16 + n);
    const float* const p_row = (const float*)p.p + ((int64_t)bh * L + min(my_row, L - 1)) * p.T;
    plan_segments<kRows, kTile>(p.seg, p.n_seg, r0, rs, L, true, s_plan, &s_ps, tid);

    const uint32_t base = lds_address(smem);
    int pc_row[NP], pc_c[NP];
    uint32_t pc_to[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int f = tid + 256 * i;
        pc_row[i] = f / CPR;
        pc_c[i] = f % CPR;
        pc_to[i] = base + pc_row[i] * ROWB + pc_c[i] * 16;
    }
    const uint32_t v_addr = base + 8 * g * ROWB + n * 4;

    f32x4 o[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};

    uint32_t stage = 0;
    for (int sg = 0; sg < p.n_seg; ++sg) {
        SegPlan pl = s_plan[sg];
        pl.c0 = __builtin_amdgcn_readfirstlane(pl.c0);
        pl.cs = __builtin_amdgcn_readfirstlane(pl.cs);
        pl.n_tiles = __builtin_amdgcn_readfirstlane(pl.n_tiles);
        pl.uniform = __builtin_amdgcn_readfirstlane(pl.uniform);
        if (pl.n_tiles == 0) continue;

        f32x4 raw[NP];
        auto load_tile = [&](int tile) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int key = min(max(pl.c0 + pl.cs * (tile * kTile + pc_row[i]), 0), p.n_keys - 1);
                raw[i] = row_piece(vb + (int64_t)key * p.v_sl, col0 / 4 + pc_c[i], p.n_out, p.v_vec);
            }
        };
        load_tile(0);
        const RowWin win = make_row_win(cached_row_map<kRows>(&s_ps, sg, wave * 16 + n), pl);
        const WaveSpan span = span_of_rows16(win, pl.uniform != 0);
        const float* const src = p_row + p.seg[sg].slot_offset;
        auto dead = [&](int j0) { return j0 + kTile <= span.lo_min || j0 >= span.hi_max; };
        auto inside = [&](int j0) { return j0 >= span.lo_max && j0 + kTile <= span.hi_min; };
        f32x8 pr;
        auto load_probs = [&](int tile) {
            const int j0 = tile * kTile;
            if (dead(j0)) return;
            const int at = j0 + 8 * g - win.lo;
            if (inside(j0)) {
                __builtin_memcpy(&pr, src + at, 32);  // any alignment
            } else if (pl.uniform) {
                const int last = max(win.cnt - 1, 0);
#pragma unroll
                for (int e = 0; e < 8; ++e) pr[e] = src[min(max(at + e, 0), last)];  // (what is not the row's goes when it is used)
            } else {
                pr = gather_affine8<f32x8>(src, win, j0 + 8 * g);
            }
        };
        load_probs(0);

        for (int tile = 0; tile < pl.n_tiles; ++tile) {
#pragma unroll
            for (int i = 0; i < NP; ++i) lds_store128(pc_to[i] + stage, __builtin_bit_cast(u32x4, raw[i]));
            f32x8 now = pr;
            lds_barrier();  // the tile is there, and everybody is done with the one before it, whose stage comes next
            if (tile + 1 < pl.n_tiles) {
                load_tile(tile + 1);
                load_probs(tile + 1);
            }
            if (!dead(tile * kTile)) {
                if (pl.uniform && !inside(tile * kTile)) {
                    const int at = tile * kTile + 8 * g - win.lo;
#pragma unroll
                    for (int e = 0; e < 8; ++e) now[e] = (unsigned)(at + e) < (unsigned)win.cnt ? now[e] : 0.f;
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float vf[NT];
#pragma unroll
                    for (int t = 0; t < NT; ++t) vf[t] = lds_load_f32(v_addr + stage + e * ROWB + 64 * t);
#pragma unroll
                    for (int t = 0; t < NT; ++t) mma4(o[t], vf[t], now[e]);
                }
            }
            stage = STAGE - stage;
        }
    }

    if (my_row < L) {
        float* const orow = (float*)p.out + ((int64_t)bh * L + my_row) * p.n_out;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int c = col0 + 16 * t + 4 * g;
            if (p.out_vec && c + 4 <= p.n_out) {
                *reinterpret_cast<f32x4*>(orow + c) = o[t];
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (c + j < p.n_out) orow[c + j] = o[t][j];
            }
        }
    }
}

int launch_sddmm_f32(const SddmmParams& p0, bool kt, hipStream_t st) {
    if (p0.d > 128 || p0.out_dtype != SPLAT_F32) return 0;
    SddmmParams p = p0;
    p.n_row_blocks = count_row_blocks(p.L, kRows, p.row_stride);
    const int64_t blocks = (int64_t)p.B * p.H * p.n_row_blocks;
    if (blocks > 0x7ffffff0) return 0;
    // Launches that fill the chip several times over are bound by the matrix instructions, and the general kernel, whose rows leave in whole
    // lines, catches up as rows get longer, first where this one pads the contraction (33 to 56 values to 64).  Means over five kinds of masks
    // and four such launches, rows of K / K along the keys: 384, 512, 768, 1024 slots, d = 16 0.92 / 0.95, 0.98 / 1.03, 1.11 / 1.15, 1.18 / 1.23;
    // d = 32 0.80 / 0.83, 0.87 / 0.92, 0.99 / 1.04, 1.09 / 1.13; d = 48 0.99 / 1.01, 1.07 / 1.11, 1.11 / 1.15, 1.16 / 1.19; d = 64 0.86 / 0.89,
    // 0.94 / 0.98, 0.97 / 1.01, 1.02 / 1.06 (blocked masks, which skip nothing, up to 0.3 above these); d = 80 and 128 0.54 to 0.97 throughout.
    // (host_ext.cpp turns K along the keys for gathered masks where these go to the general kernel: the same line stands there.)
    if (blocks >= 1024 && p.d <= 64 && p.T > (p.d > 32 && p.d <= 56 ? 450 : 600)) return 0;
    // Few row blocks: their tiles are shared out over up to three workgroups a CU, to no more than there are tiles (every further one has
    // the prologue and nothing to do).  Over 168 launches of 16 to 640 blocks 0.87 of the time that up to four and 32 a block take (4 heads
    // of 1024 rows, two segments of 94 slots, d = 128 17.7 -> 10.6 us); from 512 blocks on two a block pay for short contractions of longer rows
    // (129 and 300 slots: d = 32, 64 0.87 to 0.93 of one, d = 96, 128 1.01 to 1.17).
    p.key_split = (int)std::min<int64_t>((p.T + kTile - 1) / kTile + 3, std::max<int64_t>(1, 768 / blocks));
    if (p.key_split == 1 && blocks < 1024 && p.d <= 64 && p.T > 64) p.key_split = 2;
    // Whole rows where their softmax follows here: the three operators, 33 to 256 slots, at 256 blocks 0.83 to 0.94 of the time with shared ones
    // (d = 64; d = 128 0.96 to 1.05), at 512 0.84 to 0.98, at 1024 and 2048 0.80 to 0.99; beyond, up to 200 slots, 0.87 to 1.06.
    if (own_rows_fit(p) && blocks >= (p.d <= 64 ? 256 : 384)) p.key_split = 1;
    if (p.key_split != 1 || (p.T <= 200 && blocks > 2048) || !own_rows_fit(p)) p.probs = nullptr;
    p.total = (int)(blocks * p.key_split);
    p.by_split = divisor(p.key_split), p.by_blocks = divisor(p.n_row_blocks), p.by_h = divisor(p.H);
    const int grid = ((p.total + 7) / 8) * 8;
    auto go = [&](auto kq) {
        constexpr int KQ = decltype(kq)::value;
        by_split_of<kSoftmax32, kSoftmax256>(p, [&](auto sm) {
            constexpr int SM = decltype(sm)::value;
            if (kt)
                sddmm_f32_kernel<KQ, true, SM><<<grid, 256, 0, st>>>(p);
            else
                sddmm_f32_kernel<KQ, false, SM><<<grid, 256, 0, st>>>(p);
        });
    };
    if (p.d <= 32) go(std::integral_constant<int, 2>{});
    else if (p.d <= 64) go(std::integral_constant<int, 4>{});
    else if (p.d <= 96) go(std::integral_constant<int, 6>{});
    else go(std::integral_constant<int, 8>{});
    return p.probs ? 2 : 1;
}

int launch_spmm_f32(const SpmmParams& p0, hipStream_t st) {
    if (p0.n_out > 128 || p0.out_dtype != SPLAT_F32) return 0;
    SpmmParams p = p0;
    p.n_row_blocks = count_row_blocks(p.L, kRows, p.row_stride);
    const int64_t blocks = (int64_t)p.B * p.H * p.n_row_blocks;
    if (blocks > 0x7ffffff0) return 0;
    // Launches of few row blocks share the columns out as well: a wavefront's chain of matrix instructions, 32 cycles each, is what they wait
    // for.  Times over those of one workgroup a row block, masks of 33 to 300 slots: 32 columns a workgroup, up to 3 workgroups a CU
    // 0.48 to 0.98 (4 heads of 1024 rows, 300 slots, d = 128: 27.4 -> 13.1 us), at 4 0.84 to 1.07, above 0.95 to 1.48; 64 of 128 columns, up to
    // 4 a CU 0.67 to 0.95, at 8 1.08 to 1.21.
    const int tiles = (p.n_out + 15) / 16;
    const int nt = tiles <= 2 || blocks * ((tiles + 1) / 2) <= 768 ? 2 : tiles <= 4 || (tiles > 6 && blocks * 2 <= 1024) ? 4 : tiles <= 6 ? 6 : 8;
    p.n_col_chunks = (tiles + nt - 1) / nt;
    if (blocks * p.n_col_chunks > 0x7ffffff0) return 0;
    p.total = (int)(blocks * p.n_col_chunks);
    p.by_chunks = divisor(p.n_col_chunks), p.by_blocks = divisor(p.n_row_blocks), p.by_h = divisor(p.H);
    const int grid = ((p.total + 7) / 8) * 8;
    if (nt == 2) spmm_f32_kernel<2><<<grid, 256, 0, st>>>(p);
    else if (nt == 4) spmm_f32_kernel<4><<<grid, 256, 0, st>>>(p);
    else if (nt == 6) spmm_f32_kernel<6><<<grid, 256, 0, st>>>(p);
    else spmm_f32_kernel<8><<<grid, 256, 0, st>>>(p);
    return 1;
}

}  // namespace splat

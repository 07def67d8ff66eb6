// Fused ACSR sparse-attention forward in float32 (online softmax), gfx950.
//
// The float32 matrix instructions run at a sixteenth of the rate of the 16-bit ones (154 TFLOP/s in a large product), so both
// products are taken on the latter, of operands split into three bfloat16 parts (split3.hpp: six products for one, three eighths
// of the time, and closer to float64).  Bound: the 16-bit matrix instructions at the clock that the power limit leaves under
// them, and the vector instructions beside them, 200 a tile and wavefront in about as many cycles, half of them splitting.
//   * 16 rows a wavefront, 16x16x32 instructions, tiles of 32 positions, the layouts of attention_rows16.hip: 160 registers at
//     d = 64, three wavefronts a SIMD (two at d = 128), which overlap each other's vector and matrix phases.
//   * K and V are split once a workgroup: every thread holds its pieces of the next tile in registers, splits them, and writes the
//     parts between two barriers into the one stage of planes.  A second stage that is written during the products costs the LDS of
//     the third workgroup a CU (d = 64, 64 heads of 2048 rows, window 256 / 32: 72 / 35.4 us against 68 / 32.7; d = 128, of
//     the second: 204 / 102 against 127 / 59), 128 rows a workgroup halve the splitting but leave one or two of them a CU
//     (70 / 35.8 and 143 / 78), 32 rows a wavefront with the scores a tile ahead take 216 registers and run no faster.
//   * 64 rows a workgroup, so that launches that fill the chip once or twice spread over more CUs (those that do not:
//     attention_shared_f32.hip), and little that runs once: the instructions of the beginning and the end come from memory.
// Measured against the kernel on the float32 instructions that it replaces: B = 32, H = 12, L = 1024, window 257, d = 64: 252 -> 197 us;
// 64 heads of 4096 rows, blocks of 512, d = 64 517 -> 376; 64 heads of 2048 rows, d = 128, window 256 180 -> 127, window 32 66 -> 59;
// one head of 512 rows, window 64: 9.5 -> 8.7.  Relative error against float64 (norms) 2.5e-7 -> 1.6e-7 there, 4.0e-7 -> 3.0e-7 at
// window 257, 6.6e-7 -> 5.4e-7 at blocks of 1024 and d = 128.
#include <algorithm>

#include "rows16.hpp"
#include "split3.hpp"

namespace splat {

// The walk of a workgroup's own 64 rows.  It starts `at0` positions into the row block's (the plan's c0 moves along; the windows in the
// plan table are relative to the row block's): at the row block's tile that holds the first position that one of the rows sees, or,
// where that saves a tile, at that position, as for windows to both sides, which start in the middle of a tile (d = 128, window 33,
// 4 heads of 512 rows 12.4 -> 10.6 us, 64 of 2048 66.8 -> 57.6; the kernel on the float32 instructions, which skipped positions 16 at a
// time, took 12.0 for the former).  Dense walks start at a multiple of 16, and only there, since K stored along the keys is
// read in runs of 32 keys: causal windows of 8 to 128, from wherever they start, took 2 to 3 % longer with it at 64 heads of 2048.
struct OwnWalk {
    int seg, tile, end, at0;
    SegPlan pl;
};

template <int D, bool KT, bool PLANNED>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void attn_fwd_f32_kernel(const AttnParams p) {
    constexpr int BN = 32, ROWB = 2 * D, PLANE = BN * ROWB, TILE = 3 * PLANE;  // positions a tile; bytes of a row, a plane, an operand
    constexpr int KS = D / 32, DT = D / 16;
    constexpr int CPR = D / 8;                // 8-value pieces of a row
    constexpr int NP = 2 * BN * CPR / 256;    // pieces a thread: the first half of them K's, the others V's
    static_assert(kPlanBM == 2 * kHalfRows && kBN % BN == 0, "half a row block of the plan per workgroup");

    extern __shared__ __attribute__((aligned(1024))) char smem[];  // three planes of K, three of V
    __shared__ SegPlan s_plan[SPLAT_MAX_SEGMENTS];
    __shared__ PlanScratch<kPlanBM> s_ps;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;

    load_args(p.total, p.n_row_blocks, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.H, p.row_stride, p.L, p.n_seg, p.plan, p.scale_log2e,
              p.q, p.q_sb, p.q_sh, p.q_sl, p.k, p.k_sb, p.k_sh, p.k_sd, p.k_sl, p.v, p.v_sb, p.v_sh, p.v_sl);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int per_head = 2 * p.n_row_blocks;
    const int bh = quotient(logical, p.by_blocks);
    const int at = per_head - 1 - (logical - bh * per_head);  // later rows of causal patterns carry the most keys: first
    const int rb = at >> 1, half = at & 1;
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride, L = p.L;
    const int k0 = half * kHalfRows;                    // the workgroup's first row within its row block
    const int r0 = block_first_row(rb, kPlanBM, rs) + rs * k0;
    if (r0 >= L) return;

    const float* qb = (const float*)p.q + b * p.q_sb + h * p.q_sh;
    const float* kb = (const float*)p.k + b * p.k_sb + h * p.k_sh;
    const float* vb = (const float*)p.v + b * p.v_sb + h * p.v_sh;
    float* ob = (float*)p.o + b * p.o_sb + h * p.o_sh;
    const int my_row = r0 + rs * (wave * 16 + n);

    // ---- Q, resident: B operand of S^T; requested now, split once the first tile is on its way ----
    Frag<float> q_raw[KS];
    {
        const float* qr = qb + (int64_t)min(my_row, L - 1) * p.q_sl;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) q_raw[ks] = global_frag<float>(qr + 32 * ks + 8 * g);
    }

    // ---- plan: the row block's walk, cut down to the tiles that this half of it sees ----
    const PlanRec* const pt = p.plan;
    const int n_rb = p.n_row_blocks;
    if constexpr (!PLANNED) plan_segments<kPlanBM, kBN>(p.seg, p.n_seg, block_first_row(rb, kPlanBM, rs), rs, L, true, s_plan, &s_ps, tid);
    auto walk_of = [&](int sg) {
        OwnWalk w;
        w.seg = sg;
        int lo, hi;
        if constexpr (PLANNED) {
            const PlanRec r = plan_uniform_load(pt + plan_seg_at(p.n_seg, rb, sg));
            w.pl.c0 = r.x, w.pl.cs = r.y, w.pl.n_tiles = r.z, w.pl.uniform = r.w;
            const PlanRec s0 = plan_uniform_load(pt + plan_span_at(n_rb, p.n_seg, rb, sg, 2 * half));
            const PlanRec s1 = plan_uniform_load(pt + plan_span_at(n_rb, p.n_seg, rb, sg, 2 * half + 1));
            lo = min(s0.x, s1.x), hi = max(s0.w, s1.w);
        } else {
            const SegPlan l = s_plan[sg];
            w.pl.c0 = __builtin_amdgcn_readfirstlane(l.c0);
            w.pl.cs = __builtin_amdgcn_readfirstlane(l.cs);
            w.pl.n_tiles = __builtin_amdgcn_readfirstlane(l.n_tiles);
            w.pl.uniform = __builtin_amdgcn_readfirstlane(l.uniform);
            const RowWin win = make_row_win(cached_row_map<kPlanBM>(&s_ps, sg, k0 + lane), w.pl);
            lo = __builtin_amdgcn_readfirstlane(wave_min_i(win.cnt > 0 ? win.lo : 0x3fffffff));
            hi = __builtin_amdgcn_readfirstlane(wave_max_i(win.cnt > 0 ? win.lo + win.cnt : 0));
        }
        hi = min(hi, w.pl.n_tiles * kBN);
        w.at0 = 0, w.tile = 0, w.end = 0;
        if (lo < hi) {
            const int tiled = max(lo, 0) & ~(BN - 1), own = max(lo, 0) & (w.pl.cs == 1 ? ~15 : ~0);
            w.end = (hi - own + BN - 1) / BN;
            w.at0 = (hi - tiled + BN - 1) / BN > w.end ? own : tiled;
            w.pl.c0 += w.pl.cs * w.at0;
        }
        return w;
    };
    auto next_segment = [&](OwnWalk& w) {  // the first segment from w.seg on that has tiles
        for (int sg = w.seg; sg < p.n_seg; ++sg) {
            w = walk_of(sg);
            if (w.end > w.tile) return;
        }
        w.seg = p.n_seg, w.tile = 0, w.end = 0x7fffffff;
    };
    OwnWalk fetch;
    fetch.seg = 0;
    next_segment(fetch);
    int total = fetch.end - fetch.tile;
    for (int sg = fetch.seg + 1; sg < p.n_seg; ++sg) total += walk_of(sg).end;
    total = fetch.seg < p.n_seg ? __builtin_amdgcn_readfirstlane(total) : 0;

    // ---- a tile's way into LDS: pieces of 8 values, by their position in the tile's rows.  K stored along the keys is turned here:
    // lanes are keys, a piece is 8 loads, one of each d, wherever its rows start (32 heads of 2041 keys, window 256, against a launch that
    // turns K first: d = 64 58.6 -> 45.2 us, d = 128 125 -> 73, of which this kernel's own part is 49 -> 43 and 111 -> 67). ----
    int pc_row[NP], pc_c[NP];  // tile row and piece of the row
    uint32_t pc_to[NP];        // LDS address of its first part
    const uint32_t smem_base = lds_address(smem);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int f = (tid + 256 * i) % (BN * CPR);
        const bool is_k = i < NP / 2;
        const int row = KT && is_k ? f % BN : f / CPR, c = KT && is_k ? f / BN : f % CPR;
        const int to = is_k ? c ^ swz<ROWB>(row) : (((c >> 1) ^ swz32<ROWB>(row)) << 1) | (c & 1);
        pc_row[i] = row, pc_c[i] = c;
        pc_to[i] = smem_base + (is_k ? 0 : TILE) + row * ROWB + to * 16;
    }
    f32x8 raw[NP];
    // an operand of one head within 32-bit offsets, and strides that 24-bit products take
    const int64_t k_far = KT ? p.k_sd * D + L : p.k_sl * L, v_far = p.v_sl * L;
    const bool narrow = max(k_far, v_far) * 4 < ((int64_t)1 << 32) && max(KT ? p.k_sd : p.k_sl, p.v_sl) * 4 < (1 << 24) && p.k_sd >= 0;
    auto load_next = [&](OwnWalk& w) {  // the tile the walk stands at, which moves on
        const int c0 = w.pl.c0 + w.pl.cs * w.tile * BN;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const bool is_k = i < NP / 2;
            const char* base = reinterpret_cast<const char*>(is_k ? kb : vb);
            const int key = min(max(c0 + w.pl.cs * pc_row[i], 0), L - 1);
            if (KT && is_k) {
                if (narrow) {
                    uint32_t off = __umul24(8 * pc_c[i], (uint32_t)p.k_sd * 4) + 4 * key;
#pragma unroll
                    for (int e = 0; e < 8; ++e, off += (uint32_t)p.k_sd * 4) raw[i][e] = *reinterpret_cast<const float*>(base + off);
                } else {
                    const float* src = kb + (int64_t)(8 * pc_c[i]) * p.k_sd + key;
#pragma unroll
                    for (int e = 0; e < 8; ++e) raw[i][e] = src[e * p.k_sd];
                }
            } else {
                const int64_t sl = is_k ? p.k_sl : p.v_sl;
                if (narrow)
                    raw[i] = global_frag<float>(reinterpret_cast<const float*>(base + (__umul24(key, (uint32_t)sl * 4) + 32 * pc_c[i]))).v;
                else
                    raw[i] = global_frag<float>(reinterpret_cast<const float*>(base) + key * sl + 8 * pc_c[i]).v;
            }
        }
        if (++w.tile >= w.end) {
            ++w.seg;
            next_segment(w);
        }
    };

    // ---- LDS read addresses ----
    const int tr_row = (lane & 15) >> 2, tr_byte = 8 * (lane & 3);  // transposing reads: lane s of a group reads row s / 4
    uint32_t k_addr[KS], v_addr[DT];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) k_addr[ks] = smem_base + lds_off<ROWB, true>(n, (32 * ks + 8 * g) * 2);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        v_addr[dt] = smem_base + TILE + (4 * g + tr_row) * ROWB + (dt ^ swz32<ROWB>(4 * g + tr_row)) * 32 + tr_byte;

    // the row windows of the first segment with tiles, then the first tile, are requested before Q is looked at
    OwnWalk cur = fetch;
    PlanRec win_rec = {0, 0, 1, 0};
    if constexpr (PLANNED) {
        if (total > 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + wave * 16 + n)];
    }
    if (total > 0) load_next(fetch);
    Split3 qf[KS];
    float q_most = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        qf[ks] = split3(q_raw[ks].v);
#pragma unroll
        for (int e = 0; e < 8; ++e) q_most = fmaxf(q_most, fabsf(q_raw[ks].v[e]));
    }
    bool beyond = out_of_split(q_most);  // something that the split operands do not hold

    f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float c2 = p.scale_log2e, slack = kRescaleThreshold / c2;
    float m_ref = kNegBigA, l_run = 0.f;
    bool entered = false;
    RowState rows;

    for (int it = 0; it < total; ++it) {
        if (!entered) {
            RowWin w;
            int phase;
            if constexpr (PLANNED) {
                if (it > 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + wave * 16 + n)];
                w.lo = win_rec.x - cur.at0, w.cnt = win_rec.y, w.lin = win_rec.z, phase = win_rec.w;
                if (!cur.pl.uniform) {
                    phase -= cur.at0 % w.lin;
                    if (phase < 0) phase += w.lin;
                }
            } else {
                w = make_row_win(cached_row_map<kPlanBM>(&s_ps, cur.seg, k0 + wave * 16 + n), cur.pl);
                phase = cur.pl.uniform ? 0 : win_phase(w);
            }
            rows.template enter<BN>(w, phase, cur.pl.uniform != 0, cur.tile);
            entered = true;
        }
        const int j0 = cur.tile * BN;
        lds_barrier();  // everybody is done with tile it - 1
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const Split3 s = split3(raw[i]);
#pragma unroll
            for (int k = 0; k < 3; ++k) lds_store128(pc_to[i] + k * PLANE, __builtin_bit_cast(u32x4, s.p[k].v));
        }
        if (it + 1 < total) load_next(fetch);
        lds_barrier();  // tile `it` is there

        if (j0 + BN > rows.lo_min && j0 < rows.hi_max) {
            // ---- S^T = K . Q^T, of two subtiles of 16 positions.  Fragments are requested ahead of their products, part k of a
            // step as the one of the step before is done with ----
            Frag<bf16> kf[2][3];
            auto load_kf = [&](int ks, int k) {
#pragma unroll
                for (int u = 0; u < 2; ++u) kf[u][k].v = __builtin_bit_cast(bf16x8, lds_load128(k_addr[ks] + k * PLANE + 16 * u * ROWB));
            };
#pragma unroll
            for (int k = 2; k >= 0; --k) load_kf(0, k);
            __builtin_amdgcn_sched_barrier(0);
            f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int m = 0; m < 12 * KS; ++m) {
                const int ks = m / 12, i = (m % 12) / 2, u = m % 2;
                mma16(s[u], kf[u][kSplitA[i]], qf[ks].p[kSplitB[i]]);
                if (u == 1 && kSplitLast[kSplitA[i]] == i && ks + 1 < KS) load_kf(ks + 1, kSplitA[i]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (!(j0 >= rows.lo_max && j0 + BN <= rows.hi_min)) rows.mask_tile(s, j0, g, cur.pl.uniform != 0);
            // ---- online softmax against a lazily moved reference (see attention.hip): the row's maximum is only taken over its four
            // lanes where one of them has outrun the reference ----
            float mx = m_ref;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) mx = fmaxf(mx, s[u][j]);
            if (__any(mx - m_ref > slack)) {
                mx = over_groups(mx, [](float x, float y) { return fmaxf(x, y); });
                const float m_new = mx - m_ref > slack ? mx : m_ref;
                const float alpha = fast_exp2((m_ref - m_new) * c2);
                m_ref = m_new;
                l_run *= alpha;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
            }
            // a row that has seen no live score keeps offset 0, so that its (all masked) entries map to 0
            const float mb = m_ref > 0.5f * kNegBigA ? m_ref * c2 : 0.f;
            Frag<bf16> vf[2][3];
            auto load_vf = [&](int d2, int k) {
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    const uint32_t a0 = v_addr[2 * d2 + y] + k * PLANE;
                    vf[y][k] = frag_from_tr<bf16>(lds_load_tr16(a0), lds_load_tr16(a0 + 16 * ROWB));
                }
            };
#pragma unroll
            for (int k = 2; k >= 0; --k) load_vf(0, k);
            __builtin_amdgcn_sched_barrier(0);
            f32x8 e;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                e[j] = fast_exp2(fmaf(s[j >> 2][j & 3], c2, -mb));
                l_run += e[j];
            }
            const Split3 pf = split3(e);
            // ---- O^T += V^T . P^T, of two tiles of 16 columns at a time ----
#pragma unroll
            for (int m = 0; m < 6 * DT; ++m) {
                const int d2 = m / 12, i = (m % 12) / 2, y = m % 2;
                mma16(o[2 * d2 + y], vf[y][kSplitA[i]], pf.p[kSplitB[i]]);
                if (y == 1 && kSplitLast[kSplitA[i]] == i && 2 * d2 + 2 < DT) load_vf(d2 + 1, kSplitA[i]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (!cur.pl.uniform) rows.next_tile();
        if (++cur.tile >= cur.end) {
            ++cur.seg;
            next_segment(cur);
            entered = false;
        }
    }

    const float l_tot = over_groups(l_run, [](float x, float y) { return x + y; });
    // What is not finite anywhere stays so in a row's sum or outputs.  An output far below normal is one whose probabilities or values
    // are (one less than twice its bits: the smallest magnitude but zero).
    float chk = l_tot * 0.f;
    uint32_t least = ~0u;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float x = o[dt][j];  // (a bit cast of the element itself takes the vector's first)
            chk = fmaf(x, 0.f, chk);
            least = min(least, (__builtin_bit_cast(uint32_t, x) << 1) - 1);
        }
    beyond |= chk != 0.f || least < __builtin_bit_cast(uint32_t, 0x1p-104f * l_tot) << 1;  // (NaN compares unequal)
    if (__any(beyond)) {
        // ---- this wavefront's rows once more in float32 arithmetic, position by position, each lane a quarter of a row's columns,
        // live positions only.  64 heads of 2048 rows, d = 64, window 256, 67 us: with NaN in V at the last 64 keys, which the mask leaves to
        // their own rows but whose tiles others share, 255; at every 64th key, which sends every row here, 615 ----
        constexpr int QD = D / 4;
        const float* qr = qb + (int64_t)min(my_row, L - 1) * p.q_sl + g * QD;
        float q[QD], acc[QD];
#pragma unroll
        for (int i = 0; i < QD; ++i) q[i] = qr[i], acc[i] = 0.f;
        float m = -__builtin_inff(), l = 0.f;
        for (int sg = 0; sg < p.n_seg; ++sg) {
            const OwnWalk w = walk_of(sg);
            RowWin win;
            if constexpr (PLANNED) {
                const PlanRec wr = pt[plan_row_at(n_rb, p.n_seg, rb, sg, k0 + wave * 16 + n)];
                win.lo = wr.x - w.at0, win.cnt = wr.y, win.lin = wr.z;
            } else {
                win = make_row_win(cached_row_map<kPlanBM>(&s_ps, sg, k0 + wave * 16 + n), w.pl);
            }
            for (int j = 0; j < w.end * BN; ++j) {
                const bool live = win_live(win, j);
                if (!__any(live)) continue;
                const int64_t key = min(max(w.pl.c0 + w.pl.cs * j, 0), L - 1);
                const float* kr = KT ? kb + (int64_t)(g * QD) * p.k_sd + key : kb + key * p.k_sl + g * QD;
                float s = 0.f;
#pragma unroll
                for (int i = 0; i < QD; ++i) s = fmaf(q[i], kr[KT ? i * p.k_sd : i], s);
                s = over_groups(s, [](float x, float y) { return x + y; }) * c2;
                if (live) {
                    const float m_new = fmaxf(m, s);
                    const float off = m_new > -__builtin_inff() ? m_new : 0.f;
                    const float alpha = m > -__builtin_inff() ? fast_exp2(m - off) : 1.f;
                    const float e = fast_exp2(s - off);
                    m = m_new;
                    l = fmaf(l, alpha, e);
                    const float* vr = vb + key * p.v_sl + g * QD;
#pragma unroll
                    for (int i = 0; i < QD; ++i) acc[i] = fmaf(acc[i], alpha, e * vr[i]);
                }
            }
        }
        const float inv = l > 0.f ? 1.0f / l : 0.f;
        if (my_row < L) {
            if (p.lse != nullptr && g == 0)
                p.lse[(int64_t)bh * L + my_row] = l > 0.f ? (m + __log2f(l)) * 0.6931471805599453f : __builtin_inff();
            float* orow = ob + (int64_t)my_row * p.o_sl + g * QD;
#pragma unroll
            for (int i = 0; i < QD; ++i) orow[i] = acc[i] * inv;
        }
        return;
    }

    // ---- epilogue: a lane holds columns 16 dt + 4g .. + 3 of its row ----
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    if (my_row < L) {
        if (p.lse != nullptr && g == 0)
            p.lse[(int64_t)bh * L + my_row] = l_tot > 0.f ? (m_ref * c2 + __log2f(l_tot)) * 0.6931471805599453f : __builtin_inff();
        float* orow = ob + (int64_t)my_row * p.o_sl;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(orow + 16 * dt + 4 * g) = o[dt] * inv;
    }
}

template <int D, bool KT, bool PLANNED>
static int launch(const AttnParams& p0, hipStream_t st) {
    begin_launch();
    AttnParams p = p0;
    p.n_row_blocks = count_row_blocks(p.L, kPlanBM, p.row_stride);
    p.total = p.B * p.H * 2 * p.n_row_blocks;
    p.by_blocks = divisor(2 * p.n_row_blocks), p.by_h = divisor(p.H);
    const size_t lds = 6 * 32 * D * 2;
    auto kern = attn_fwd_f32_kernel<D, KT, PLANNED>;
    static uint64_t lds_reserved = 0;
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), lds, "splat_attention_fwd")) return rc;
    kern<<<((p.total + 7) / 8) * 8, 256, lds, st>>>(p);
    return check_launch("splat_attention_fwd");
}

int launch_attn_f32(const AttnParams& p, int d, bool kt, hipStream_t st) {
    // Few row blocks: the kernel whose wavefronts share the keys (attention_shared_f32.hip), of 16 rows up to 32 blocks, of 32 up to 64: as
    // long as its workgroups, one a CU or two at d = 64, are on the chip together.  This kernel -> that one, causal windows of 16 / 64 / 200 / 400:
    // d = 64, 4 heads of 1024 rows 7.3 -> 5.6, 8.5 -> 6.0, 14.9 -> 7.8, 22.2 -> 10.6 us, 8 heads 7.4 -> 7.2, 8.6 -> 7.7, 15.0 -> 10.0, 22.0 -> 13.7, 10 heads
    // 7.5 -> 9.8, 8.7 -> 10.3, 15.1 -> 14.4, 22.2 -> 20.5; d = 128, 4 heads 10.6 -> 8.0, 12.6 -> 8.8, 22.8 -> 12.2, 34.7 -> 17.4, 8 heads 10.8 -> 11.4 (a
    // twelfth of the walk live: those stay), 12.8 -> 12.3, 23.1 -> 16.7, 34.7 -> 23.5.
    const int64_t blocks = (int64_t)p.B * p.H * count_row_blocks(p.L, kPlanBM, p.row_stride);
    const int64_t row_bytes = 4 * std::max(p.v_sl, kt ? 0 : p.k_sl);  // (that kernel's offsets)
    if (row_bytes < (1 << 24) && row_bytes * p.L < ((int64_t)1 << 32)) {
        if (blocks <= 32) return launch_attn_shared_f32(p, d, kt, 16, st);
        if (blocks <= 64 && (d == 64 || p.live_percent == 0 || p.live_percent >= 20)) return launch_attn_shared_f32(p, d, kt, 32, st);
    }
    if (p.plan) {
        if (d == 64) return kt ? launch<64, true, true>(p, st) : launch<64, false, true>(p, st);
        return kt ? launch<128, true, true>(p, st) : launch<128, false, true>(p, st);
    }
    if (d == 64) return kt ? launch<64, true, false>(p, st) : launch<64, false, false>(p, st);
    return kt ? launch<128, true, false>(p, st) : launch<128, false, false>(p, st);
}

}  // namespace splat

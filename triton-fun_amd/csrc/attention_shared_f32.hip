// Fused ACSR sparse-attention forward in float32 in launches of few rows, gfx950: the wavefronts of a workgroup share the keys.
//
// Bound: latency, as in attention_shared.hip, whose division of the work this is: four wavefronts hold the same rows, 16 or 32, tile k
// of 32 positions goes to wavefront k % 4, and the parts meet in LDS at the end.  Products and their precision are those of
// attention_f32.hip (operands split into three bfloat16 parts, 16x16x32).  A wavefront is the only one to read its tiles, so that
// they go from memory into registers and are split there: no LDS, no barrier.
//   * scores: lane (n, g) holds columns 32 ks + 8g .. + 7 of key n and of Q's row n, which are the places they have in the other float32
//     kernels: a score has the same bits here, in a larger launch, and where the backward takes it again.  (With other columns in those
//     places, P of the backward was off from the statistic by both roundings: dQ of small training steps, windows 8 to 90, 3.6e-7 instead of 3.2e-7
//     against float64.)
//   * output: row r of tile dt of V^T is column (D / 16) r + dt, so that one position's columns of all tiles lie side by side in
//     memory, and a lane ends with D / 4 consecutive columns of its row.
// 32 rows (RG = 2) share every split of a tile, at twice the products of a wavefront: they come in where workgroups of 16 would run in
// two rounds.  Eight wavefronts instead of four: 3 to 8 % slower up to windows of 400.  One head of 512 rows, window 64, d = 64: 8.4 -> 6.0 us
// against attention_f32.hip; the lines stand there.  Relative error against float64, windows 64 / 400, d = 64: 1.9e-7, 2.5e-7 -> 1.7e-7, 1.8e-7.
#include "rows16.hpp"
#include "split3.hpp"

namespace splat {

// The walk of the 32 rows that the workgroup's are all or half of, over one segment, in tiles of 32 positions.  It starts at the first position that
// one of them sees, `at0` positions into the row block's.
struct SharedWalkF32 {
    int seg, tile, end, at0;
    int last;            // the last position that one of the rows sees
    int lo_max, hi_min;  // positions between them are live for every row
    SegPlan pl;
};

template <int D, bool KT, bool PLANNED, int RG>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void attn_fwd_shared_f32_kernel(const AttnParams p) {
    constexpr int KG = 4, BN = 32, KS = D / 32, DT = D / 16;
    constexpr int ROWS = 16 * RG;     // rows of the workgroup
    constexpr int OROW = D * 4 + 16;  // bytes of a row of a part

    extern __shared__ __attribute__((aligned(1024))) char smem[];  // the parts
    __shared__ SegPlan s_plan[SPLAT_MAX_SEGMENTS];
    __shared__ PlanScratch<kPlanBM> s_ps;
    __shared__ float s_ref[KG][ROWS], s_sum[KG][ROWS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;

    load_args(p.total, p.n_row_blocks, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.H, p.row_stride, p.L, p.n_seg, p.plan, p.scale_log2e,
              p.q, p.q_sb, p.q_sh, p.q_sl, p.k, p.k_sb, p.k_sh, p.k_sd, p.k_sl, p.v, p.v_sb, p.v_sh, p.v_sl);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    constexpr int PER = kPlanBM / ROWS;  // workgroups of a row block
    const int per_head = PER * p.n_row_blocks;
    const int bh = quotient(logical, p.by_blocks), b = quotient(bh, p.by_h);
    const int at = per_head - 1 - (logical - bh * per_head), h = bh - b * p.H;
    const int rb = at / PER, quarter = at % PER * RG / 2;
    const int rs = p.row_stride, L = p.L;
    const int k0 = at % PER * ROWS;
    const int r0 = block_first_row(rb, kPlanBM, rs) + rs * k0;
    if (r0 >= L) return;

    const float* qb = (const float*)p.q + b * p.q_sb + h * p.q_sh;
    const float* kb = (const float*)p.k + b * p.k_sb + h * p.k_sh;
    const float* vb = (const float*)p.v + b * p.v_sb + h * p.v_sh;
    float* ob = (float*)p.o + b * p.o_sb + h * p.o_sh;

    // ---- plan ----
    const PlanRec* const pt = p.plan;
    const int n_rb = p.n_row_blocks;
    if constexpr (!PLANNED) plan_segments<kPlanBM, kBN>(p.seg, p.n_seg, block_first_row(rb, kPlanBM, rs), rs, L, true, s_plan, &s_ps, tid);
    auto walk_of = [&](int sg) {
        SharedWalkF32 w;
        w.seg = sg;
        int lo, hi;
        if constexpr (PLANNED) {
            const PlanRec r = plan_uniform_load(pt + plan_seg_at(p.n_seg, rb, sg));
            const PlanRec sp = plan_uniform_load(pt + plan_span_at(n_rb, p.n_seg, rb, sg, quarter));
            w.pl.c0 = r.x, w.pl.cs = r.y, w.pl.n_tiles = r.z, w.pl.uniform = r.w;
            lo = sp.x, hi = sp.w, w.lo_max = sp.y, w.hi_min = sp.z;
        } else {
            const SegPlan l = s_plan[sg];
            w.pl.c0 = __builtin_amdgcn_readfirstlane(l.c0);
            w.pl.cs = __builtin_amdgcn_readfirstlane(l.cs);
            w.pl.n_tiles = __builtin_amdgcn_readfirstlane(l.n_tiles);
            w.pl.uniform = __builtin_amdgcn_readfirstlane(l.uniform);
            const WaveSpan sp = wave_span(make_row_win(cached_row_map<kPlanBM>(&s_ps, sg, 32 * quarter + (lane & 31)), w.pl), w.pl.uniform != 0);
            lo = __builtin_amdgcn_readfirstlane(sp.lo_min), hi = __builtin_amdgcn_readfirstlane(sp.hi_max);
            w.lo_max = __builtin_amdgcn_readfirstlane(sp.lo_max), w.hi_min = __builtin_amdgcn_readfirstlane(sp.hi_min);
        }
        hi = min(hi, w.pl.n_tiles * kBN);
        w.tile = 0, w.end = 0, w.at0 = 0, w.last = 0;
        if (lo < hi) {
            w.at0 = max(lo, 0);
            w.end = (hi - w.at0 + BN - 1) / BN;
            w.pl.c0 += w.pl.cs * w.at0;
            w.last = hi - 1 - w.at0;
            w.lo_max -= w.at0, w.hi_min -= w.at0;
        }
        return w;
    };
    auto settle = [&](SharedWalkF32& w, int over) {  // the walk `over` tiles past the beginning of segment w.seg
        for (int sg = w.seg; sg < p.n_seg; ++sg) {
            w = walk_of(sg);
            if (over < w.end) {
                w.tile = over;
                return;
            }
            over -= w.end;
        }
        w.seg = p.n_seg, w.tile = 0, w.end = 0;
    };
    SharedWalkF32 cur = walk_of(0);
    int total = cur.end;
    for (int sg = 1; sg < p.n_seg; ++sg) total += walk_of(sg).end;
    cur.tile = wave;
    if (wave >= cur.end) {
        const int over = wave - cur.end;
        cur.seg = 1;
        settle(cur, over);
    }
    auto window = [&](const SharedWalkF32& w, int rg, const PlanRec& rec) {  // of row n of the 16, in positions of w
        RowWin win;
        if constexpr (PLANNED) {
            win.lo = rec.x, win.cnt = rec.y, win.lin = rec.z;
        } else {
            SegPlan whole = w.pl;
            whole.c0 -= whole.cs * w.at0;
            win = make_row_win(cached_row_map<kPlanBM>(&s_ps, w.seg, k0 + 16 * rg + n), whole);
        }
        win.lo -= w.at0;
        return win;
    };
    PlanRec win_rec[RG];
    auto request_windows = [&](int sg) {
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
            if constexpr (PLANNED)
                win_rec[rg] = pt[plan_row_at(n_rb, p.n_seg, rb, sg, k0 + 16 * rg + n)];
            else
                win_rec[rg] = PlanRec{0, 0, 1, 0};
        }
    };
    if (cur.seg < p.n_seg) request_windows(cur.seg);

    // ---- requests of a tile, an operand of one head within 32-bit offsets ----
    auto load4 = [](const float* base, uint32_t off) { return *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(base) + off); };
    auto key_at = [&](const SharedWalkF32& w, int row) { return (uint32_t)min(max(w.pl.c0 + w.pl.cs * min(w.tile * BN + row, w.last), 0), L - 1); };
    f32x4 kr[2][2 * KS], vr[8][DT / 4];
    const uint32_t k_row = (uint32_t)p.k_sl * 4, v_row = (uint32_t)p.v_sl * 4;
    auto request_k = [&](const SharedWalkF32& w) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t key = key_at(w, 16 * u + n);
            if constexpr (KT) {
                const float* from = kb + (int64_t)(8 * g) * p.k_sd + key;
#pragma unroll
                for (int i = 0; i < 2 * KS; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) kr[u][i][e] = from[(16 * (i & ~1) + 4 * (i & 1) + e) * p.k_sd];
            } else {
                const uint32_t off = __umul24(key, k_row) + 32 * g;
#pragma unroll
                for (int i = 0; i < 2 * KS; ++i) kr[u][i] = load4(kb, off + 64 * (i & ~1) + 16 * (i & 1));
            }
        }
    };
    auto request_v = [&](const SharedWalkF32& w) {  // contraction slot 8g + e: position 4g + e of the first (e < 4) or of the second subtile
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t off = __umul24(key_at(w, 16 * (e >> 2) + 4 * g + (e & 3)), v_row) + D / 4 * n;
#pragma unroll
            for (int i = 0; i < DT / 4; ++i) vr[e][i] = load4(vb, off + 16 * i);
        }
    };
    f32x4 q_raw[RG][2 * KS];
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        const float* qr = qb + (int64_t)min(r0 + rs * (16 * rg + n), L - 1) * p.q_sl + 8 * g;
#pragma unroll
        for (int i = 0; i < 2 * KS; ++i) q_raw[rg][i] = *reinterpret_cast<const f32x4*>(qr + 16 * (i & ~1) + 4 * (i & 1));
    }
    if (cur.seg < p.n_seg) request_k(cur), request_v(cur);

    auto eight = [](const f32x4& x, const f32x4& y) { return f32x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]}; };
    f32x4 o[RG][DT];
    const float c2 = p.scale_log2e, slack = kRescaleThreshold / c2;
    float m_ref[RG], l_run[RG];
    Split3 qf[RG][KS];
    float q_most = 0.f;
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        m_ref[rg] = kNegBigA, l_run[rg] = 0.f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[rg][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const f32x8 x = eight(q_raw[rg][2 * ks], q_raw[rg][2 * ks + 1]);
            qf[rg][ks] = split3(x);
#pragma unroll
            for (int e = 0; e < 8; ++e) q_most = fmaxf(q_most, fabsf(x[e]));
        }
    }
    // What a reference takes off the scores, rounded once: parts and steps with different references meet by the differences of what was
    // taken off, which with large scores are not the rounded differences of the references.
    auto offset_of = [&](float ref) {
        float x = ref * c2;
#if defined(__HIP_DEVICE_COMPILE__)
        asm("" : "+v"(x));  // (no part of a fused operation)
#endif
        return x;
    };
    const bool beyond = out_of_split(q_most);  // something that the split operands do not hold
    RowWin win[RG];
    uint64_t pat[RG];
    int in_seg = -1;

    while (cur.seg < p.n_seg) {
        if (cur.seg != in_seg) {
            if (in_seg >= 0) request_windows(cur.seg);
#pragma unroll
            for (int rg = 0; rg < RG; ++rg) {
                win[rg] = window(cur, rg, win_rec[rg]);
                pat[rg] = ~0ull;
                if (!cur.pl.uniform) {
                    pat[rg] = 0;
                    for (int q = 0; q < 64; q += win[rg].lin) pat[rg] |= 1ull << q;
                }
            }
            in_seg = cur.seg;
        }
        const int j0 = cur.tile * BN;
        const bool full = j0 >= cur.lo_max && j0 + BN <= cur.hi_min, uniform = cur.pl.uniform != 0;
        SharedWalkF32 next = cur;
        next.tile += KG;
        if (next.tile >= next.end) {
            const int over = next.tile - next.end;
            ++next.seg;
            settle(next, over);
        }
        const bool more = next.seg < p.n_seg;

        // ---- S^T = K . Q^T, of two subtiles of 16 positions ----
        f32x4 s[RG][2];
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) s[rg][0] = s[rg][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            Split3 kf[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) kf[u] = split3(eight(kr[u][2 * ks], kr[u][2 * ks + 1]));
#pragma unroll
            for (int i = 0; i < 6; ++i)
#pragma unroll
                for (int m = 0; m < 2 * RG; ++m) mma16(s[m / 2][m % 2], kf[m % 2].p[kSplitA[i]], qf[m / 2][ks].p[kSplitB[i]]);
        }
        if (more) request_k(next);
        Split3 pf[RG];
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
            if (!full) {
                if (uniform) {
                    const int from = j0 + 4 * g - win[rg].lo;
#pragma unroll
                    for (int u = 0; u < 2; ++u)
#pragma unroll
                        for (int j = 0; j < 4; ++j) s[rg][u][j] = (unsigned)(from + 16 * u + j) < (unsigned)win[rg].cnt ? s[rg][u][j] : kNegBigA;
                } else {
                    int first = (win[rg].lo - j0) % win[rg].lin;
                    if (first < 0) first += win[rg].lin;
                    const uint32_t bits = (uint32_t)row_live_bits(win[rg], j0, first, pat[rg]) >> (4 * g);
#pragma unroll
                    for (int u = 0; u < 2; ++u)
#pragma unroll
                        for (int j = 0; j < 4; ++j) s[rg][u][j] = keep_or_mask(s[rg][u][j], ((int)((bits >> (16 * u)) << (31 - j))) >> 31);
                }
            }
            // ---- online softmax against a lazily moved reference (see attention_f32.hip) ----
            float mx = m_ref[rg];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) mx = fmaxf(mx, s[rg][u][j]);
            if (__any(mx - m_ref[rg] > slack)) {
                mx = over_groups(mx, [](float x, float y) { return fmaxf(x, y); });
                const float m_new = mx - m_ref[rg] > slack ? mx : m_ref[rg];
                const float alpha = fast_exp2(offset_of(m_ref[rg]) - offset_of(m_new));
                m_ref[rg] = m_new;
                l_run[rg] *= alpha;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) o[rg][dt] *= alpha;
            }
            const float mb = m_ref[rg] > 0.5f * kNegBigA ? offset_of(m_ref[rg]) : 0.f;
            f32x8 e8;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                e8[j] = fast_exp2(fmaf(s[rg][j >> 2][j & 3], c2, -mb));
                l_run[rg] += e8[j];
            }
            pf[rg] = split3(e8);
        }
        // ---- O^T += V^T . P^T, of two tiles of 16 columns at a time ----
#pragma unroll
        for (int d2 = 0; d2 < DT / 2; ++d2) {
            Split3 vf[2];
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                f32x8 x;
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = vr[e][(2 * d2 + y) / 4][(2 * d2 + y) % 4];
                vf[y] = split3(x);
            }
#pragma unroll
            for (int i = 0; i < 6; ++i)
#pragma unroll
                for (int m = 0; m < 2 * RG; ++m) mma16(o[m / 2][2 * d2 + m % 2], vf[m % 2].p[kSplitA[i]], pf[m / 2].p[kSplitB[i]]);
        }
        if (more) request_v(next);
        cur = next;
    }

    // ---- the parts meet ----
    const int used = total > 2 ? 4 : 2;  // parts that are read
    if (wave < used) {
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
            const float l_tot = over_groups(l_run[rg], [](float x, float y) { return x + y; });
            if (g == 0) s_ref[wave][16 * rg + n] = offset_of(m_ref[rg]), s_sum[wave][16 * rg + n] = l_tot;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < DT / 4; ++i) {
                    const f32x4 x = {o[rg][4 * i][j], o[rg][4 * i + 1][j], o[rg][4 * i + 2][j], o[rg][4 * i + 3][j]};
                    lds_store128(lds_address(smem) + (wave * ROWS + 16 * rg + n) * OROW + (4 * g + j) * (DT * 4) + 16 * i, __builtin_bit_cast(u32x4, x));
                }
        }
    }
    lds_barrier();
    constexpr int NP = ROWS * D / 4 / 256;  // pieces of 4 columns, pieces a thread
    bool again = beyond;
    f32x4 out[NP];
    float sum[NP], ref[NP];
    auto meet = [&](auto parts) __attribute__((always_inline)) {  // of wavefronts 0 .. parts - 1
        constexpr int N = decltype(parts)::value;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int f = tid + 256 * i, row = f / (D / 4), c = f % (D / 4);
            f32x4 x[N];
            float r[N], l[N];
#pragma unroll
            for (int w = 0; w < N; ++w) {
                r[w] = s_ref[w][row], l[w] = s_sum[w][row];
                x[w] = __builtin_bit_cast(f32x4, lds_load128(lds_address(smem) + (w * ROWS + row) * OROW + 16 * c));
            }
            float m = r[0];
#pragma unroll
            for (int w = 1; w < N; ++w) m = fmaxf(m, r[w]);
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            float l_all = 0.f;
#pragma unroll
            for (int w = 0; w < N; ++w) {
                const float e = fast_exp2(r[w] - m);
                l_all = fmaf(l[w], e, l_all);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = fmaf(x[w][j], e, acc[j]);
            }
            out[i] = acc, sum[i] = l_all, ref[i] = m;
            // (see attention_f32.hip: what is not finite stays so, and what is far below normal may have lost bits)
            float chk = l_all * 0.f;
            uint32_t least = ~0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float y = acc[j];
                chk = fmaf(y, 0.f, chk);
                least = min(least, (__builtin_bit_cast(uint32_t, y) << 1) - 1);
            }
            again |= chk != 0.f || least < __builtin_bit_cast(uint32_t, 0x1p-104f * l_all) << 1;
        }
    };
    if (total > 2)
        meet(std::integral_constant<int, 4>{});
    else
        meet(std::integral_constant<int, 2>{});
    if (__syncthreads_or(again ? 1 : 0)) {
        // ---- the rows once more in float32 arithmetic, position by position, each lane a quarter of a row's columns, live positions only ----
        if (wave >= RG) return;
        const int my_row = r0 + rs * (16 * wave + n);
        constexpr int QD = D / 4;
        const float* qr = qb + (int64_t)min(my_row, L - 1) * p.q_sl + g * QD;
        float q[QD], acc[QD];
#pragma unroll
        for (int i = 0; i < QD; ++i) q[i] = qr[i], acc[i] = 0.f;
        float m = -__builtin_inff(), l = 0.f;
        for (int sg = 0; sg < p.n_seg; ++sg) {
            const SharedWalkF32 w = walk_of(sg);
            PlanRec rec = {0, 0, 1, 0};
            if constexpr (PLANNED) rec = pt[plan_row_at(n_rb, p.n_seg, rb, sg, k0 + 16 * wave + n)];
            const RowWin own = window(w, wave, rec);
            for (int j = 0; j < w.end * BN; ++j) {
                const bool live = win_live(own, j);
                if (!__any(live)) continue;
                const int64_t key = min(max(w.pl.c0 + w.pl.cs * j, 0), L - 1);
                const float* from = KT ? kb + (int64_t)(g * QD) * p.k_sd + key : kb + key * p.k_sl + g * QD;
                float s = 0.f;
#pragma unroll
                for (int i = 0; i < QD; ++i) s = fmaf(q[i], from[KT ? i * p.k_sd : i], s);
                s = over_groups(s, [](float x, float y) { return x + y; }) * c2;
                if (live) {
                    const float m_new = fmaxf(m, s);
                    const float off = m_new > -__builtin_inff() ? m_new : 0.f;
                    const float alpha = m > -__builtin_inff() ? fast_exp2(m - off) : 1.f;
                    const float e = fast_exp2(s - off);
                    m = m_new;
                    l = fmaf(l, alpha, e);
                    const float* v = vb + key * p.v_sl + g * QD;
#pragma unroll
                    for (int i = 0; i < QD; ++i) acc[i] = fmaf(acc[i], alpha, e * v[i]);
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
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int f = tid + 256 * i, row = f / (D / 4), c = f % (D / 4), r = r0 + rs * row;
        if (r >= L) continue;
        const float inv = sum[i] > 0.f ? 1.0f / sum[i] : 0.f;
        *reinterpret_cast<f32x4*>(ob + (int64_t)r * p.o_sl + 4 * c) = out[i] * inv;
        if (p.lse != nullptr && c == 0)
            p.lse[(int64_t)bh * L + r] = sum[i] > 0.f ? (ref[i] + __log2f(sum[i])) * 0.6931471805599453f : __builtin_inff();
    }
}

template <int D, bool KT, bool PLANNED, int RG>
static int launch(const AttnParams& p0, hipStream_t st) {
    begin_launch();
    constexpr int PER = kPlanBM / (16 * RG);
    AttnParams p = p0;
    p.n_row_blocks = count_row_blocks(p.L, kPlanBM, p.row_stride);
    p.total = p.B * p.H * PER * p.n_row_blocks;
    p.by_blocks = divisor(PER * p.n_row_blocks), p.by_h = divisor(p.H);
    constexpr size_t lds = (size_t)4 * 16 * RG * (D * 4 + 16);
    auto kern = attn_fwd_shared_f32_kernel<D, KT, PLANNED, RG>;
    static uint64_t lds_reserved = 0;
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), lds, "splat_attention_fwd")) return rc;
    kern<<<((p.total + 7) / 8) * 8, 256, lds, st>>>(p);
    return check_launch("splat_attention_fwd");
}

template <int D, int RG>
static int launch_layout(const AttnParams& p, bool kt, hipStream_t st) {
    if (p.plan) return kt ? launch<D, true, true, RG>(p, st) : launch<D, false, true, RG>(p, st);
    return kt ? launch<D, true, false, RG>(p, st) : launch<D, false, false, RG>(p, st);
}
int launch_attn_shared_f32(const AttnParams& p, int d, bool kt, int rows, hipStream_t st) {
    if (rows == 16) return d == 64 ? launch_layout<64, 1>(p, kt, st) : launch_layout<128, 1>(p, kt, st);
    return d == 64 ? launch_layout<64, 2>(p, kt, st) : launch_layout<128, 2>(p, kt, st);
}

}  // namespace splat

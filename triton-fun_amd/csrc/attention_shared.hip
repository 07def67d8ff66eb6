// Fused ACSR sparse-attention forward for 16-bit types in launches of few rows, gfx950: the wavefronts of a workgroup share the keys.
//
// Bound: latency.  A launch that leaves most of the chip idle takes as long as one workgroup's walk over its tiles, one after the other.
// Here a workgroup is 32 rows, every one of its KG wavefronts holds all of them, and tile k of 32 positions goes to wavefront k % KG: each
// copies its tiles into LDS of its own, so that nothing but Q and the end needs a barrier, and keeps a softmax of its own.  At the end
// the parts meet in LDS, scaled to the largest of their references.  What is left is a chain that runs once, of a workgroup's 8600 cycles
// (one tile, d = 128, four wavefronts, time stamps): arguments and plan 800, requests of Q and the tile 1500 (64 bytes a cycle and CU: eight
// wavefronts take 2500), their latency 700, the tile 2200, the end 2500.  Q through LDS, because fragments that every wavefront loads for
// itself hold up the address path for 1000 cycles; the end reads the parts of two, four or all wavefronts, as many as had a tile.
// Against attention_rows16.hip, which took these launches: bf16, 4 heads of 1024 rows, windows 32 / 128 / 512: d = 64 5.7 -> 4.2 us,
// 6.6 -> 4.8, 11.2 -> 6.1; d = 128 6.7 -> 4.9, 7.9 -> 6.0, 14.4 -> 7.7; the lines are in dispatch_attn (attention.hip).
//
// Eight wavefronts at d = 64 on keys that lie anywhere have 44 bytes of scratch: two addresses of K's rows are read again each tile, beside K's
// own loads and in front of them, the rest before and after the walk.  A counted wait leaves the youngest requests open, so what stands
// between them makes it wait for more, never for less.
//
// Layouts are those of attention.hip (32x32x16, transposed products, one lane a row).  K's tile is free once the scores are
// taken and V's once the output is, so that one stage of each holds the next tile's copies while the other product runs.
#include <type_traits>

#include "attn_tile.hpp"

namespace splat {

constexpr int kSharedRows = 32;  // rows of a workgroup: a quarter of a row block of the plan
enum { kSharedKeyRows, kSharedKeysWhole, kSharedKeysAnywhere };  // how K is stored, as in attention_rows16.hip

// The walk of a workgroup's own 32 rows over one segment, in tiles of 32 positions.  It starts `at0` positions into the row block's.
struct SharedWalk {
    int seg, tile, end, at0;
    int last;            // the last position that one of the rows sees
    int lo_max, hi_min;  // positions between them are live for every row
    SegPlan pl;
};

template <typename T, int D, int LAYOUT, bool PLANNED, int KG>
__global__ __launch_bounds__(64 * KG, D == 64 ? (KG == 8 ? 4 : 3) : 2) void attn_fwd_shared_kernel(const AttnParams p) {
    constexpr bool KT = LAYOUT != kSharedKeyRows, ANY = LAYOUT == kSharedKeysAnywhere;
    constexpr int ES = 2, BN = 32;
    static_assert(sizeof(T) == ES && kPlanBM == 4 * kSharedRows, "tile shape");
    constexpr int KS = D / 16, DT = D / 32;
    constexpr int V_ROWB = D * ES, K_ROWB = KT ? BN * ES : D * ES;
    constexpr int TILE = BN * D * ES;
    constexpr int NI = TILE / 1024;  // copy blocks of an operand's tile
    constexpr int V_CPR = V_ROWB / 16, K_CPR = K_ROWB / 16, K_RPI = 1024 / K_ROWB;

    extern __shared__ __attribute__((aligned(1024))) char smem[];  // per wavefront: a tile of K, a tile of V; then Q
    __shared__ SegPlan s_plan[SPLAT_MAX_SEGMENTS];
    __shared__ PlanScratch<kPlanBM> s_ps;
    __shared__ float s_ref[KG][kSharedRows], s_sum[KG][kSharedRows];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 31, g = lane >> 5;

    load_args(p.total, p.n_row_blocks, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.H, p.row_stride, p.L, p.n_seg, p.plan, p.scale_log2e,
              p.q, p.q_sb, p.q_sh, p.q_sl, p.k, p.k_sb, p.k_sh, p.k_sd, p.k_sl, p.v, p.v_sb, p.v_sh, p.v_sl);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int per_head = 4 * p.n_row_blocks;
    const int bh = quotient(logical, p.by_blocks), b = quotient(bh, p.by_h);
    const int at = per_head - 1 - (logical - bh * per_head), h = bh - b * p.H;
    const int rb = at >> 2, quarter = at & 3;
    const int rs = p.row_stride, L = p.L;
    const int k0 = quarter * kSharedRows;
    const int r0 = block_first_row(rb, kPlanBM, rs) + rs * k0;
    if (r0 >= L) return;

    const T* qb = (const T*)p.q + b * p.q_sb + h * p.q_sh;
    const T* kb = (const T*)p.k + b * p.k_sb + h * p.k_sh;
    const T* vb = (const T*)p.v + b * p.v_sb + h * p.v_sh;

    // ---- plan: the row block's walk, cut down to what this quarter of it sees ----
    const PlanRec* const pt = p.plan;
    const int n_rb = p.n_row_blocks;
    if constexpr (!PLANNED) plan_segments<kPlanBM, kBN>(p.seg, p.n_seg, block_first_row(rb, kPlanBM, rs), rs, L, !KT, s_plan, &s_ps, tid);
    auto walk_of = [&](int sg) {
        SharedWalk w;
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
            const WaveSpan sp = wave_span(make_row_win(cached_row_map<kPlanBM>(&s_ps, sg, k0 + lm), w.pl), w.pl.uniform != 0);
            lo = __builtin_amdgcn_readfirstlane(sp.lo_min), hi = __builtin_amdgcn_readfirstlane(sp.hi_max);
            w.lo_max = __builtin_amdgcn_readfirstlane(sp.lo_max), w.hi_min = __builtin_amdgcn_readfirstlane(sp.hi_min);
        }
        hi = min(hi, w.pl.n_tiles * kBN);
        w.tile = 0, w.end = 0, w.at0 = 0, w.last = 0;
        if (lo < hi) {
            w.at0 = max(lo, 0) & (w.pl.cs == 1 ? ~7 : ~0);  // (K^T is copied in pieces of 8 keys)
            w.end = (hi - w.at0 + BN - 1) / BN;
            w.pl.c0 += w.pl.cs * w.at0;
            w.last = hi - 1 - w.at0;
            w.lo_max -= w.at0, w.hi_min -= w.at0;
        }
        return w;
    };
    // the walk at `over` tiles past the beginning of segment w.seg
    auto settle = [&](SharedWalk& w, int over) {
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
    auto advance = [&](SharedWalk& w) {
        w.tile += KG;
        if (w.tile >= w.end) {
            const int over = w.tile - w.end;
            ++w.seg;
            settle(w, over);
        }
    };
    SharedWalk cur = walk_of(0);
    int total = cur.end;
    for (int sg = 1; sg < p.n_seg; ++sg) total += walk_of(sg).end;
    cur.tile = wave;
    if (wave >= cur.end) {
        const int over = wave - cur.end;
        cur.seg = 1;
        settle(cur, over);
    }

    // ---- copies of this wavefront's tiles ----
    char* const k_lds = smem + wave * 2 * TILE;
    char* const v_lds = k_lds + TILE;
    const uint32_t v_row = (uint32_t)p.v_sl * ES, k_row = (uint32_t)p.k_sl * ES;  // (an operand of one head lies within 32-bit offsets)
    // Rows of the tile's positions, NI blocks of 1 KiB.  What lies past the last position that one of the rows sees comes from that
    // position once more: it meets probabilities of zero, which only leave finite values out.
    auto copy_rows = [&](auto cpr, auto swz_mode, const SharedWalk& w, const T* base, uint32_t row_bytes, char* lds) {
        constexpr int CPR = decltype(cpr)::value, RPI = 64 / CPR;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int row = RPI * i + lane / CPR, c = logical_chunk<CPR * 16, decltype(swz_mode)::value>(row, lane % CPR) * 16;
            const int key = min(max(w.pl.c0 + w.pl.cs * min(w.tile * BN + row, w.last), 0), L - 1);
            dma16_uniform(base, __umul24(key, row_bytes) + c, lds + i * 1024);
        }
    };
    u32x4 k_reg[ANY ? NI : 1];
    auto fetch_k = [&](const SharedWalk& w) {
        const int c0 = w.pl.c0 + w.tile * BN;
        if constexpr (ANY) {
#pragma unroll
            for (int i = 0; i < NI; ++i)
                k_reg[i] = keys_piece(kb + (int64_t)(K_RPI * i + lane / K_CPR) * p.k_sd, c0 + 8 * (lane % K_CPR), L);
        } else if constexpr (KT) {
            // rows = d, 32 consecutive keys each (dense walk); a piece past the last key is replaced by the last whole one
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int row = K_RPI * i + lane / K_CPR, c = min(c0 + 8 * (lane % K_CPR), L - 8);
                dma16(kb + (int64_t)row * p.k_sd + c, k_lds + i * 1024);
            }
        } else {
            copy_rows(std::integral_constant<int, K_CPR>{}, std::integral_constant<int, 1>{}, w, kb, k_row, k_lds);
        }
    };
    auto fetch_v = [&](const SharedWalk& w) {
        copy_rows(std::integral_constant<int, V_CPR>{}, std::integral_constant<int, 2>{}, w, vb, v_row, v_lds);
    };

    // the row windows of the first segment, Q, then the first tile
    PlanRec win_rec = {0, 0, 1, 0};
    if constexpr (PLANNED) {
        if (cur.seg < p.n_seg) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + lm)];
    }
    char* const q_lds = smem + KG * 2 * TILE;
#pragma unroll
    for (int i = 0; i < (NI + KG - 1) / KG; ++i) {
        const int blk = wave + KG * i, row = 64 / V_CPR * blk + lane / V_CPR;
        if (NI % KG == 0 || blk < NI)
            dma16(qb + (int64_t)min(r0 + rs * row, L - 1) * p.q_sl + logical_chunk<V_ROWB, 1>(row, lane % V_CPR) * 8, q_lds + blk * 1024);
    }
    if (cur.seg < p.n_seg) fetch_k(cur), fetch_v(cur);

    // ---- LDS read addresses ----
    const int tr_row = (lane & 15) >> 2, tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    uint32_t k_addr[KT ? 1 : KS], v_addr[DT];
    if constexpr (KT) {
        k_addr[0] = lds_address(k_lds) + (8 * g + tr_row) * K_ROWB + tr_col * ES;
    } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) k_addr[ks] = lds_address(k_lds) + lds_off<K_ROWB, true>(lm, (16 * ks + 8 * g) * ES);
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        v_addr[dt] = lds_address(v_lds) + (4 * g + tr_row) * V_ROWB + ((dt ^ swz64<V_ROWB>(4 * g + tr_row)) * 64) + tr_col * ES;

    f32x16 o_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 16; ++j) o_acc[dt][j] = 0.f;
    float m_ref = kNegBigA, l_run = 0.f;
    const float c2 = p.scale_log2e;
    RowWin win = {0, 0, 1};
    uint64_t pat = ~0ull;
    int in_seg = -1;
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) asm volatile("" : "+v"(o_acc[dt]));  // set while the copies are on their way
#endif
    // Q's copies were issued before those of K and V
    if (cur.seg < p.n_seg)
        wait_loads<2 * NI>();
    else
        wait_loads<0>();
    __builtin_amdgcn_s_barrier();
    Frag<T> qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
        qf[ks].v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128(lds_address(q_lds) + lds_off<V_ROWB, true>(lm, (16 * ks + 8 * g) * ES)));

    while (cur.seg < p.n_seg) {
        if (cur.seg != in_seg) {
            if constexpr (PLANNED) {
                if (in_seg >= 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + lm)];
                win.lo = win_rec.x, win.cnt = win_rec.y, win.lin = win_rec.z;
            } else {
                SegPlan whole = cur.pl;  // (a window is relative to the row block's walk)
                whole.c0 -= whole.cs * cur.at0;
                win = make_row_win(cached_row_map<kPlanBM>(&s_ps, cur.seg, k0 + lm), whole);
            }
            win.lo -= cur.at0;
            pat = ~0ull;
            if (!cur.pl.uniform) {
                pat = 0;
                for (int q = 0; q < 64; q += win.lin) pat |= 1ull << q;
            }
            in_seg = cur.seg;
        }
        const int j0 = cur.tile * BN;
        const bool full = j0 >= cur.lo_max && j0 + BN <= cur.hi_min;
        const bool uniform = cur.pl.uniform != 0;
        SharedWalk next = cur;
        advance(next);
        const bool more = next.seg < p.n_seg;

        // ---- S^T = K . Q^T ----
        if constexpr (ANY) {
#pragma unroll
            for (int i = 0; i < NI; ++i) lds_store128(lds_address(k_lds) + i * 1024 + lane * 16, k_reg[i]);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        } else {
            wait_loads<NI>();  // K has landed; V's copies were issued after it
        }
        f32x16 s[1];
#pragma unroll
        for (int j = 0; j < 16; ++j) s[0][j] = 0.f;
        Frag<T> kf[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            if constexpr (KT) {
                const uint32_t a0 = k_addr[0] + 16 * ks * K_ROWB;
                kf[ks] = frag_from_tr<T>(lds_load_tr16(a0), lds_load_tr16(a0 + 4 * K_ROWB));
            } else {
                kf[ks].v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128(k_addr[ks]));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) mma32(s[0], kf[ks], qf[ks]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // K's tile is read
        if (more) fetch_k(next);
        if (!full) {
            int first = 0;
            if (!uniform) {
                first = (win.lo - j0) % win.lin;
                if (first < 0) first += win.lin;
            }
            mask_half(s[0], (uint32_t)row_live_bits(win, j0, first, pat) >> (4 * g));
        }
        Frag<T> pf[1][2];
        softmax_tile<1, T, DT>(s, pf, m_ref, l_run, o_acc, c2);

        // ---- O^T += V^T . P^T ----
        if (more)
            wait_loads<NI>();  // V has landed; the next K's copies were issued after it
        else
            wait_loads<0>();
        Frag<T> vf[2][DT];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const uint32_t a0 = v_addr[dt] + 16 * t * V_ROWB;
                vf[t][dt] = frag_from_tr<T>(lds_load_tr16(a0), lds_load_tr16(a0 + 8 * V_ROWB));
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) mma32(o_acc[dt], vf[t][dt], pf[0][t]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // V's tile is read
        if (more) fetch_v(next);
        cur = next;
    }

    // ---- the parts meet: each wavefront leaves its O (float32, 32 rows of D) in its own tiles, 16-byte chunks swizzled by row ----
    {
        constexpr int OCH = D / 4;  // chunks of a row
        if (wave < max(total, KG > 4 && total > 4 ? KG : total > 2 ? 4 : 2)) {  // (what is read below)
            const float l_tot = with_lane_xor<32, 64>(l_run, [](float x, float y) { return x + y; });
            if (g == 0) s_ref[wave][lm] = m_ref, s_sum[wave][lm] = l_tot;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    const f32x4v x = {o_acc[dt][4 * jj], o_acc[dt][4 * jj + 1], o_acc[dt][4 * jj + 2], o_acc[dt][4 * jj + 3]};
                    const int c = (8 * dt + 2 * jj + g) ^ (lm & (OCH - 1));
                    lds_store128(lds_address(k_lds) + lm * (D * 4) + c * 16, __builtin_bit_cast(u32x4, x));
                }
        }
        lds_barrier();
        constexpr int PCS = 32 * D / 8, NP = (PCS + 64 * KG - 1) / (64 * KG);  // pieces of 8 columns, pieces a thread
        auto meet = [&](auto parts) __attribute__((always_inline)) {  // of wavefronts 0 .. parts - 1
            constexpr int N = decltype(parts)::value;
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int f = tid + 64 * KG * i, row = f / (D / 8), c = f % (D / 8), r = r0 + rs * row;
                if (PCS % (64 * KG) != 0 && f >= PCS) break;
                f32x4v x[N][2];
                float ref[N], sum[N];
#pragma unroll
                for (int w = 0; w < N; ++w) {
                    ref[w] = s_ref[w][row], sum[w] = s_sum[w][row];
#pragma unroll
                    for (int k = 0; k < 2; ++k)
                        x[w][k] = __builtin_bit_cast(f32x4v, lds_load128(lds_address(smem) + w * 2 * TILE + row * (D * 4) + (((2 * c + k) ^ (row & (OCH - 1))) * 16)));
                }
                float m = ref[0], l = sum[0];
                if constexpr (N > 1) {
#pragma unroll
                    for (int w = 1; w < N; ++w) m = fmaxf(m, ref[w]);
                    l = 0.f;
#pragma unroll
                    for (int w = 0; w < N; ++w) {
                        const float e = fast_exp2((ref[w] - m) * c2);
                        l = fmaf(sum[w], e, l);
#pragma unroll
                        for (int k = 0; k < 2; ++k)
#pragma unroll
                            for (int j = 0; j < 4; ++j) x[0][k][j] = w == 0 ? x[0][k][j] * e : fmaf(x[w][k][j], e, x[0][k][j]);
                    }
                }
                const float inv = l > 0.f ? 1.0f / l : 0.f;
                if (r < L) {
                    Frag<T> y;
#pragma unroll
                    for (int j = 0; j < 8; ++j) y.v[j] = (T)(x[0][j >> 2][j & 3] * inv);
                    T* const to = (T*)p.o + b * p.o_sb + h * p.o_sh + (int64_t)r * p.o_sl + 8 * c;
                    *reinterpret_cast<u32x4*>(to) = __builtin_bit_cast(u32x4, y.v);
                    if (p.lse != nullptr && c == 0) p.lse[(int64_t)bh * L + r] = l > 0.f ? (m * c2 + __log2f(l)) * 0.6931471805599453f : __builtin_inff();
                }
            }
        };
        if (total >= 5 && KG > 4)
            meet(std::integral_constant<int, KG>{});
        else if (total >= 3)
            meet(std::integral_constant<int, 4>{});
        else
            meet(std::integral_constant<int, 2>{});
    }
}

template <typename T, int D, int LAYOUT, bool PLANNED, int KG>
static int launch(const AttnParams& p0, hipStream_t st) {
    begin_launch();
    AttnParams p = p0;
    p.n_row_blocks = count_row_blocks(p.L, kPlanBM, p.row_stride);
    p.total = p.B * p.H * 4 * p.n_row_blocks;
    p.by_blocks = divisor(4 * p.n_row_blocks), p.by_h = divisor(p.H);
    if (PLANNED && LAYOUT != kSharedKeyRows) p.plan += plan_variant_recs(p.n_row_blocks, p.n_seg);  // the dense-walk variant
    constexpr size_t lds = (size_t)(KG * 2 + 1) * 32 * D * 2;
    auto kern = attn_fwd_shared_kernel<T, D, LAYOUT, PLANNED, KG>;
    static uint64_t lds_reserved = 0;
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), lds, "splat_attention_fwd")) return rc;
    kern<<<((p.total + 7) / 8) * 8, 64 * KG, lds, st>>>(p);
    return check_launch("splat_attention_fwd");
}

template <typename T, int D, int KG>
static int launch_layout(const AttnParams& p, bool kt, hipStream_t st) {
    if (p.keys_anywhere) return launch<T, D, kSharedKeysAnywhere, true, KG>(p, st);
    if (p.plan) return kt ? launch<T, D, kSharedKeysWhole, true, KG>(p, st) : launch<T, D, kSharedKeyRows, true, KG>(p, st);
    return kt ? launch<T, D, kSharedKeysWhole, false, KG>(p, st) : launch<T, D, kSharedKeyRows, false, KG>(p, st);
}
template <typename T>
int launch_attn_shared(const AttnParams& p, int d, bool kt, int waves, hipStream_t st) {
    if (waves == 8) return d == 64 ? launch_layout<T, 64, 8>(p, kt, st) : launch_layout<T, 128, 8>(p, kt, st);
    return d == 64 ? launch_layout<T, 64, 4>(p, kt, st) : launch_layout<T, 128, 4>(p, kt, st);
}
template int launch_attn_shared<f16>(const AttnParams&, int, bool, int, hipStream_t);
template int launch_attn_shared<bf16>(const AttnParams&, int, bool, int, hipStream_t);

}  // namespace splat

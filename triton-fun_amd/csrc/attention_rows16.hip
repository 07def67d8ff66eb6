// Fused ACSR sparse-attention forward for 16-bit types in launches of too many row blocks for attention_shared.hip that still leave the
// chip part idle, gfx950.
//
// Bound: latency.  A launch of the kernel in attention.hip (128 rows a workgroup, 32 a wavefront, tiles of 64 keys one ahead)
// that does not fill the chip takes as long as one of its workgroups: the chain kernel arguments -> plan -> first tile, then
// every tile's copy and its barrier one after the other, with most SIMDs of a CU idle.  Here a workgroup is 64 rows and a
// wavefront 16 of them, so that the same launch spreads over twice the workgroups and each walks fewer tiles, and pairs of
// subtiles of 16 keys outside a wavefront's rows are skipped.  16x16x32 matrix instructions run at the rate of the 32x32x16 ones,
// but every operand read from LDS then serves 16 rows instead of 32: in launches that fill the chip the LDS becomes the bound
// and the other kernel is the faster one unless much of the walk is masked (dispatch_attn in attention.hip has the lines).  Measured, bf16, 16 heads of 1024 rows,
// that kernel -> this one: d = 64, window 32: 8.3 -> 6.5 us, 128: 9.2 -> 7.3, 512: 14.6 -> 11.9; d = 128: 9.8 -> 7.5, 10.9 -> 9.0,
// 18.1 -> 15.6 (rings of three stages and tiles of 32 keys: equal at d = 64, up to 12 % slower at d = 128).
//
// Layouts: S^T (16 keys x 16 rows) = K . Q^T leaves lane (n, g) with keys 4g .. 4g + 3 of query n.  Two subtiles side by side are
// the B operand of O^T += V^T . P^T as they stand, when contraction slot 8g + e stands for key 4g + e of the first (e < 4) or of
// the second subtile; V^T comes from the row-major V tile through the transposing LDS read in that order of keys.
#include "rows16.hpp"

namespace splat {

// How K is stored: rows of keys, or K^T with the keys contiguous, whose rows are whole 16-byte pieces or start anywhere.  The last
// cannot take the asynchronous copies, which move aligned words: its pieces come through registers, a tile ahead, instead of a launch
// that turns K first.  bf16, K^T of 12 heads of 1037 keys, window 201, turned first -> read where it lies: d = 128 15.9 -> 12.1 us (rows
// of K 11.4; three workgroups' worth of registers would spill 19 of them: 13.0), d = 64 11.8 -> 9.2; 11 heads of 2041, window 101
// 16.1 -> 12.5 and 12.1 -> 8.4.
enum { kKeyRows, kKeysWhole, kKeysAnywhere };

template <typename T, int D, int LAYOUT, bool PLANNED>
__global__ __launch_bounds__(256, LAYOUT == kKeysAnywhere && D == 128 ? 2 : 3) void attn_fwd_rows16_kernel(const AttnParams p) {
    constexpr bool KT = LAYOUT != kKeyRows, ANY = LAYOUT == kKeysAnywhere;
    constexpr int ES = 2, BN = 64, SUB = BN / 16;
    static_assert(sizeof(T) == ES && kPlanBM == 2 * kHalfRows && kBN % BN == 0, "tile shape");
    constexpr int KS = D / 32;  // contraction steps of the score product
    constexpr int DT = D / 16;  // 16-row tiles of O^T
    constexpr int V_ROWB = D * ES, K_ROWB = KT ? BN * ES : D * ES;
    constexpr int TILE = BN * D * ES, STAGE = 2 * TILE;
    constexpr int NI = TILE / 4096;  // copy blocks per wavefront and operand
    constexpr int K_SWZ = KT ? 4 : 1, V_SWZ = 4;
    constexpr int V_CPR = V_ROWB / 16, V_RPI = 1024 / V_ROWB, K_CPR = K_ROWB / 16, K_RPI = 1024 / K_ROWB;

    extern __shared__ __attribute__((aligned(1024))) char smem[];
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
    const int at = per_head - 1 - (logical - bh * per_head);
    const int rb = at >> 1, half = at & 1;
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride, L = p.L;
    const int k0 = half * kHalfRows;
    const int r0 = block_first_row(rb, kPlanBM, rs) + rs * k0;
    if (r0 >= L) return;

    const T* qb = (const T*)p.q + b * p.q_sb + h * p.q_sh;
    const T* kb = (const T*)p.k + b * p.k_sb + h * p.k_sh;
    const T* vb = (const T*)p.v + b * p.v_sb + h * p.v_sh;
    T* ob = (T*)p.o + b * p.o_sb + h * p.o_sh;
    const int my_row = r0 + rs * (wave * 16 + n);

    // ---- the lane's share of its Q row, resident: B operand of the score product ----
    Frag<T> qf[KS];
    {
        const T* qr = qb + (int64_t)min(my_row, L - 1) * p.q_sl;
#pragma unroll
        for (int s = 0; s < KS; ++s) qf[s] = global_frag<T>(qr + 32 * s + 8 * g);
    }

    // ---- plan: the row block's walk, cut down to the tiles that this half of it sees ----
    const PlanRec* const pt = p.plan;
    const int n_rb = p.n_row_blocks;
    if constexpr (!PLANNED) plan_segments<kPlanBM, kBN>(p.seg, p.n_seg, block_first_row(rb, kPlanBM, rs), rs, L, !KT, s_plan, &s_ps, tid);
    auto walk_of = [&](int sg) {
        HalfWalk w;
        w.seg = sg;
        if constexpr (PLANNED) {
            w = half_walk<BN>(pt, n_rb, p.n_seg, rb, half, sg);
        } else {
            const SegPlan l = s_plan[sg];
            w.pl.c0 = __builtin_amdgcn_readfirstlane(l.c0);
            w.pl.cs = __builtin_amdgcn_readfirstlane(l.cs);
            w.pl.n_tiles = __builtin_amdgcn_readfirstlane(l.n_tiles);
            w.pl.uniform = __builtin_amdgcn_readfirstlane(l.uniform);
            w.tile = 0, w.end = w.pl.n_tiles * (kBN / BN);
        }
        return w;
    };
    auto next_segment = [&](HalfWalk& w) {  // the first segment from w.seg on that has tiles
        for (int sg = w.seg; sg < p.n_seg; ++sg) {
            w = walk_of(sg);
            if (w.end > w.tile) return;
        }
        w.seg = p.n_seg, w.tile = 0, w.end = 0x7fffffff;
    };
    int total = 0;
    for (int sg = 0; sg < p.n_seg; ++sg) {
        const HalfWalk w = walk_of(sg);
        total += w.end - w.tile;
    }
    total = __builtin_amdgcn_readfirstlane(total);

    // ---- asynchronous copies of one tile (1 KiB blocks, wavefront w issues blocks w, w + 4, ...): from running wavefront-uniform
    // pointers and per-lane offsets where every position of the tile exists, else with an address per lane.  The swizzles do
    // not depend on the block, so one offset serves all blocks of an operand ----
    auto issue_general = [&](const HalfWalk& w, int stage) {
        const int j0 = w.tile * BN;
        char* ks_w = smem + stage * STAGE;
        auto key_row = [&](int row) { return min(max(w.pl.c0 + w.pl.cs * (j0 + row), 0), L - 1); };
        dma_tile<T, V_ROWB, BN, V_SWZ>(ks_w + TILE, wave, lane, [&](int row) { return vb + (int64_t)key_row(row) * p.v_sl; });
        if constexpr (ANY) {
        } else if constexpr (KT) {
            // rows = d, BN consecutive keys each (dense walk); a chunk past the last key is replaced by the last whole one
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int blk = wave + 4 * i, flat = blk * 64 + lane;
                const int row = flat / K_CPR;
                const int c = min(w.pl.c0 + j0 + logical_chunk<K_ROWB, K_SWZ>(row, flat % K_CPR) * 8, L - 8);
                dma16(kb + (int64_t)row * p.k_sd + c, ks_w + blk * 1024);
            }
        } else {
            dma_tile<T, K_ROWB, BN, K_SWZ>(ks_w, wave, lane, [&](int row) { return kb + (int64_t)key_row(row) * p.k_sl; });
        }
    };
    uint32_t v_off = 0, k_off = 0;
    const char *v_next = nullptr, *k_next = nullptr;
    int64_t v_row = 0, k_row = 0;  // bytes from one tile row to the next
    bool off_fits = true;          // the copy instruction takes a 32-bit offset
    auto set_offsets = [&](const HalfWalk& w) {
        v_row = (int64_t)p.v_sl * ES * w.pl.cs;
        k_row = KT ? (int64_t)p.k_sd * ES : (int64_t)p.k_sl * ES * w.pl.cs;
        off_fits = v_row * V_RPI < ((int64_t)1 << 31) && k_row * K_RPI < ((int64_t)1 << 31);
        v_off = (uint32_t)(v_row * (lane / V_CPR)) + logical_chunk<V_ROWB, V_SWZ>(wave * V_RPI + lane / V_CPR, lane % V_CPR) * 16;
        k_off = (uint32_t)(k_row * (lane / K_CPR)) + logical_chunk<K_ROWB, K_SWZ>(wave * K_RPI + lane / K_CPR, lane % K_CPR) * 16;
        const int64_t first = w.pl.c0 + (int64_t)w.pl.cs * BN * w.tile;
        v_next = reinterpret_cast<const char*>(vb) + first * p.v_sl * ES + wave * V_RPI * v_row;
        k_next = reinterpret_cast<const char*>(kb) + (KT ? first * ES : first * p.k_sl * ES) + wave * K_RPI * k_row;
    };
    // K^T whose rows start anywhere comes through registers: requested with V's copies, written to the stage a tile later
    u32x4 k_reg[ANY ? NI : 1];
    auto load_keys = [&](const HalfWalk& w) {
        const int c0 = w.pl.c0 + w.tile * BN;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int flat = tid + 256 * i;
            k_reg[i] = keys_piece(kb + (int64_t)(flat / K_CPR) * p.k_sd, c0 + 8 * (flat % K_CPR), L);
        }
    };
    auto store_keys = [&](int stage) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int flat = tid + 256 * i, row = flat / K_CPR, c = flat % K_CPR;
            const int to = (((c >> 1) ^ swz32<K_ROWB>(row)) << 1) | (c & 1);
            lds_store128(lds_address(smem) + stage * STAGE + row * K_ROWB + to * 16, k_reg[i]);
        }
    };
    auto issue_next = [&](HalfWalk& w, int stage) {
        if constexpr (ANY) load_keys(w);
        const int last = w.pl.c0 + w.pl.cs * (w.tile * BN + BN - 1);
        if (off_fits && last < L && w.pl.c0 + w.pl.cs * w.tile * BN >= 0) {
            char* ks_w = smem + stage * STAGE;
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                if constexpr (!ANY) dma16_uniform(k_next + 4 * i * K_RPI * k_row, k_off, ks_w + (wave + 4 * i) * 1024);
                dma16_uniform(v_next + 4 * i * V_RPI * v_row, v_off, ks_w + TILE + (wave + 4 * i) * 1024);
            }
        } else {
            issue_general(w, stage);
        }
        v_next += BN * v_row;
        k_next += KT ? (int64_t)(BN * ES) : BN * k_row;
        if (++w.tile >= w.end) {
            ++w.seg;
            next_segment(w);
            if (w.seg < p.n_seg) set_offsets(w);
        }
    };

    // ---- LDS read addresses: of stage 0, moved on once a tile ----
    const uint32_t smem_base = lds_address(smem);
    const int tr_row = (lane & 15) >> 2, tr_byte = 8 * (lane & 3);  // transposing reads: lane s of a group reads row s / 4
    uint32_t k_addr[KT ? SUB : KS], v_addr[DT];
    if constexpr (KT) {
#pragma unroll
        for (int u = 0; u < SUB; ++u) k_addr[u] = smem_base + (8 * g + tr_row) * K_ROWB + (u ^ swz32<K_ROWB>(8 * g + tr_row)) * 32 + tr_byte;
    } else {
#pragma unroll
        for (int s = 0; s < KS; ++s) k_addr[s] = smem_base + lds_off<K_ROWB, true>(n, (32 * s + 8 * g) * ES);
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        v_addr[dt] = smem_base + TILE + (4 * g + tr_row) * V_ROWB + (dt ^ swz32<V_ROWB>(4 * g + tr_row)) * 32 + tr_byte;

    HalfWalk fetch, cur;
    fetch.seg = 0;
    next_segment(fetch);
    if (fetch.seg < p.n_seg) set_offsets(fetch);
    cur = fetch;
    PlanRec win_rec = {0, 0, 1, 0};
    if constexpr (PLANNED) {
        if (cur.seg < p.n_seg) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + wave * 16 + n)];
    }
    if (total > 0) issue_next(fetch, 0);

    f32x4v o[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i) o[i] = f32x4v{0.f, 0.f, 0.f, 0.f};
    float m_ref = kNegBigA, l_run = 0.f;
    const float c2 = p.scale_log2e;
    RowState rows;
    bool entered = false;
    int stage = 0;
#if defined(__HIP_DEVICE_COMPILE__)
    // Q is in its registers before the loop, so that no wait of the compiler's for it holds up the copies in flight there
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" ::"v"(qf[s].v));
#endif

    for (int it = 0; it < total; ++it) {
        if (!entered) {
            RowWin w;
            int phase;
            if constexpr (PLANNED) {
                if (it > 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + wave * 16 + n)];
                w.lo = win_rec.x, w.cnt = win_rec.y, w.lin = win_rec.z, phase = win_rec.w;
            } else {
                w = make_row_win(cached_row_map<kPlanBM>(&s_ps, cur.seg, k0 + wave * 16 + n), cur.pl);
                phase = cur.pl.uniform ? 0 : win_phase(w);
            }
            rows.template enter<BN>(w, phase, cur.pl.uniform != 0, cur.tile);
            entered = true;
        }
        const int j0 = cur.tile * BN;

        // this wavefront's copies of tile `it` have landed; after the barrier everybody's have, and everybody is done with
        // tile it - 1, whose stage the next fetch overwrites
        wait_loads<0>();
        if constexpr (ANY) {
            store_keys(stage);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        __builtin_amdgcn_s_barrier();
        if (it + 1 < total) issue_next(fetch, stage ^ 1);

        if (j0 + BN > rows.lo_min && j0 < rows.hi_max) {
            const bool full = j0 >= rows.lo_max && j0 + BN <= rows.hi_min;
            // pairs of subtiles that some row of the wavefront has entries in
            auto pair_live = [&](int u) { return j0 + 32 * u + 32 > rows.lo_min && j0 + 32 * u < rows.hi_max; };
            f32x4 s[SUB];
#pragma unroll
            for (int pr = 0; pr < SUB / 2; ++pr) {
                Frag<T> kf[2][KS];
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks) {
                        if constexpr (KT) {
                            const uint32_t a0 = k_addr[2 * pr + u] + 32 * ks * K_ROWB;
                            kf[u][ks] = frag_from_tr<T>(lds_load_tr16(a0), lds_load_tr16(a0 + 4 * K_ROWB));
                        } else {
                            kf[u][ks].v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128(k_addr[ks] + 16 * (2 * pr + u) * K_ROWB));
                        }
                    }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < 2; ++u) s[2 * pr + u] = pair_live(pr) ? f32x4{0.f, 0.f, 0.f, 0.f} : f32x4{kNegBigA, kNegBigA, kNegBigA, kNegBigA};
                if (!pair_live(pr)) continue;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                    for (int u = 0; u < 2; ++u) mma16(s[2 * pr + u], kf[u][ks], qf[ks]);
            }
            Frag<T> vf[DT];
            auto load_v = [&](int pr) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
                    vf[dt] = frag_from_tr<T>(lds_load_tr16(v_addr[dt] + 32 * pr * V_ROWB), lds_load_tr16(v_addr[dt] + (32 * pr + 16) * V_ROWB));
            };
            load_v(0);
            __builtin_amdgcn_sched_barrier(0);
            if (!full) rows.mask_tile(s, j0, g, cur.pl.uniform != 0);
            // ---- online softmax against a lazily moved reference (see attention.hip) ----
            float mx = s[0][0];
#pragma unroll
            for (int u = 0; u < SUB; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) mx = fmaxf(mx, s[u][j]);
            mx = over_groups(mx, [](float x, float y) { return fmaxf(x, y); });
            if (__any((mx - m_ref) * c2 > kRescaleThreshold)) {
                const float m_new = ((mx - m_ref) * c2 > kRescaleThreshold) ? mx : m_ref;
                const float alpha = fast_exp2((m_ref - m_new) * c2);
                m_ref = m_new;
                l_run *= alpha;
#pragma unroll
                for (int i = 0; i < DT; ++i) o[i] *= alpha;
            }
            // a row that has seen no live score keeps offset 0, so that its (all masked) entries map to 0
            const float mb = m_ref > 0.5f * kNegBigA ? m_ref * c2 : 0.f;
#pragma unroll
            for (int pr = 0; pr < SUB / 2; ++pr) {
                if (pr > 0) {
                    load_v(pr);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (!pair_live(pr)) continue;
                Frag<T> pf;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x = fast_exp2(fmaf(s[2 * pr + (e >> 2)][e & 3], c2, -mb));
                    l_run += x;
                    pf.v[e] = (T)x;
                }
                // ---- O^T += V^T . P^T ----
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) mma16(o[dt], vf[dt], pf);
            }
        }
        if (!cur.pl.uniform) rows.next_tile();
        stage ^= 1;
        const int delta = stage == 0 ? -STAGE : STAGE;
#pragma unroll
        for (int i = 0; i < (KT ? SUB : KS); ++i) k_addr[i] += delta;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) v_addr[dt] += delta;
        if (++cur.tile >= cur.end) {
            ++cur.seg;
            next_segment(cur);
            entered = false;
        }
    }

    // ---- epilogue: a lane holds columns 16 dt + 4g .. + 3 of its row ----
    const float l_tot = over_groups(l_run, [](float x, float y) { return x + y; });
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    if (my_row < L) {
        if (p.lse != nullptr && g == 0)
            p.lse[(int64_t)bh * L + my_row] = l_tot > 0.f ? (m_ref * c2 + __log2f(l_tot)) * 0.6931471805599453f : __builtin_inff();
        T* orow = ob + (int64_t)my_row * p.o_sl;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            typedef T vec4 __attribute__((ext_vector_type(4)));
            vec4 x;
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = (T)(o[dt][i] * inv);
            *reinterpret_cast<vec4*>(orow + 16 * dt + 4 * g) = x;
        }
    }
}

template <typename T, int D, int LAYOUT, bool PLANNED>
static int launch(const AttnParams& p0, hipStream_t st) {
    begin_launch();
    AttnParams p = p0;
    p.n_row_blocks = count_row_blocks(p.L, kPlanBM, p.row_stride);
    p.total = p.B * p.H * 2 * p.n_row_blocks;
    p.by_blocks = divisor(2 * p.n_row_blocks), p.by_h = divisor(p.H);
    if (PLANNED && LAYOUT != kKeyRows) p.plan += plan_variant_recs(p.n_row_blocks, p.n_seg);  // the dense-walk variant
    constexpr size_t lds = 2 * 2 * 64 * D * 2;  // two stages of two tiles of 64 positions
    auto kern = attn_fwd_rows16_kernel<T, D, LAYOUT, PLANNED>;
    static uint64_t lds_reserved = 0;
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), lds, "splat_attention_fwd")) return rc;
    kern<<<((p.total + 7) / 8) * 8, 256, lds, st>>>(p);
    return check_launch("splat_attention_fwd");
}

template <typename T, int D>
static int launch_layout(const AttnParams& p, bool kt, hipStream_t st) {
    if (p.keys_anywhere) return launch<T, D, kKeysAnywhere, true>(p, st);
    if (p.plan) return kt ? launch<T, D, kKeysWhole, true>(p, st) : launch<T, D, kKeyRows, true>(p, st);
    return kt ? launch<T, D, kKeysWhole, false>(p, st) : launch<T, D, kKeyRows, false>(p, st);
}
template <typename T>
int launch_attn_rows16(const AttnParams& p, int d, bool kt, hipStream_t st) {
    return d == 64 ? launch_layout<T, 64>(p, kt, st) : launch_layout<T, 128>(p, kt, st);
}
template int launch_attn_rows16<f16>(const AttnParams&, int, bool, hipStream_t);
template int launch_attn_rows16<bf16>(const AttnParams&, int, bool, hipStream_t);

}  // namespace splat

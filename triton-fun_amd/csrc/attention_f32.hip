// Fused ACSR sparse-attention forward in float32 (online softmax), gfx950.
//
// Bound: the float32 matrix instructions (157 TFLOP/s nominal on this chip, 154 measured in a large product: a sixteenth of
// what the 16-bit ones give), so everything here serves two ends: no matrix work on masked positions, and matrix work on every
// SIMD at every moment.
//   * 16x16x4 instructions: a wavefront owns 16 query rows and takes keys in subtiles of 16, skipping the subtiles outside its
//     rows' spans (a window of 257 costs 272 + 15 positions on average; the 32x32x2 form, with 32 rows and tiles of 64 keys,
//     346).  Both forms run at the same rate.
//   * little vector arithmetic: these matrix instructions run on the vector units (a loop of them takes 33 cycles each, with
//     four v_fma beside each 46), so every address that can be wavefront-uniform is, and masks are built only where needed.
//   * small tiles: 16 KB a stage (32 keys at d = 64, 16 at d = 128) in a ring of two, so that four workgroups fit a CU (three at
//     d = 128, by registers) and one computes while another waits; 64 rows a workgroup, so that short problems spread over more CUs.
//     (Tiles of half or twice the size and rings of three measured equal or slower, up to 10 %.)
//   * the layouts of tile_f32.hpp: 16-byte LDS reads throughout and no exchange of probabilities between lanes.
// Measured against the 32x32x2 kernel it replaces (128 rows a workgroup, tiles of 64 keys): B = 32, H = 12, L = 1024, window 257,
// d = 64: 347 -> 255 us (matrix units busy 63 % of the time); one head of 512 rows, window 64: 20.0 -> 9.8 us.  Masks with little or
// nothing to skip, where a read from LDS serves half the rows it served there, gain less and lose nothing: 64 heads of 4096 rows,
// blocks of 512 d = 64 571 -> 521 us, d = 128 1197 -> 1039, no mask 2224 -> 2100 and 4972 -> 4112; 32 heads of 2048 rows, blocks of
// 512 147 -> 143 and 315 -> 308, of 128 45 -> 42 and 94 -> 95; one head of 1024 rows, no mask 82 -> 49 and 156 -> 87.
#include "tile_f32.hpp"

namespace splat {

constexpr int kF32Stages = 2;

template <int D, bool KT, bool PLANNED>
__global__ __launch_bounds__(256, 3) void attn_fwd_f32_kernel(const AttnParams p) {
    constexpr int BN = f32_tile(D), SUB = BN / 16, NSTAGE = kF32Stages, PD = NSTAGE - 1;
    constexpr int KQ = D / 16;  // groups of 16 contraction values of the score product
    constexpr int DH = D / 64;  // 64-column halves of the output
    constexpr int V_ROWB = D * 4, K_ROWB = KT ? BN * 4 : D * 4;
    constexpr int TILE = BN * D * 4, STAGE = 2 * TILE;
    constexpr int NDMA = STAGE / 4096;  // copy instructions per wavefront and tile
    constexpr int K_SWZ = KT ? (K_ROWB == 128 ? 2 : 0) : 1;
    static_assert(kPlanBM == 2 * kHalfRows && kBN % BN == 0, "half a row block of the plan per workgroup");

    extern __shared__ __attribute__((aligned(1024))) char smem[];
    __shared__ SegPlan s_plan[SPLAT_MAX_SEGMENTS];
    __shared__ PlanScratch<kPlanBM> s_ps;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;

    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    if (logical >= p.total) return;
    const int per_head = 2 * p.n_row_blocks;
    const int bh = logical / per_head;
    const int at = per_head - 1 - logical % per_head;  // later rows of causal patterns carry the most keys: first
    const int rb = at >> 1, half = at & 1;
    const int b = bh / p.H, h = bh % p.H;
    const int rs = p.row_stride, L = p.L;
    const int k0 = half * kHalfRows;                    // the workgroup's first row within its row block
    const int r0 = block_first_row(rb, kPlanBM, rs) + rs * k0;
    if (r0 >= L) return;

    const float* qb = (const float*)p.q + b * p.q_sb + h * p.q_sh;
    const float* kb = (const float*)p.k + b * p.k_sb + h * p.k_sh;
    const float* vb = (const float*)p.v + b * p.v_sb + h * p.v_sh;
    float* ob = (float*)p.o + b * p.o_sb + h * p.o_sh;
    const int my_row = r0 + rs * (wave * 16 + n);

    // ---- the lane's share of its Q row, resident: B operand of the score product ----
    float q[D / 4];
    {
        const float* qr = qb + (int64_t)min(my_row, L - 1) * p.q_sl;
#pragma unroll
        for (int t = 0; t < KQ; ++t) {
            if constexpr (KT) {  // instruction s takes d = 4s + g
#pragma unroll
                for (int j = 0; j < 4; ++j) q[4 * t + j] = qr[16 * t + 4 * j + g];
            } else {
                const f32x4 x = *reinterpret_cast<const f32x4*>(qr + 16 * t + 4 * g);
#pragma unroll
                for (int j = 0; j < 4; ++j) q[4 * t + j] = x[j];
            }
        }
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

    // ---- asynchronous copies of one tile: 1 KiB blocks, wavefront w issues blocks w, w + 4, ...  The vector arithmetic shares
    // its units with the float32 matrix instructions, so a tile whose positions all exist is copied from running wavefront-
    // uniform pointers and per-lane offsets that stay the same for the whole segment ----
    constexpr int NI = TILE / 4096;  // blocks per wavefront and operand
    constexpr int V_CPR = V_ROWB / 16, V_RPI = 1024 / V_ROWB, K_CPR = K_ROWB / 16, K_RPI = 1024 / K_ROWB;
    auto issue_general = [&](const HalfWalk& w, int stage) {
        const int j0 = w.tile * BN;
        char* ks_w = smem + stage * STAGE;
        auto key_row = [&](int row) { return min(max(w.pl.c0 + w.pl.cs * (j0 + row), 0), L - 1); };
        dma_tile<float, V_ROWB, BN, 0>(ks_w + TILE, wave, lane, [&](int row) { return vb + (int64_t)key_row(row) * p.v_sl; });
        if constexpr (KT) {
            // rows = d, BN consecutive keys each (dense walk); a chunk past the last key is replaced by the last whole one
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int blk = wave + 4 * i, flat = blk * 64 + lane;
                const int row = flat / K_CPR;
                const int c = min(w.pl.c0 + j0 + logical_chunk<K_ROWB, K_SWZ>(row, flat % K_CPR) * 4, L - 4);
                dma16(kb + (int64_t)row * p.k_sd + c, ks_w + blk * 1024);
            }
        } else {
            dma_tile<float, K_ROWB, BN, K_SWZ>(ks_w, wave, lane, [&](int row) { return kb + (int64_t)key_row(row) * p.k_sl; });
        }
    };
    uint32_t v_off = 0, k_off[NI];
    const char *v_next = nullptr, *k_next = nullptr;
    int64_t v_row = 0, k_row = 0;  // bytes from one tile row to the next
    bool off_fits = true;          // the copy instruction takes a 32-bit offset
    auto set_offsets = [&](const HalfWalk& w) {
        v_row = (int64_t)p.v_sl * 4 * w.pl.cs;
        k_row = KT ? (int64_t)p.k_sd * 4 : (int64_t)p.k_sl * 4 * w.pl.cs;
        off_fits = v_row * V_RPI < ((int64_t)1 << 31) && k_row * K_RPI < ((int64_t)1 << 31);
        v_off = (uint32_t)(v_row * (lane / V_CPR)) + (lane % V_CPR) * 16;
#pragma unroll
        for (int i = 0; i < NI; ++i)
            k_off[i] = (uint32_t)(k_row * (lane / K_CPR)) +
                       logical_chunk<K_ROWB, K_SWZ>((wave + 4 * i) * K_RPI + lane / K_CPR, lane % K_CPR) * 16;
        const int64_t first = w.pl.c0 + (int64_t)w.pl.cs * BN * w.tile;
        v_next = reinterpret_cast<const char*>(vb) + first * p.v_sl * 4 + wave * V_RPI * v_row;
        k_next = reinterpret_cast<const char*>(kb) + (KT ? first * 4 : first * p.k_sl * 4) + wave * K_RPI * k_row;
    };
    // copy tile `w.tile` into the stage and move on (w: the fetching walk; its pointers stand at that tile)
    auto issue_next = [&](HalfWalk& w, int stage) {
        const int last = w.pl.c0 + w.pl.cs * (w.tile * BN + BN - 1);
        if (off_fits && last < L && w.pl.c0 + w.pl.cs * w.tile * BN >= 0) {
            char* ks_w = smem + stage * STAGE;
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                dma16_uniform(k_next + 4 * i * K_RPI * k_row, k_off[i], ks_w + (wave + 4 * i) * 1024);
                dma16_uniform(v_next + 4 * i * V_RPI * v_row, v_off, ks_w + TILE + (wave + 4 * i) * 1024);
            }
        } else {
            issue_general(w, stage);
        }
        v_next += BN * v_row;
        k_next += KT ? (int64_t)(BN * 4) : BN * k_row;
        if (++w.tile >= w.end) {
            ++w.seg;
            next_segment(w);
            if (w.seg < p.n_seg) set_offsets(w);
        }
    };

    // ---- LDS read addresses: of stage 0, moved on once a tile ----
    const uint32_t smem_base = lds_address(smem);
    uint32_t k_addr[KT ? 1 : KQ];
    if constexpr (KT)
        k_addr[0] = smem_base + g * K_ROWB + n * 4;
    else
#pragma unroll
        for (int t = 0; t < KQ; ++t) k_addr[t] = smem_base + lds_off<K_ROWB, true>(n, (16 * t + 4 * g) * 4);
    uint32_t v_addr = smem_base + TILE + 4 * g * V_ROWB + n * 16;

    HalfWalk fetch, cur;
    fetch.seg = 0;
    next_segment(fetch);
    if (fetch.seg < p.n_seg) set_offsets(fetch);
    cur = fetch;
    PlanRec win_rec = {0, 0, 1, 0};
    if constexpr (PLANNED) {
        if (cur.seg < p.n_seg) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + wave * 16 + n)];
    }
#pragma unroll
    for (int i = 0; i < PD; ++i) {
        if (i < total) {
            issue_next(fetch, i);
        }
    }

    f32x4 o[4 * DH];
#pragma unroll
    for (int i = 0; i < 4 * DH; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_ref = kNegBigA, l_run = 0.f;
    const float c2 = p.scale_log2e;
    RowState rows;
    bool entered = false;
    int stage = 0, stage_pf = PD;

#if defined(__HIP_DEVICE_COMPILE__)
    // Q is in its registers before the loop, so that no wait of the compiler's for it holds up the copies in flight there
#pragma unroll
    for (int i = 0; i < D / 4; ++i) asm volatile("" ::"v"(q[i]));
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

        // this wavefront's copies of tile `it` have landed once only those of the later tiles are outstanding; after the
        // barrier everybody's have, and everybody is done with tile it - 1, whose stage the next fetch overwrites
        if (total - 1 - it >= PD - 1)
            wait_loads<NDMA*(PD - 1)>();
        else
            wait_loads<0>();
        __builtin_amdgcn_s_barrier();
        if (it + PD < total) {
            issue_next(fetch, stage_pf);
            stage_pf = stage_pf + 1 == NSTAGE ? 0 : stage_pf + 1;
        }

        if (j0 + BN > rows.lo_min && j0 < rows.hi_max) {
            auto sub_live = [&](int s) { return SUB == 1 || (j0 + 16 * s + 16 > rows.lo_min && j0 + 16 * s < rows.hi_max); };
            const bool full = j0 >= rows.lo_max && j0 + BN <= rows.hi_min;
            // Fragments are requested a phase ahead of their use (all of the tile's K now, V before the exponentials), outside
            // the branches of the subtiles; the barriers to scheduling keep the compiler from moving the requests down again.
            f32x4 kf[SUB][KQ];
#pragma unroll
            for (int u = 0; u < SUB; ++u)
#pragma unroll
                for (int t = 0; t < KQ; ++t) {
                    if constexpr (KT) {
                        const uint32_t blk = K_ROWB == 128 ? (u ^ ((g >> 1) & 1)) * 64 : 0;
#pragma unroll
                        for (int j = 0; j < 4; ++j) kf[u][t][j] = lds_load_f32(k_addr[0] + blk + (16 * t + 4 * j) * K_ROWB);
                    } else {
                        kf[u][t] = lds_load_f32x4(k_addr[t] + 16 * u * K_ROWB);
                    }
                }
            __builtin_amdgcn_sched_barrier(0);
            f32x4 s[SUB];
#pragma unroll
            for (int u = 0; u < SUB; ++u) {
                if (!sub_live(u)) {
                    s[u] = f32x4{kNegBigA, kNegBigA, kNegBigA, kNegBigA};
                    continue;
                }
                s[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int t = 0; t < KQ; ++t)
#pragma unroll
                    for (int j = 0; j < 4; ++j) mma4(s[u], kf[u][t][j], q[4 * t + j]);
            }
            f32x4 vf[2][4][DH];
            auto load_v = [&](int u) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int hh = 0; hh < DH; ++hh) vf[u & 1][j][hh] = lds_load_f32x4(v_addr + (16 * u + j) * V_ROWB + 256 * hh);
            };
            load_v(0);
            __builtin_amdgcn_sched_barrier(0);
            if (!full) rows.mask_tile(s, j0, g, cur.pl.uniform != 0);
            float mx = s[0][0];
#pragma unroll
            for (int u = 0; u < SUB; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) mx = fmaxf(mx, s[u][j]);
            // ---- online softmax against a lazily moved reference (see attention.hip) ----
            mx = over_groups(mx, [](float x, float y) { return fmaxf(x, y); });
            if (__any((mx - m_ref) * c2 > kRescaleThreshold)) {
                const float m_new = ((mx - m_ref) * c2 > kRescaleThreshold) ? mx : m_ref;
                const float alpha = fast_exp2((m_ref - m_new) * c2);
                m_ref = m_new;
                l_run *= alpha;
#pragma unroll
                for (int i = 0; i < 4 * DH; ++i) o[i] *= alpha;
            }
            // a row that has seen no live score keeps offset 0, so that its (all masked) entries map to 0
            const float mb = m_ref > 0.5f * kNegBigA ? m_ref * c2 : 0.f;
#pragma unroll
            for (int u = 0; u < SUB; ++u) {
                if (u + 1 < SUB) {
                    load_v(u + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (!sub_live(u)) continue;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s[u][j] = fast_exp2(fmaf(s[u][j], c2, -mb));
                    l_run += s[u][j];
                }
                // ---- O^T += V^T . P^T ----
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int hh = 0; hh < DH; ++hh)
#pragma unroll
                        for (int dt = 0; dt < 4; ++dt) mma4(o[4 * hh + dt], vf[u & 1][j][hh][dt], s[u][j]);
            }
        }
        if (!cur.pl.uniform) rows.next_tile();
        stage = stage + 1 == NSTAGE ? 0 : stage + 1;
        const int delta = stage == 0 ? -(NSTAGE - 1) * STAGE : STAGE;
        v_addr += delta;
#pragma unroll
        for (int t = 0; t < (KT ? 1 : KQ); ++t) k_addr[t] += delta;
        if (++cur.tile >= cur.end) {
            ++cur.seg;
            next_segment(cur);
            entered = false;
        }
    }

    // ---- epilogue: a lane holds 16 consecutive columns (per 64) of its row ----
    const float l_tot = over_groups(l_run, [](float x, float y) { return x + y; });
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    if (my_row < L) {
        if (p.lse != nullptr && g == 0)
            p.lse[(int64_t)bh * L + my_row] = l_tot > 0.f ? (m_ref * c2 + __log2f(l_tot)) * 0.6931471805599453f : __builtin_inff();
        float* orow = ob + (int64_t)my_row * p.o_sl;
#pragma unroll
        for (int hh = 0; hh < DH; ++hh)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4 x = {o[4 * hh][i] * inv, o[4 * hh + 1][i] * inv, o[4 * hh + 2][i] * inv, o[4 * hh + 3][i] * inv};
                *reinterpret_cast<f32x4*>(orow + 64 * hh + 16 * g + 4 * i) = x;
            }
    }
}

template <int D, bool KT, bool PLANNED>
static int launch(const AttnParams& p0, hipStream_t st) {
    begin_launch();
    AttnParams p = p0;
    p.n_row_blocks = count_row_blocks(p.L, kPlanBM, p.row_stride);
    p.total = p.B * p.H * 2 * p.n_row_blocks;
    if (PLANNED && KT) p.plan += plan_variant_recs(p.n_row_blocks, p.n_seg);  // the dense-walk variant
    const size_t lds = kF32Stages * 2 * f32_tile(D) * D * 4;
    auto kern = attn_fwd_f32_kernel<D, KT, PLANNED>;
    static uint64_t lds_reserved = 0;
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), lds, "splat_attention_fwd")) return rc;
    kern<<<((p.total + 7) / 8) * 8, 256, lds, st>>>(p);
    return check_launch("splat_attention_fwd");
}

int launch_attn_f32(const AttnParams& p, int d, bool kt, hipStream_t st) {
    if (p.plan) {
        if (d == 64) return kt ? launch<64, true, true>(p, st) : launch<64, false, true>(p, st);
        return kt ? launch<128, true, true>(p, st) : launch<128, false, true>(p, st);
    }
    if (d == 64) return kt ? launch<64, true, false>(p, st) : launch<64, false, false>(p, st);
    return kt ? launch<128, true, false>(p, st) : launch<128, false, false>(p, st);
}

}  // namespace splat

// The keys' side of the fused backward at d = 128, 16-bit types, in launches of at most 1024 row blocks (run_bwd_keys in
// attention_bwd.hip has the line): dK and dV from one walk over the transposed mask's plan.
//
// Products, layouts and plan are those of attention_bwd.hip's dK + dV mode (rows are keys, positions queries; X = Q, Y = dO):
//     S^T = X K^T;  P;  dP^T = Y V^T;  dS = P (dP - D);  dK^T += X^T dS^T;  dV^T += Y^T P^T
// Both accumulators of 32 keys need over 300 registers there, and a launch for each takes the scores, the exponentials and the copies
// of both tiles twice (five products for four).  Here a workgroup is eight wavefronts over the same 128 keys, and two wavefronts
// share 32 of them: of every tile of 64 positions each computes S, P, dP and dS of its own 32, one wavefront of the pair keeps
// dK and the other dV, and what the other one needs (dS of the one half, P of the other: 2 KiB as ready B operands) goes through
// LDS.  The accumulating products run one tile behind the scores, so that the pair needs no barrier but the tile's own and the
// exponentials issue between matrix instructions that do not wait for them; the tiles come through a ring of three stages.
// One workgroup of 133 KiB a CU: two wavefronts a SIMD, as two workgroups of the four-wavefront kernel would give.  A second one
// would take more than a smaller ring: 64 registers of accumulators and 64 of K and V fragments are all that the 128 registers of
// a wavefront at four a SIMD hold.
// Bound: the latency of the walk (its launches leave the chip part idle); where they fill it, what one workgroup a CU leaves
// uncovered: B = 2, H = 32, L = 8192, dilated 512 / 2, bfloat16: 545 us against 322 + 233 for the two launches.  Measured and not
// taken there: one role's wavefronts at a higher priority 559, four or three fragments ahead instead of six 549 / 554.
#include "attn_bwd.hpp"

namespace splat {

typedef float f32x2 __attribute__((ext_vector_type(2)));

template <typename T>
__global__ __launch_bounds__(512, 2) void attn_bwd_pair_kernel(const BwdParams p) {
    constexpr int D = 128, ES = 2, BM = 128, BN = 64, HALF = 32;
    static_assert(sizeof(T) == ES && BM == kPlanBM, "16-bit element types, the plan's row blocks");
    constexpr int KS = D / 16;        // contraction steps of the products over d
    constexpr int DT = D / 32;        // 32-row tiles of the transposed accumulator
    constexpr int ROWB = D * ES, TILE = BN * ROWB, STAGE = 2 * TILE, NSTAGE = 3;
    constexpr int XCH_AT = NSTAGE * STAGE;            // two buffers of 2 KiB for each wavefront
    constexpr int STATS_AT = XCH_AT + 2 * 8 * 2048;   // lse[64], D[64] of every stage
    constexpr int STATS = 2 * BN * 4;
    constexpr int CPR = ROWB / 16, RPI = 1024 / ROWB;  // chunks per row, rows per 1 KiB copy block
    constexpr int NI = TILE / 8192;                    // copy blocks per wavefront and tile
    constexpr int NDMA = 2 * NI;

    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pair = wave & 3, role = wave >> 2;  // role 0: positions 0 .. 31 of a tile and dK, 1: positions 32 .. 63 and dV
    const int lm = lane & 31, g = lane >> 5;

    load_args(p.total, p.n_row_blocks, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.H, p.row_stride, p.L, p.n_seg, p.plan, p.scale_log2e,
              p.a, p.a_sb, p.a_sh, p.a_sl, p.b, p.b_sb, p.b_sh, p.b_sl, p.x, p.x_sb, p.x_sh, p.x_sl, p.y, p.y_sb, p.y_sh, p.y_sl, p.lse, p.delta);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int bh = quotient(logical, p.by_blocks);
    const int rb = p.n_row_blocks - 1 - (logical - bh * p.n_row_blocks);
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride;
    const int r0 = block_first_row(rb, BM, rs);
    const int L = p.L, Lr = p.Lr;

    const T* xb = (const T*)p.x + b * p.x_sb + h * p.x_sh;
    const T* yb = (const T*)p.y + b * p.y_sb + h * p.y_sh;
    const float* lse_b = p.lse + (int64_t)bh * L;
    const float* del_b = p.delta + (int64_t)bh * L;

    // ---- register operands: fragments of this lane's rows of K and V ----
    int my_row = min(r0 + rs * (pair * 32 + lm), Lr - 1);
    if (p.row_map) my_row = min(max(p.row_map[my_row], 0), L - 1);
    Frag<T> af[KS], bf[KS];
    {
        const T* ar = (const T*)p.a + b * p.a_sb + h * p.a_sh + (int64_t)my_row * p.a_sl + 8 * g;
        const T* br = (const T*)p.b + b * p.b_sb + h * p.b_sh + (int64_t)my_row * p.b_sl + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) af[ks] = global_frag<T>(ar + 16 * ks);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) bf[ks] = global_frag<T>(br + 16 * ks);
    }
    const float c2 = p.scale_log2e;

    // ---- plan ----
    const PlanRec* const pt = p.plan;
    const int n_rb = p.n_row_blocks;
    auto seg_plan_of = [&](int sg) {
        const PlanRec r = plan_uniform_load(pt + plan_seg_at(p.n_seg, rb, sg));
        SegPlan t;
        t.c0 = r.x, t.cs = r.y, t.n_tiles = r.z, t.uniform = r.w;
        return t;
    };
    int total_tiles = 0;
    for (int sg = 0; sg < p.n_seg; ++sg) total_tiles += seg_plan_of(sg).n_tiles;
    total_tiles = __builtin_amdgcn_readfirstlane(total_tiles);

    // ---- tile copies (see attention_bwd.hip): wavefront w issues blocks w, w + 8 of X and of Y; the swizzle has a period of 16
    // rows, so a lane's source offset does not depend on the block ----
    auto position_row = [&](const SegPlan& pl, int j) { return min(max(pl.c0 + pl.cs * j, 0), L - 1); };
    const int c_row = wave * RPI + lane / CPR;  // tile row of this lane's chunk in block `wave`
    const int c_byte = logical_chunk<ROWB, 3>(c_row, lane % CPR) * 16;
    auto issue_tile_general = [&](const SegPlan& pl, int tile, int stage) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int64_t r = position_row(pl, tile * BN + c_row + 8 * RPI * i);
            char* const to = smem + stage * STAGE + (wave + 8 * i) * 1024;
            dma16(reinterpret_cast<const char*>(xb + r * p.x_sl) + c_byte, to);
            dma16(reinterpret_cast<const char*>(yb + r * p.y_sl) + c_byte, to + TILE);
        }
    };
    auto issue_stats = [&](const SegPlan& pl, int tile, int stage) {
        char* const to = smem + STATS_AT + stage * STATS;
        if (wave == 0) dma4(lse_b + position_row(pl, tile * BN + lane), to);
        if (wave == 1) dma4(del_b + position_row(pl, tile * BN + lane), to + BN * 4);
    };
    uint32_t x_lane_off = 0, y_lane_off = 0;
    bool lane_off_fits = true;
    const char *x_next = nullptr, *y_next = nullptr;
    int64_t x_key = 0, y_key = 0;  // bytes from one tile position to the next
    auto set_lane_offsets = [&](const SegPlan& pl) {
        const int r = lane / CPR;
        const int64_t x_far = (int64_t)pl.cs * (RPI - 1) * p.x_sl * ES + ROWB, y_far = (int64_t)pl.cs * (RPI - 1) * p.y_sl * ES + ROWB;
        lane_off_fits = x_far < ((int64_t)1 << 32) && y_far < ((int64_t)1 << 32);
        x_key = (int64_t)p.x_sl * ES * pl.cs;
        y_key = (int64_t)p.y_sl * ES * pl.cs;
        x_lane_off = (uint32_t)(x_key * r) + c_byte;
        y_lane_off = (uint32_t)(y_key * r) + c_byte;
        x_next = reinterpret_cast<const char*>(xb) + (int64_t)pl.c0 * p.x_sl * ES + (int64_t)wave * RPI * x_key;
        y_next = reinterpret_cast<const char*>(yb) + (int64_t)pl.c0 * p.y_sl * ES + (int64_t)wave * RPI * y_key;
    };
    auto tile_is_fast = [&](const SegPlan& pl, int tile) {
        const int j0 = tile * BN;
        return lane_off_fits && pl.c0 + pl.cs * j0 >= 0 && pl.c0 + pl.cs * (j0 + BN - 1) < L;
    };
    auto issue_step = [&](int i, int stage) {
        char* const to = smem + stage * STAGE + wave * 1024;
        if (i < NI)
            dma16_uniform(x_next + (int64_t)(8 * RPI * i) * x_key, x_lane_off, to + 8192 * i);
        else
            dma16_uniform(y_next + (int64_t)(8 * RPI * (i - NI)) * y_key, y_lane_off, to + TILE + 8192 * (i - NI));
    };
    int pf_seg = 0, pf_tile = 0;
    SegPlan ppl = {0, 1, 0, 1};
    auto pf_enter_segment = [&]() {
        pf_tile = 0;
        while (pf_seg < p.n_seg) {
            ppl = seg_plan_of(pf_seg);
            if (ppl.n_tiles > 0) break;
            ++pf_seg;
        }
        if (pf_seg < p.n_seg) set_lane_offsets(ppl);
    };
    auto advance_fetch = [&]() {
        x_next += BN * x_key;
        y_next += BN * y_key;
        if (++pf_tile >= ppl.n_tiles) {
            ++pf_seg;
            pf_enter_segment();
        }
    };

    // ---- LDS read addresses of stage 0, moved on once a tile: row reads of this wavefront's half (X; Y is TILE further), and
    // transposing reads of the accumulated operand (role 0: X, role 1: Y) from its half, whose other half is `other` away ----
    const uint32_t smem_base = lds_address(smem);
    const int tr_row = (lane & 15) >> 2;
    const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);  // element column inside a 32-element block
    auto dual_off = [&](int row, int byte_col) { return row * ROWB + dual_chunk<ROWB>(row, byte_col >> 4) * 16 + (byte_col & 15); };
    // (one register each: the swizzle XORs the chunk with bits of the row, so contraction step ks flips bits 5 .. 7 of the
    // address, feature block dt bits 6 and 7, and 8 rows on bit 5)
    const uint32_t mine_at = smem_base + role * (HALF * ROWB);
    uint32_t xr_addr = mine_at + dual_off(lm, 8 * g * ES), yr_addr = xr_addr + TILE;
    uint32_t tr_addr = mine_at + role * TILE + dual_off(4 * g + tr_row, tr_col * ES);
    const uint32_t other = role == 0 ? HALF * ROWB : (uint32_t)(-HALF * ROWB);
    uint32_t st_addr = smem_base + STATS_AT + role * (HALF * 4) + 16 * g;  // lse of positions 4g .. of the half; D is BN * 4 further
    const uint32_t xch_out = smem_base + XCH_AT + wave * 2048 + lane * 16, xch_in = smem_base + XCH_AT + (wave ^ 4) * 2048 + lane * 16;

    pf_enter_segment();
    PlanRec win_rec = {0, 0, 1, 0};
    if (pf_seg < p.n_seg) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, pf_seg, pair * 32 + lm)];
    if (total_tiles > 0) {
        if (tile_is_fast(ppl, pf_tile)) {
#pragma unroll
            for (int s = 0; s < NDMA; ++s) issue_step(s, 0);
        } else {
            issue_tile_general(ppl, pf_tile, 0);
        }
        issue_stats(ppl, pf_tile, 0);
        advance_fetch();
    }
    f32x16 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[dt][j] = 0.f;

    int cur_seg = -1, cur_tile = 0;
    RowWin win = {0, 0, 1};
    int first = 0, dec = 0;
    uint64_t pat = ~0ull;
    int w_lo_min = 0, w_lo_max = 0, w_hi_min = 0, w_hi_max = 0;
    SegPlan cpl = {0, 1, 0, 1};
    int stage_it = 0, stage_pf = 1;
    Frag<T> own[2];  // B operands of the half computed in the step before, 16 positions each: dS (role 0) or P (role 1)
    bool prev_mine = false, prev_other = false;  // which halves of the step before hold entries of the pair's rows
#pragma unroll
    for (int t = 0; t < 2; ++t) own[t].v = __builtin_bit_cast(typename Frag<T>::vec, u32x4{0u, 0u, 0u, 0u});
#if defined(__HIP_DEVICE_COMPILE__)
    // the register operands are in their registers before the loop (see attention_bwd.hip)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(af[ks].v), "v"(bf[ks].v));
#endif

    // step `it`: scores of tile `it`, accumulation of tile it - 1
    for (int it = 0; it <= total_tiles; ++it) {
        const bool has_tile = it < total_tiles;
        int j0 = 0;
        if (has_tile) {
            if (cur_seg < 0 || cur_tile >= cpl.n_tiles) {
                do {
                    ++cur_seg;
                    cpl = seg_plan_of(cur_seg);
                } while (cpl.n_tiles == 0);
                cur_tile = 0;
                if (it > 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur_seg, pair * 32 + lm)];
                win.lo = win_rec.x, win.cnt = win_rec.y, win.lin = win_rec.z;
                first = win_rec.w;
                const PlanRec r = plan_uniform_load(pt + plan_span_at(n_rb, p.n_seg, rb, cur_seg, pair));
                pat = ~0ull;
                if (!cpl.uniform) {
                    dec = BN % win.lin;
                    pat = 0;
                    for (int q = 0; q < 64; q += win.lin) pat |= 1ull << q;
                }
                w_lo_min = r.x, w_lo_max = r.y, w_hi_min = r.z, w_hi_max = r.w;
            }
            j0 = cur_tile * BN;
            ++cur_tile;
        }

        // this wavefront's copies of tile `it` have landed and its half of step it - 1 is in the exchange; after the barrier
        // everybody's, and everybody is done with tile it - 2, whose stage the next fetch overwrites
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

        const bool fetch = it + 1 < total_tiles;
        bool spread = false;
        if (fetch) {
            spread = tile_is_fast(ppl, pf_tile);
            if (!spread) issue_tile_general(ppl, pf_tile, stage_pf);
            issue_stats(ppl, pf_tile, stage_pf);
        }
        auto half_live = [&](int hf) { return has_tile && j0 + HALF * hf + HALF > w_lo_min && j0 + HALF * hf < w_hi_max; };
        const bool mine = half_live(role), others = half_live(1 - role);

        const uint32_t in_at = xch_in + ((it + 1) & 1) * (8 * 2048), out_at = xch_out + (it & 1) * (8 * 2048);
        Frag<T> in[2];
        auto load_in = [&]() {
#pragma unroll
            for (int t = 0; t < 2; ++t) in[t].v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128(in_at + 1024 * t));
        };
        const uint32_t to_addr = tr_addr + other;
        // instruction i of the accumulation: 16 positions i / 4 (this wavefront's half first), 32 features i % 4
        auto load_t = [&](int i) {
            const uint32_t from = (i >= 8 ? to_addr : tr_addr) ^ (64u * (i & 3)), at = 16 * ((i >> 2) & 1) * ROWB;
            return frag_from_tr<T>(lds_load_tr16(from + at), lds_load_tr16((from ^ 32u) + at + 8 * ROWB));
        };
        auto b_of = [&](int i) { return i >= 8 ? in[(i >> 2) & 1] : own[(i >> 2) & 1]; };

        f32x16 s, dp;
        Frag<T> pn[2], dn[2];  // P and dS of this step
        auto load_x = [&](int i) {  // i < KS: X, then Y
            Frag<T> f;
            f.v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128((i < KS ? xr_addr : yr_addr) ^ (32u * (i % KS))));
            return f;
        };
        auto scores = [&]() {
            constexpr int N = 2 * KS, AHEAD = 6;
            Frag<T> xf[N];
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) xf[i] = load_x(i);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 16; ++j) s[j] = 0.f, dp[j] = 0.f;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                if (i < KS)
                    mma32(s, xf[i], af[i % KS]);
                else
                    mma32(dp, xf[i], bf[i % KS]);
                if (i + AHEAD < N) {
                    xf[i + AHEAD] = load_x(i + AHEAD);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (i % 2 == 0 && i / 2 < NDMA) {
                    if (spread) issue_step(i / 2, stage_pf);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (!(j0 + HALF * role >= w_lo_max && j0 + HALF * role + HALF <= w_hi_min)) {
                const uint32_t bits = (uint32_t)(row_live_bits(win, j0, first, pat) >> (HALF * role)) >> (4 * g);
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int c = 8 * (j >> 2) + (j & 3);
                    s[j] = keep_or_mask(s[j], ((int)(bits << (31 - c))) >> 31);
                }
            }
        };
        f32x2 lse2[2], d2[2];
        auto load_stats = [&](int k) {  // of registers 2k, 2k + 1
            const uint32_t at = st_addr + 32 * (k >> 1) + 8 * (k & 1);
            lse2[k & 1] = *reinterpret_cast<__attribute__((address_space(3))) const f32x2*>((uintptr_t)at);
            d2[k & 1] = *reinterpret_cast<__attribute__((address_space(3))) const f32x2*>((uintptr_t)(at + BN * 4));
        };
        auto element = [&](int j) {  // P and dS of register j
            const float e = fast_exp2(fmaf(s[j], c2, -1.4426950408889634f * lse2[(j >> 1) & 1][j & 1]));
            pn[j >> 3].v[j & 7] = (T)e;
            dn[j >> 3].v[j & 7] = (T)(e * (dp[j] - d2[(j >> 1) & 1][j & 1]) * p.scale);
        };

        if (mine && prev_mine && prev_other) {
            // the body of a walk: exponentials between the matrix instructions of the tile before
            scores();
            constexpr int N = 16, AHEAD = 3;
            Frag<T> tf[N];
            load_stats(0);
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) tf[i] = load_t(i);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < N; ++i) {
                mma32(acc[i & 3], tf[i], b_of(i));
                if (i + AHEAD < N) tf[i + AHEAD] = load_t(i + AHEAD);
                if (i == 4) load_in();
                if (i % 2 == 0 && i + 2 < N) load_stats(i / 2 + 1);
                element(i);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            if (mine) {
                scores();
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    load_stats(k);
                    element(2 * k);
                    element(2 * k + 1);
                }
            } else if (spread) {
#pragma unroll
                for (int i = 0; i < NDMA; ++i) issue_step(i, stage_pf);
            }
            if (prev_mine) {
#pragma unroll
                for (int i = 0; i < 8; ++i) mma32(acc[i & 3], load_t(i), b_of(i));
            }
            if (prev_other) {
                load_in();
#pragma unroll
                for (int i = 8; i < 16; ++i) mma32(acc[i & 3], load_t(i), b_of(i));
            }
        }
        if (mine) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const u32x4 pw = __builtin_bit_cast(u32x4, pn[t].v), dw = __builtin_bit_cast(u32x4, dn[t].v);
                own[t].v = __builtin_bit_cast(typename Frag<T>::vec, role == 0 ? dw : pw);
                *reinterpret_cast<__attribute__((address_space(3))) u32x4*>((uintptr_t)(out_at + 1024 * t)) = role == 0 ? pw : dw;
            }
        }
        prev_mine = mine, prev_other = others;

        if (fetch) {
            advance_fetch();
            stage_pf = stage_pf + 1 == NSTAGE ? 0 : stage_pf + 1;
        }
        if (!cpl.uniform) {
            const int f = first - dec;
            first = f < 0 ? f + win.lin : f;
        }
        // the row reads move on to tile it + 1, the transposing ones (a tile behind) to tile `it`
        if (it > 0) {
            const int d_tr = stage_it == 0 ? -(NSTAGE - 1) * STAGE : STAGE;
            tr_addr += d_tr;
        }
        stage_it = stage_it + 1 == NSTAGE ? 0 : stage_it + 1;
        const int d_xr = stage_it == 0 ? -(NSTAGE - 1) * STAGE : STAGE;
        xr_addr += d_xr, yr_addr += d_xr;
        asm volatile("" : "+v"(yr_addr));  // (kept apart from xr_addr: a common set of eight addresses would not fit)
        st_addr += stage_it == 0 ? -(NSTAGE - 1) * STATS : STATS;
    }
    __syncthreads();  // everyone has read the last tile: the stages become the staging area of the output

    // ---- epilogue: out = acc^T transposed through LDS, whole rows per store (each wavefront through a stretch of its own) ----
    {
        constexpr int OROW = D * ES + 16;
        static_assert(8 * 32 * OROW <= NSTAGE * STAGE, "staging space");
        char* const stg = smem + wave * (32 * OROW);
        typedef T vec4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                vec4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = (T)acc[dt][4 * jj + i];
                *reinterpret_cast<vec4*>(stg + lm * OROW + (32 * dt + 8 * jj + 4 * g) * ES) = o;
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        T* const dst = (T*)(role == 0 ? p.out : p.out2) + b * p.o_sb + h * p.o_sh;
#pragma unroll
        for (int i = 0; i < 32 * CPR / 64; ++i) {
            const int flat = i * 64 + lane;
            const int row = flat / CPR, c = flat % CPR;
            const int r = r0 + rs * (pair * 32 + row);
            const u32x4 val = *reinterpret_cast<const u32x4*>(stg + row * OROW + c * 16);
            if (r < Lr) __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(reinterpret_cast<char*>(dst + (int64_t)r * p.o_sl) + c * 16));
        }
    }
}

template <typename T>
int launch_bwd_pair(const BwdParams& p, hipStream_t st) {
    begin_launch();
    constexpr int LDS_BYTES = 3 * 2 * 64 * 128 * 2 + 2 * 8 * 2048 + 3 * 2 * 64 * 4;
    auto kern = attn_bwd_pair_kernel<T>;
    static uint64_t lds_reserved = 0;
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), LDS_BYTES, "splat_attention_bwd")) return rc;
    kern<<<((p.total + 7) / 8) * 8, 512, LDS_BYTES, st>>>(p);
    return check_launch("splat_attention_bwd");
}
template int launch_bwd_pair<f16>(const BwdParams&, hipStream_t);
template int launch_bwd_pair<bf16>(const BwdParams&, hipStream_t);

}  // namespace splat

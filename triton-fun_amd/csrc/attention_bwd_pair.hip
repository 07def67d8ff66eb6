// The keys' side of the fused backward, 16-bit types: dK and dV from one walk over the transposed mask's plan.
//
// Rows are keys, positions queries; the register operands are K and V, the tiles X = Q, Y = dO:
//     S^T = X K^T;  P;  dP^T = Y V^T;  dS = P (dP - D);  dK^T += X^T dS^T;  dV^T += Y^T P^T
// Both accumulators of 32 keys need over 300 registers at d = 128, and a launch for each takes the scores, the exponentials and the copies
// of both tiles twice (five products for four).  Here a workgroup is four wavefronts over 64 keys, half a row block of the plan, and two
// wavefronts share 32 of them: of every tile of 64 positions each computes S, P, dP and dS of its own 32, one wavefront of the pair keeps
// dK and the other dV, and what the other one needs (dS of the one half, P of the other: 2 KiB as ready B operands) goes through
// LDS, between two barriers a tile: its own half each wavefront accumulates before the second.  73 KiB and 256 registers a wavefront at
// d = 128, two workgroups a CU, whose phases cover each other; 41 KiB and 168 at d = 64, three.  At d = 128 two of a lane's sixteen fragments of
// K and V do not fit: 36 bytes of scratch, of which every tile reads 16 before its scores and 16 before dP, and the second wait is one for the
// next tile's copies, which were requested in between.
// lse and D belong to the positions: 64 floats each a tile, copied into LDS beside the tiles, whose swizzle serves the row-wise reads of
// the scores and the transposing ones of the accumulation (tile_copy.hpp: dual_chunk).
// K and V come through LDS as well, where tile 1 will lie: loaded by every wavefront for itself, 32 bytes of 32 rows an
// instruction, they hold up the address path (the whole backward below: 732 us).
// Bound: as the forward, matrix pipe, LDS reads and the power limit together.  The whole backward, us, against dK and dV in two launches of
// four wavefronts a row block: bfloat16, d = 128, B = 2, H = 32, L = 8192, dilated 512 / 2 764 -> 696; H = 16, causal windows 128 / 512 206 ->
// 191, 371 -> 337, window 33 195 -> 184; 32 heads of 4096, two segments 165 -> 139; 8 heads of 2048, window 512 65 -> 44 (one workgroup of
// eight wavefronts and three stages a CU, which was the faster one there and up to 1024 row blocks: 55).  At d = 64, where one wavefront can
// hold both accumulators (205 registers): 36 heads of 7552, window 150 115 -> 111, 264 of 1252, window 25 105 -> 102, 64 of 4096, window 256
// 124 -> 122.
#include "attn_bwd.hpp"
#include "rows16.hpp"

namespace splat {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T, int D>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void attn_bwd_pair_kernel(const BwdParams p) {
    constexpr int ES = 2, BN = 64, HALF = 32;
    static_assert(sizeof(T) == ES && kPlanBM == 2 * kHalfRows, "16-bit element types, the plan's row blocks");
    constexpr int KS = D / 16;        // contraction steps of the products over d
    constexpr int DT = D / 32;        // 32-row tiles of the transposed accumulator
    constexpr int ROWB = D * ES, TILE = BN * ROWB, STAGE = 2 * TILE, NSTAGE = 2;
    constexpr int XCH_AT = NSTAGE * STAGE;            // 2 KiB for each wavefront
    constexpr int STATS_AT = XCH_AT + 4 * 2048;   // lse[64], D[64] of every stage
    constexpr int STATS = 2 * BN * 4;
    constexpr int CPR = ROWB / 16, RPI = 1024 / ROWB;  // chunks per row, rows per 1 KiB copy block
    constexpr int NI = TILE / 4096;                    // copy blocks per wavefront and tile
    constexpr int NDMA = 2 * NI;

    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pair = wave & 1, role = wave >> 1;  // role 0: positions 0 .. 31 of a tile and dK, 1: positions 32 .. 63 and dV
    const int lm = lane & 31, g = lane >> 5;

    load_args(p.total, p.n_row_blocks, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.H, p.row_stride, p.L, p.n_seg, p.plan, p.scale_log2e,
              p.a, p.a_sb, p.a_sh, p.a_sl, p.b, p.b_sb, p.b_sh, p.b_sl, p.x, p.x_sb, p.x_sh, p.x_sl, p.y, p.y_sb, p.y_sh, p.y_sl, p.lse, p.delta);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int per_head = 2 * p.n_row_blocks;
    const int bh = quotient(logical, p.by_blocks);
    const int at = per_head - 1 - (logical - bh * per_head);
    const int rb = at >> 1, half = at & 1;
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride;
    const int k0 = half * kHalfRows;  // the workgroup's first row within its row block
    const int r0 = block_first_row(rb, kPlanBM, rs) + rs * k0;
    const int L = p.L, Lr = p.Lr;
    if (r0 >= Lr) return;

    const T* xb = (const T*)p.x + b * p.x_sb + h * p.x_sh;
    const T* yb = (const T*)p.y + b * p.y_sb + h * p.y_sh;
    const float* lse_b = p.lse + (int64_t)bh * L;
    const float* del_b = p.delta + (int64_t)bh * L;

    const float c2 = p.scale_log2e;

    // ---- plan ----
    const PlanRec* const pt = p.plan;
    const int n_rb = p.n_row_blocks;
    auto next_segment = [&](HalfWalk& w) {  // the first segment from w.seg on of which this half sees something
        for (int sg = w.seg; sg < p.n_seg; ++sg) {
            w = half_walk<BN>(pt, n_rb, p.n_seg, rb, half, sg);
            if (w.end > w.tile) return;
        }
        w.seg = p.n_seg, w.tile = 0, w.end = 0;
    };
    int total_tiles = 0;
    for (int sg = 0; sg < p.n_seg; ++sg) {
        const HalfWalk w = half_walk<BN>(pt, n_rb, p.n_seg, rb, half, sg);
        total_tiles += w.end - w.tile;
    }
    total_tiles = __builtin_amdgcn_readfirstlane(total_tiles);

    // ---- tile copies (see attention_bwd.hip): wavefront w issues blocks w, w + 4, ... of X and of Y; the swizzle has a period of 16
    // rows, so a lane's source offset does not depend on the block ----
    auto position_row = [&](const SegPlan& pl, int j) { return min(max(pl.c0 + pl.cs * j, 0), L - 1); };
    const int c_row = wave * RPI + lane / CPR;  // tile row of this lane's chunk in block `wave`
    const int c_byte = logical_chunk<ROWB, 3>(c_row, lane % CPR) * 16;
    // the workgroup's own rows of K and V, in the same manner, to where tile 1 will lie: fragments that every wavefront loads for itself take
    // three times as long on the address path
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        int r = min(r0 + rs * (c_row + 4 * RPI * i), Lr - 1);
        if (p.row_map) r = min(max(p.row_map[r], 0), L - 1);
        char* const to = smem + STAGE + (wave + 4 * i) * 1024;
        dma16(reinterpret_cast<const char*>((const T*)p.a + b * p.a_sb + h * p.a_sh + (int64_t)r * p.a_sl) + c_byte, to);
        dma16(reinterpret_cast<const char*>((const T*)p.b + b * p.b_sb + h * p.b_sh + (int64_t)r * p.b_sl) + c_byte, to + TILE);
    }
    auto issue_tile_general = [&](const SegPlan& pl, int tile, int stage) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int64_t r = position_row(pl, tile * BN + c_row + 4 * RPI * i);
            char* const to = smem + stage * STAGE + (wave + 4 * i) * 1024;
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
    auto set_lane_offsets = [&](const HalfWalk& w) {
        const SegPlan& pl = w.pl;
        const int r = lane / CPR;
        const int64_t x_far = (int64_t)pl.cs * (RPI - 1) * p.x_sl * ES + ROWB, y_far = (int64_t)pl.cs * (RPI - 1) * p.y_sl * ES + ROWB;
        lane_off_fits = x_far < ((int64_t)1 << 32) && y_far < ((int64_t)1 << 32);
        x_key = (int64_t)p.x_sl * ES * pl.cs;
        y_key = (int64_t)p.y_sl * ES * pl.cs;
        x_lane_off = (uint32_t)(x_key * r) + c_byte;
        y_lane_off = (uint32_t)(y_key * r) + c_byte;
        const int64_t from = pl.c0 + (int64_t)pl.cs * BN * w.tile;
        x_next = reinterpret_cast<const char*>(xb) + from * p.x_sl * ES + (int64_t)wave * RPI * x_key;
        y_next = reinterpret_cast<const char*>(yb) + from * p.y_sl * ES + (int64_t)wave * RPI * y_key;
    };
    auto tile_is_fast = [&](const SegPlan& pl, int tile) {
        const int j0 = tile * BN;
        return lane_off_fits && pl.c0 + pl.cs * j0 >= 0 && pl.c0 + pl.cs * (j0 + BN - 1) < L;
    };
    auto issue_step = [&](int i, int stage) {
        char* const to = smem + stage * STAGE + wave * 1024;
        if (i < NI)
            dma16_uniform(x_next + (int64_t)(4 * RPI * i) * x_key, x_lane_off, to + 4096 * i);
        else
            dma16_uniform(y_next + (int64_t)(4 * RPI * (i - NI)) * y_key, y_lane_off, to + TILE + 4096 * (i - NI));
    };
    HalfWalk fetch, cur;
    auto advance_fetch = [&]() {
        x_next += BN * x_key;
        y_next += BN * y_key;
        if (++fetch.tile >= fetch.end) {
            ++fetch.seg;
            next_segment(fetch);
            if (fetch.seg < p.n_seg) set_lane_offsets(fetch);
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
    uint32_t xr_addr = mine_at + dual_off(lm, 8 * g * ES);
    uint32_t tr_addr = mine_at + role * TILE + dual_off(4 * g + tr_row, tr_col * ES);
    const uint32_t other = role == 0 ? HALF * ROWB : (uint32_t)(-HALF * ROWB);
    uint32_t st_addr = smem_base + STATS_AT + role * (HALF * 4) + 16 * g;  // lse of positions 4g .. of the half; D is BN * 4 further
    const uint32_t xch_out = smem_base + XCH_AT + wave * 2048 + lane * 16, xch_in = smem_base + XCH_AT + (wave ^ 2) * 2048 + lane * 16;

    fetch.seg = 0;
    next_segment(fetch);
    if (fetch.seg < p.n_seg) set_lane_offsets(fetch);
    cur = fetch;
    PlanRec win_rec = {0, 0, 1, 0};
    if (cur.seg < p.n_seg) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + pair * 32 + lm)];
    if (total_tiles > 0) {
        if (tile_is_fast(fetch.pl, fetch.tile)) {
#pragma unroll
            for (int s = 0; s < NDMA; ++s) issue_step(s, 0);
        } else {
            issue_tile_general(fetch.pl, fetch.tile, 0);
        }
        issue_stats(fetch.pl, fetch.tile, 0);
        advance_fetch();
    }
    f32x16 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[dt][j] = 0.f;

    RowWin win = {0, 0, 1};
    int first = 0, dec = 0;
    uint64_t pat = ~0ull;
    int w_lo_min = 0, w_lo_max = 0, w_hi_min = 0, w_hi_max = 0;
    bool entered = false;
    int stage = 0;
    // K and V as register operands: fragments of this lane's row (in registers before the first fetch into their place)
    wait_loads<0>();
    __builtin_amdgcn_s_barrier();
    Frag<T> af[KS], bf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const uint32_t from = (smem_base + STAGE + dual_off(pair * 32 + lm, 8 * g * ES)) ^ (32u * ks);
        af[ks].v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128(from));
        bf[ks].v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128(from + TILE));
    }
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(af[ks].v), "v"(bf[ks].v));
#endif

    for (int it = 0; it < total_tiles; ++it) {
        if (!entered) {
            if (it > 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + pair * 32 + lm)];
            win.lo = win_rec.x, win.cnt = win_rec.y, win.lin = win_rec.z;
            first = win_rec.w;
            const PlanRec r = plan_uniform_load(pt + plan_span_at(n_rb, p.n_seg, rb, cur.seg, 2 * half + pair));
            pat = ~0ull;
            if (!cur.pl.uniform) {
                dec = BN % win.lin;
                first -= (cur.tile * BN) % win.lin;
                if (first < 0) first += win.lin;
                pat = 0;
                for (int q = 0; q < 64; q += win.lin) pat |= 1ull << q;
            }
            w_lo_min = r.x, w_lo_max = r.y, w_hi_min = r.z, w_hi_max = r.w;
            entered = true;
        }
        const int j0 = cur.tile * BN;

        // this wavefront's copies of tile `it` have landed; after the barrier everybody's have, and everybody is done with tile
        // it - 1, whose stage the next fetch overwrites, and with what it found in the exchange
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

        const bool more = it + 1 < total_tiles;
        bool spread = false;
        if (more) {
            spread = tile_is_fast(fetch.pl, fetch.tile);
            if (!spread) issue_tile_general(fetch.pl, fetch.tile, stage ^ 1);
            issue_stats(fetch.pl, fetch.tile, stage ^ 1);
        }
        auto half_live = [&](int hf) { return j0 + HALF * hf + HALF > w_lo_min && j0 + HALF * hf < w_hi_max; };
        const bool mine = half_live(role), others = half_live(1 - role);

        // fragment of the accumulated operand: step t of 16 positions of this wavefront's half or the other one, features 32 dt ..
        auto load_t = [&](bool its, int t, int dt) {
            const uint32_t from = (its ? tr_addr + other : tr_addr) ^ (64u * dt);
            return frag_from_tr<T>(lds_load_tr16(from + 16 * t * ROWB), lds_load_tr16((from ^ 32u) + (16 * t + 8) * ROWB));
        };
        if (mine) {
            // ---- S^T = X K^T, then dP^T = Y V^T, whose fragments take the places of X's, with the exponentials between its products ----
            f32x16 s, dp;
#pragma unroll
            for (int j = 0; j < 16; ++j) s[j] = 0.f, dp[j] = 0.f;
            Frag<T> xf[KS], yf[KS];
            auto load_row = [&](int ks, int from) {
                Frag<T> f;
                f.v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128((xr_addr ^ (32u * ks)) + from));
                return f;
            };
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) xf[ks] = load_row(ks, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                mma32(s, xf[ks], af[ks]);
                yf[ks] = load_row(ks, TILE);
                if (spread) issue_step(ks, stage ^ 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            static_assert(NDMA == KS, "a copy instruction per product");
            if (!(j0 + HALF * role >= w_lo_max && j0 + HALF * role + HALF <= w_hi_min))
                mask_half(s, (uint32_t)(row_live_bits(win, j0, first, pat) >> (HALF * role)) >> (4 * g));
            f32x4 lse4[2], d4[2];
            auto load_stat = [&](int k4, int from) { return __builtin_bit_cast(f32x4, lds_load128(st_addr + from + 32 * k4)); };
            lse4[0] = load_stat(0, 0);
            Frag<T> tf[2][DT];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                mma32(dp, yf[ks], bf[ks]);
#pragma unroll
                for (int i = 0; i < 16 / KS; ++i) {
                    const int j = 16 / KS * ks + i;
                    if (j % 4 == 0 && j < 12) lse4[(j / 4 + 1) & 1] = load_stat(j / 4 + 1, 0);
                    s[j] = fast_exp2(fmaf(s[j], c2, -1.4426950408889634f * lse4[(j / 4) & 1][j % 4]));
                }
                if (ks >= KS - DT) tf[0][ks - (KS - DT)] = load_t(false, 0, ks - (KS - DT));
                __builtin_amdgcn_sched_barrier(0);
            }
            // ---- P and dS; this role's part accumulates at once, 16 positions at a time, the other one's goes into the exchange ----
            Frag<T> pn[2], dn[2];
            auto element = [&](int j) {
                if (j % 4 == 0) d4[(j / 4) & 1] = load_stat(j / 4, BN * 4);
                pn[j >> 3].v[j & 7] = (T)s[j];
                dn[j >> 3].v[j & 7] = (T)(s[j] * (dp[j] - d4[(j / 4) & 1][j % 4]) * p.scale);
            };
            auto hand_over = [&](int t) {
                const u32x4 pw = __builtin_bit_cast(u32x4, pn[t].v), dw = __builtin_bit_cast(u32x4, dn[t].v);
                lds_store128(xch_out + 1024 * t, role == 0 ? pw : dw);
                Frag<T> own;
                own.v = __builtin_bit_cast(typename Frag<T>::vec, role == 0 ? dw : pw);
                return own;
            };
#pragma unroll
            for (int j = 0; j < 8; ++j) element(j);
            const Frag<T> own0 = hand_over(0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                mma32(acc[dt], tf[0][dt], own0);
                tf[1][dt] = load_t(false, 1, dt);
#pragma unroll
                for (int i = 0; i < 8 / DT; ++i) element(8 + 8 / DT * dt + i);
                __builtin_amdgcn_sched_barrier(0);
            }
            const Frag<T> own1 = hand_over(1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) mma32(acc[dt], tf[1][dt], own1);
        } else if (spread) {
#pragma unroll
            for (int i = 0; i < NDMA; ++i) issue_step(i, stage ^ 1);
        }
        Frag<T> tf[2][DT];
        if (others) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) tf[t][dt] = load_t(true, t, dt);
        }
        lds_barrier();  // both halves are in the exchange
        if (others) {
            Frag<T> in[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) in[t].v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128(xch_in + 1024 * t));
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) mma32(acc[dt], tf[t][dt], in[t]);
        }

        if (more) advance_fetch();
        if (!cur.pl.uniform) {
            const int f = first - dec;
            first = f < 0 ? f + win.lin : f;
        }
        stage ^= 1;
        const int delta = stage == 0 ? -STAGE : STAGE;
        xr_addr += delta, tr_addr += delta;
        st_addr += stage == 0 ? -STATS : STATS;
        if (++cur.tile >= cur.end) {
            ++cur.seg;
            next_segment(cur);
            entered = false;
        }
    }
    __syncthreads();  // everyone has read the last tile: the stages become the staging area of the output

    // ---- epilogue: out = acc^T transposed through LDS, whole rows per store (each wavefront through a stretch of its own) ----
    {
        constexpr int OROW = D * ES + 16;
        static_assert(4 * 32 * OROW <= NSTAGE * STAGE, "staging space");
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

template <typename T, int D>
static int launch(const BwdParams& p0, hipStream_t st) {
    begin_launch();
    constexpr int LDS_BYTES = 2 * 2 * 64 * D * 2 + 4 * 2048 + 2 * 2 * 64 * 4;
    static_assert(LDS_BYTES <= 160 * 1024 / (D == 64 ? 3 : 2), "workgroups per compute unit");
    BwdParams p = p0;
    p.total = p.B * p.H * 2 * p.n_row_blocks;
    p.by_blocks = divisor(2 * p.n_row_blocks), p.by_h = divisor(p.H);
    auto kern = attn_bwd_pair_kernel<T, D>;
    static uint64_t lds_reserved = 0;
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), LDS_BYTES, "splat_attention_bwd")) return rc;
    kern<<<((p.total + 7) / 8) * 8, 256, LDS_BYTES, st>>>(p);
    return check_launch("splat_attention_bwd");
}
template <typename T>
int launch_bwd_pair(const BwdParams& p, int d, hipStream_t st) {
    return d == 64 ? launch<T, 64>(p, st) : launch<T, 128>(p, st);
}
template int launch_bwd_pair<f16>(const BwdParams&, int, hipStream_t);
template int launch_bwd_pair<bf16>(const BwdParams&, int, hipStream_t);

}  // namespace splat

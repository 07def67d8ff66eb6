// Fused backward of the ACSR attention: dQ, dK and dV without any compressed [B, H, L, T] matrix in memory.
//
// With S = scale * Q K^T on the live columns, P = exp(S - lse) (lse: the forward's row statistic), O = P V and the
// upstream gradient dO:  D = rowsum(dO * O),  dP = dO V^T,  dS = P * (dP - D),
//     dQ = scale * dS K        dK = scale * dS^T Q        dV = P^T dO.
// dQ here: rows are queries, positions keys, X = K, Y = V, the register operands A = Q, B = dO; dK + dV in attention_bwd_pair.hip.  Per
// half of a tile, 32 positions:    S^T = X A^T; P; dP^T = Y B^T; dS; acc^T += X^T dS^T
// Built like the forward (attention.hip): a workgroup of 4 wavefronts owns 128 rows, one lane one row (two lanes share it), and walks
// 64-position tiles of the rows' spans as the mask's plan table lists them; per tile X and Y arrive in LDS through the
// asynchronous copy ring.  The dQ launch comes first: its lanes hold their dO rows, so it also computes D (one more read of the
// lane's O row) and stores it for the other.  The X tile is read row-wise (16-byte fragments for S^T) and through the transposing read
// (for acc^T), hence the swizzle that serves both (tile_copy.hpp: dual_chunk).  Probabilities come straight from the
// statistic: no running maximum, no rescale, no second pass.  16-bit types, d = 64 or 128, rows of every operand
// contiguous.
// Bound: as the forward, matrix pipe, LDS reads and the power limit together.  dP's products come right after the scores', with the
// exponentials between them and dP's fragments in the registers of the scores' (64 heads of 8192, dilated 512 / 2, d = 128, dQ: 1 to 3 %).
#include <initializer_list>

#include "attn_bwd.hpp"

namespace splat {

template <typename T, int D>
__global__ __launch_bounds__(256, 2) void attn_bwd_kernel(const BwdParams p) {
    constexpr int ES = 2, BM = 128, BN = 64;
    static_assert(sizeof(T) == ES, "16-bit element types");
    constexpr int KS = D / 16;  // contraction steps of the products over d
    constexpr int DT = D / 32;  // 32-row tiles of the transposed accumulator
    constexpr int ROWB = D * ES;
    constexpr int TILE = BN * ROWB;             // bytes of one operand tile
    constexpr int STAGE = 2 * TILE;               // X, Y
    constexpr int CPR = ROWB / 16, RPI = 1024 / ROWB;  // chunks per row, rows per 1 KiB copy block
    constexpr int NI = TILE / 4096;                   // copy blocks per wavefront and tile
    constexpr int NDMA = 2 * NI;

    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 31, g = lane >> 5;

    load_args(p.total, p.n_row_blocks, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.H, p.row_stride, p.L, p.n_seg, p.plan, p.scale_log2e,
              p.a, p.a_sb, p.a_sh, p.a_sl, p.b, p.b_sb, p.b_sh, p.b_sl, p.x, p.x_sb, p.x_sh, p.x_sl, p.y, p.y_sb, p.y_sh, p.y_sl, p.lse);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int bh = quotient(logical, p.by_blocks);
    const int rb = p.n_row_blocks - 1 - (logical - bh * p.n_row_blocks);
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride;
    const int r0 = block_first_row(rb, BM, rs);
    const int L = p.L;

    const T* xb = (const T*)p.x + b * p.x_sb + h * p.x_sh;
    const T* yb = (const T*)p.y + b * p.y_sb + h * p.y_sh;
    T* ob = (T*)p.out + b * p.o_sb + h * p.o_sh;

    // ---- register operands: fragments of this lane's row, resident for the whole kernel (through LDS, as in attention_bwd_pair.hip, they come
    // no sooner: a stage holds one operand's 128 rows, so that the first tile has to wait for them) ----
    const int my_row = min(r0 + rs * (wave * 32 + lm), L - 1);
    Frag<T> af[KS], bf[KS];
    auto load_row = [&](Frag<T> (&f)[KS], const void* base, int64_t sb, int64_t sh, int64_t sl) {
        const T* const from = (const T*)base + b * sb + h * sh + (int64_t)my_row * sl + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) f[ks] = global_frag<T>(from + 16 * ks);
    };
    load_row(af, p.a, p.a_sb, p.a_sh, p.a_sl);
    load_row(bf, p.b, p.b_sb, p.b_sh, p.b_sl);
    const float c2 = p.scale_log2e;
    const float row_lse2 = p.lse[(int64_t)bh * L + my_row] * 1.4426950408889634f;
    // D = rowsum(dO * O) of the lane's row (the two lanes of a row hold half of it each), kept for this launch and stored
    // for the keys' side that follows it on the stream
    Frag<T> of[KS];  // (all requested before any is used: the accumulators' registers are still free here)
    load_row(of, p.o, p.oo_sb, p.oo_sh, p.oo_sl);
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(of[ks].v));
#endif
    float s = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int e = 0; e < 8; ++e) s = fmaf((float)bf[ks].v[e], (float)of[ks].v[e], s);
    // (stored after the tile loop: a store in flight would be waited for with the first tile's copies)
    const float row_delta = with_lane_xor<32, 64>(s, [](float a, float b) { return a + b; });

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

    // ---- tile walker (see attention.hip): 1 KiB copy blocks, block q = tile rows q*RPI .., wavefront w issues blocks
    // w, w+4, ...; lane i supplies physical chunk i of the block, which holds the logical chunk the swizzle assigns ----
    auto position_row = [&](const SegPlan& pl, int j) { return min(max(pl.c0 + pl.cs * j, 0), L - 1); };
    auto issue_tile_general = [&](const SegPlan& pl, int tile, int stage) {
        const int j0 = tile * BN;
        char* xs_w = smem + stage * STAGE;
        char* ys_w = xs_w + TILE;
        dma_tile<T, ROWB, BN, 3>(xs_w, wave, lane, [&](int row) { return xb + (int64_t)position_row(pl, j0 + row) * p.x_sl; });
        dma_tile<T, ROWB, BN, 3>(ys_w, wave, lane, [&](int row) { return yb + (int64_t)position_row(pl, j0 + row) * p.y_sl; });
    };
    uint32_t x_lane_off = 0, y_lane_off = 0;
    bool lane_off_fits = true;
    const char* x_next = nullptr;
    const char* y_next = nullptr;
    int64_t x_key = 0, y_key = 0;  // bytes from one tile position to the next
    auto set_lane_offsets = [&](const SegPlan& pl) {
        const int r = lane / CPR, pc = lane % CPR;
        const int lc = logical_chunk<ROWB, 3>(wave * RPI + r, pc);
        const int64_t x_far = (int64_t)pl.cs * (RPI - 1) * p.x_sl * ES + ROWB, y_far = (int64_t)pl.cs * (RPI - 1) * p.y_sl * ES + ROWB;
        lane_off_fits = x_far < ((int64_t)1 << 32) && y_far < ((int64_t)1 << 32);
        x_key = (int64_t)p.x_sl * ES * pl.cs;
        y_key = (int64_t)p.y_sl * ES * pl.cs;
        x_lane_off = (uint32_t)(x_key * r) + lc * 16;
        y_lane_off = (uint32_t)(y_key * r) + lc * 16;
        x_next = reinterpret_cast<const char*>(xb) + (int64_t)pl.c0 * p.x_sl * ES + (int64_t)wave * RPI * x_key;
        y_next = reinterpret_cast<const char*>(yb) + (int64_t)pl.c0 * p.y_sl * ES + (int64_t)wave * RPI * y_key;
    };
    auto tile_is_fast = [&](const SegPlan& pl, int tile) {
        const int j0 = tile * BN;
        // every position of the tile exists (the first one too: a walk may begin left of column 0)
        return lane_off_fits && pl.c0 + pl.cs * j0 >= 0 && pl.c0 + pl.cs * (j0 + BN - 1) < L;
    };
    auto issue_step = [&](int i, int stage) {
        char* xs_w = smem + stage * STAGE;
        char* ys_w = xs_w + TILE;
        if (i < NI)
            dma16_uniform(x_next + (int64_t)(4 * RPI * i) * x_key, x_lane_off, xs_w + (wave + 4 * i) * 1024);
        else
            dma16_uniform(y_next + (int64_t)(4 * RPI * (i - NI)) * y_key, y_lane_off, ys_w + (wave + 4 * (i - NI)) * 1024);
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

    // ---- LDS read addresses of stage 0; the stage offset is added once per tile ----
    const uint32_t smem_base = lds_address(smem);
    const int tr_row = (lane & 15) >> 2;
    const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);  // element column inside a 32-element block
    // One register each: the swizzle XORs the chunk with bits of the row, so that contraction step ks flips bits 5 .. of the address,
    // feature block dt bits 6 .., and 8 rows on bit 5 (rows 32 on, in the second half of a tile, have the same pattern); Y lies TILE further.
    auto dual_off = [&](int row, int byte_col) { return row * ROWB + dual_chunk<ROWB>(row, byte_col >> 4) * 16 + (byte_col & 15); };
    uint32_t xr_addr = smem_base + dual_off(lm, 8 * g * ES);
    uint32_t tr_addr = smem_base + dual_off(4 * g + tr_row, tr_col * ES);
    // fragment ks of the tile's rows 32 nt .. (row lm of them): of X at `from` = 0, of Y at TILE
    auto row_frag = [&](int ks, int nt, int from) {
        Frag<T> f;
        f.v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128((xr_addr ^ (32u * ks)) + (from + 32 * nt * ROWB)));
        return f;
    };
    // X's transpose: 16 positions from 16 * step on, features 32 dt ..
    auto tr_frag = [&](int step, int dt) {
        const uint32_t at = tr_addr ^ (64u * dt);
        return frag_from_tr<T>(lds_load_tr16(at + 16 * step * ROWB), lds_load_tr16((at ^ 32u) + (16 * step + 8) * ROWB));
    };

    // ---- first tile's copies, accumulators ----
    pf_seg = 0;
    pf_enter_segment();
    PlanRec win_rec = {0, 0, 1, 0};
    if (pf_seg < p.n_seg) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, pf_seg, wave * 32 + lm)];
    if (total_tiles > 0) {
        if (tile_is_fast(ppl, pf_tile)) {
#pragma unroll
            for (int s = 0; s < NDMA; ++s) issue_step(s, 0);
        } else {
            issue_tile_general(ppl, pf_tile, 0);
        }
        advance_fetch();
    }
    f32x16 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            acc[dt][j] = 0.f;
        }

    int cur_seg = -1, cur_tile = 0;
    RowWin win = {0, 0, 1};
    int first = 0, dec = 0;
    uint64_t pat = ~0ull;
    int w_lo_min = 0, w_lo_max = 0, w_hi_min = 0, w_hi_max = 0;
    SegPlan cpl = {0, 1, 0, 1};
    int stage_it = 0, stage_pf = 1;
#if defined(__HIP_DEVICE_COMPILE__)
    // the register operands are in their registers before the loop, so that no wait of the compiler's for them ends up
    // inside it, where it would also wait for the copies in flight
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(af[ks].v), "v"(bf[ks].v));
    asm volatile("" ::"v"(row_lse2), "v"(row_delta));
#endif

    for (int it = 0; it < total_tiles; ++it) {
        if (cur_seg < 0 || cur_tile >= cpl.n_tiles) {
            do {
                ++cur_seg;
                cpl = seg_plan_of(cur_seg);
            } while (cpl.n_tiles == 0);
            cur_tile = 0;
            if (it > 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur_seg, wave * 32 + lm)];
            win.lo = win_rec.x, win.cnt = win_rec.y, win.lin = win_rec.z;
            first = win_rec.w;
            const PlanRec r = plan_uniform_load(pt + plan_span_at(n_rb, p.n_seg, rb, cur_seg, wave));
            if (!cpl.uniform) {
                dec = BN % win.lin;
                uint64_t pt_bits = 0;
                for (int q = 0; q < 64; q += win.lin) pt_bits |= 1ull << q;
                pat = pt_bits;
            } else {
                pat = ~0ull;
            }
            w_lo_min = r.x, w_lo_max = r.y, w_hi_min = r.z, w_hi_max = r.w;
            asm volatile("v_mov_b32 %0, %0" : "+v"(w_lo_min));
            asm volatile("v_mov_b32 %0, %0" : "+v"(w_lo_max));
            asm volatile("v_mov_b32 %0, %0" : "+v"(w_hi_min));
            asm volatile("v_mov_b32 %0, %0" : "+v"(w_hi_max));
        }
        const int j0 = cur_tile * BN;
        ++cur_tile;

        // this wavefront's copies of tile `it` have landed; after the barrier everybody's have, and everybody is done
        // with tile it - 1, whose stage the next fetch overwrites
        wait_loads<0>();
        __builtin_amdgcn_s_barrier();

        const bool fetch = (it + 1 < total_tiles);
        bool spread = false;
        if (fetch) {
            spread = tile_is_fast(ppl, pf_tile);
            if (!spread) issue_tile_general(ppl, pf_tile, stage_pf);
        }

        const bool skip = (j0 + BN <= w_lo_min) || (j0 >= w_hi_max);
        if (!skip) {
            const bool full = (j0 >= w_lo_max) && (j0 + BN <= w_hi_min);
            const uint64_t live = full ? ~0ull : row_live_bits(win, j0, first, pat);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                static_assert(NDMA <= KS, "the first half issues all copies");
                // half a tile that holds nothing for this wavefront, as at the ends of most spans (bfloat16, 64 heads of 4096, the
                // whole step: window 65 at d = 64 131 -> 123 us, 33 at d = 128 257 -> 252)
                if (nt == 0 ? j0 + 32 <= w_lo_min : j0 + 32 >= w_hi_max) {
                    if (nt == 0 && spread) {
#pragma unroll
                        for (int s = 0; s < NDMA; ++s) issue_step(s, stage_pf);
                    }
                    continue;
                }
                // ---- S^T (32 positions x 32 rows) = X rows . A^T; Y's fragments take the places of X's ----
                f32x16 s_acc, dp;
#pragma unroll
                for (int j = 0; j < 16; ++j) s_acc[j] = 0.f, dp[j] = 0.f;
                Frag<T> xfr[KS], yfr[KS];
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) xfr[ks] = row_frag(ks, nt, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    mma32(s_acc, xfr[ks], af[ks]);
                    yfr[ks] = row_frag(ks, nt, TILE);
                    // the copy instructions of the next tile go between these MFMAs
                    const int step = nt * KS + ks;  // 0 .. 2*KS - 1
                    if (step < NDMA && spread) issue_step(step, stage_pf);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (!(j0 + 32 * nt >= w_lo_max && j0 + 32 * nt + 32 <= w_hi_min)) mask_half(s_acc, (uint32_t)(live >> (32 * nt)) >> (4 * g));
                // ---- dP^T = Y rows . B^T, and between its matrix instructions P^T = exp2(S^T * scale*log2e - lse*log2e); masked scores
                // underflow to exactly 0 ----
                constexpr int EPM = 16 / KS;  // elements per matrix instruction
                Frag<T> tf[2][DT];
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    mma32(dp, yfr[ks], bf[ks]);
#pragma unroll
                    for (int i = 0; i < EPM; ++i) {
                        const int j = EPM * ks + i;
                        s_acc[j] = fast_exp2(fmaf(s_acc[j], c2, -row_lse2));
                    }
                    if (ks >= KS - DT) tf[0][ks - (KS - DT)] = tr_frag(2 * nt, ks - (KS - DT));
                    __builtin_amdgcn_sched_barrier(0);
                }
                // ---- dS^T = P^T * (dP^T - D) * scale, eight positions' worth of registers ahead of acc^T (d x 32 rows) += X^T . dS^T ----
                Frag<T> pf[2];  // the second product's B operand: 16 positions each
                auto d_score = [&](int j) { pf[j >> 3].v[j & 7] = (T)(s_acc[j] * (dp[j] - row_delta) * p.scale); };
#pragma unroll
                for (int j = 0; j < 8; ++j) d_score(j);
#pragma unroll
                for (int t = 0; t < 2; ++t) {
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) {
                        mma32(acc[dt], tf[t][dt], pf[t]);
                        if (t == 0) {
                            tf[1][dt] = tr_frag(2 * nt + 1, dt);
#pragma unroll
                            for (int i = 0; i < 8 / DT; ++i) d_score(8 + 8 / DT * dt + i);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        } else if (spread) {
#pragma unroll
            for (int s = 0; s < NDMA; ++s) issue_step(s, stage_pf);
        }

        if (fetch) {
            advance_fetch();
            stage_pf ^= 1;
        }
        if (!cpl.uniform) {
            const int f = first - dec;
            first = f < 0 ? f + win.lin : f;
        }
        stage_it ^= 1;
        const int delta_b = stage_it == 0 ? -STAGE : STAGE;
        xr_addr += delta_b;
        tr_addr += delta_b;
    }
    // every wavefront has finished reading the last tile before the stages are reused for the output
    wait_loads<0>();
    __syncthreads();

    if (g == 0 && r0 + rs * (wave * 32 + lm) < L) p.delta_w[(int64_t)bh * L + my_row] = row_delta;

    // ---- epilogue: out = acc^T transposed through LDS, whole rows per store (each wavefront through a stretch of its own) ----
    {
        constexpr int OROW = D * ES + 16;
        static_assert(4 * 32 * OROW <= 2 * STAGE, "staging space");
        char* stg = smem + wave * (32 * OROW);
        auto store_rows = [&](const f32x16 (&a)[DT], T* dst) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    typedef T vec4 __attribute__((ext_vector_type(4)));
                    vec4 o;
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = (T)a[dt][4 * jj + i];
                    *reinterpret_cast<vec4*>(stg + lm * OROW + (32 * dt + 8 * jj + 4 * g) * ES) = o;
                }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            constexpr int OCPR = D * ES / 16;
#pragma unroll
            for (int i = 0; i < 32 * OCPR / 64; ++i) {
                const int flat = i * 64 + lane;
                const int row = flat / OCPR, c = flat % OCPR;
                const int r = r0 + rs * (wave * 32 + row);
                const u32x4 val = *reinterpret_cast<const u32x4*>(stg + row * OROW + c * 16);
                if (r < L) __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(reinterpret_cast<char*>(dst + (int64_t)r * p.o_sl) + c * 16));
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (read out before the stretch is written again)
        };
        store_rows(acc, ob);
    }
}

template <typename T, int D>
static int launch_bwd(BwdParams p, hipStream_t st) {
    begin_launch();
    constexpr int LDS_BYTES = 2 * (2 * 64 * D * 2);  // two stages of two tiles
    p.total = p.B * p.H * p.n_row_blocks;
    p.by_blocks = divisor(p.n_row_blocks), p.by_h = divisor(p.H);
    const int grid = ((p.total + 7) / 8) * 8;
    auto kern = attn_bwd_kernel<T, D>;
    static uint64_t lds_reserved = 0;
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), LDS_BYTES, "splat_attention_bwd")) return rc;
    kern<<<grid, 256, LDS_BYTES, st>>>(p);
    return check_launch("splat_attention_bwd");
}

// Adds the shares of listed rows onto the gradients of their keys: row k of every stretch (rows k + rps * s of the share
// buffers, [B*H, n_rows, D]) belongs to key key_of_row[k] (negative: padding).  One thread takes 8 features of one listed
// key of one (b, h) and one gradient (blockIdx.y: dk, dv), eight stretches' shares requested at a time, summing in fp32
// and rounding once.
template <typename T, int D>
__global__ __launch_bounds__(256) void bwd_rows_add_kernel(const T* __restrict__ dk_rows, const T* __restrict__ dv_rows, T* dk, T* dv,
                                                           const int* __restrict__ key_of_row, int n_rows, int rps, int L, int64_t total) {
    constexpr int CPR = D / 8;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int c = (int)(idx % CPR);
    const int64_t r = idx / CPR;
    const int k = (int)(r % rps);
    const int64_t bh = r / rps;
    const int key = key_of_row[k];
    if (key < 0 || key >= L) return;
    const int n_stretches = n_rows / rps;
    const T* rows = (blockIdx.y ? dv_rows : dk_rows) + ((int64_t)bh * n_rows + k) * D + 8 * c;
    T* out = (blockIdx.y ? dv : dk) + ((int64_t)bh * L + key) * D + 8 * c;
    Frag<T> cur = global_frag<T>(out);
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = (float)cur.v[e];
    for (int st = 0; st < n_stretches; st += 8) {
        Frag<T> f[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) f[u] = global_frag<T>(rows + (int64_t)min(st + u, n_stretches - 1) * rps * D);  // (unconditional)
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float w = st + u < n_stretches ? 1.f : 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] = fmaf(w, (float)f[u].v[e], acc[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) cur.v[e] = (T)acc[e];
    *reinterpret_cast<typename Frag<T>::vec*>(out) = cur.v;
}

template <typename T>
static int launch_rows_add(const void* dk_rows, const void* dv_rows, void* dk, void* dv, const int* key_of_row, int B, int H, int L,
                           int n_rows, int rps, int d, hipStream_t st) {
    begin_launch();
    const int64_t total = (int64_t)B * H * rps * (d / 8);
    const int64_t blocks = (total + 255) / 256;
    if (blocks > 0x7ffffff0) return fail(SPLAT_E_SHAPE, "splat_attention_bwd_keys: too many listed rows");
    if (d == 64)
        bwd_rows_add_kernel<T, 64><<<dim3((unsigned)blocks, 2), 256, 0, st>>>((const T*)dk_rows, (const T*)dv_rows, (T*)dk, (T*)dv, key_of_row, n_rows, rps, L, total);
    else
        bwd_rows_add_kernel<T, 128><<<dim3((unsigned)blocks, 2), 256, 0, st>>>((const T*)dk_rows, (const T*)dv_rows, (T*)dk, (T*)dv, key_of_row, n_rows, rps, L, total);
    return check_launch("splat_attention_bwd_keys");
}

template <typename T>
static int run_bwd(const BwdParams& dq, const BwdParams& dkv, int d, hipStream_t st) {
    if (int rc = d == 64 ? launch_bwd<T, 64>(dq, st) : launch_bwd<T, 128>(dq, st)) return rc;
    return launch_bwd_pair<T>(dkv, d, st);
}

struct Rows3 {
    const void* ptr;
    int64_t sb, sh, sl;
};

// Checks shared by the two entry points; `who` names the caller in messages.
static int check_bwd_common(const char* who, bool f32, int B, int H, int L, int d, float scale, int dtype, std::initializer_list<Rows3> rows,
                            std::initializer_list<const void*> aligned16) {
    if (B <= 0 || H <= 0 || L <= 0) return fail(SPLAT_E_SHAPE, "%s: need B, H, L > 0 (got %d, %d, %d)", who, B, H, L);
    if (L > (1 << 23)) return fail(SPLAT_E_SHAPE, "%s: L is limited to 2^23 (got %d)", who, L);
    if (d != 64 && d != 128) return fail(SPLAT_E_UNSUPPORTED, "%s: head dim must be 64 or 128 (got %d)", who, d);
    if (!f32 && dtype != SPLAT_F16 && dtype != SPLAT_BF16)
        return fail(SPLAT_E_UNSUPPORTED, "%s: 16-bit element types only (got dtype %d)", who, dtype);
    const int epc = f32 ? 4 : 8;
    if (!(scale > 0.f)) return fail(SPLAT_E_UNSUPPORTED, "%s: scale must be > 0 (got %g)", who, (double)scale);
    auto mis = [&](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) != 0; };
    for (const Rows3& r : rows) {
        if (mis(r.ptr)) return fail(SPLAT_E_ALIGN, "%s: every tensor of rows must be 16-byte aligned", who);
        if ((r.sb % epc) != 0 || (r.sh % epc) != 0 || (r.sl % epc) != 0)
            return fail(SPLAT_E_ALIGN, "%s: every batch/head/row stride must be a multiple of %d elements (16 bytes)", who, epc);
        if (r.sl < d) return fail(SPLAT_E_SHAPE, "%s: row strides must be >= d", who);
    }
    for (const void* ptr : aligned16)
        if (mis(ptr)) return fail(SPLAT_E_ALIGN, "%s: the gradients and the plans must be 16-byte aligned", who);
    return 0;
}

// The launches count their workgroups in an int: at most two a row block.
static bool too_many_blocks(int B, int H, int64_t row_blocks) { return 2 * (int64_t)B * H * row_blocks > 0x7ffffff0; }

static BwdParams bwd_base(const float* lse, const float* delta, int B, int H, int L, float scale) {
    BwdParams base;
    base.lse = lse; base.delta = delta;
    base.o = nullptr; base.oo_sb = base.oo_sh = base.oo_sl = 0; base.delta_w = nullptr; base.out2 = nullptr;
    base.B = B; base.H = H; base.L = L; base.Lr = L; base.row_map = nullptr;
    base.scale = scale; base.scale_log2e = scale * 1.4426950408889634f;
    return base;
}

// dK and dV (out2): rows = `Lk` keys, the plan of the (transposed) mask's `n_seg_t` segments
// for those rows; outputs contiguous [B, H, Lk, d]
static BwdParams bwd_keys_params(const BwdParams& base, Rows3 q, Rows3 k, Rows3 v, Rows3 g, void* dk, void* dv, const splat_acsr_seg* segs_t,
                                 int n_seg_t, const void* plan_t, int Lk, const int* row_map, int d) {
    BwdParams pk = base;
    pk.a = k.ptr; pk.a_sb = k.sb; pk.a_sh = k.sh; pk.a_sl = k.sl;
    pk.b = v.ptr; pk.b_sb = v.sb; pk.b_sh = v.sh; pk.b_sl = v.sl;
    pk.x = q.ptr; pk.x_sb = q.sb; pk.x_sh = q.sh; pk.x_sl = q.sl;
    pk.y = g.ptr; pk.y_sb = g.sb; pk.y_sh = g.sh; pk.y_sl = g.sl;
    pk.out = dk; pk.out2 = dv; pk.o_sb = (int64_t)base.H * Lk * d; pk.o_sh = (int64_t)Lk * d; pk.o_sl = d;
    pk.Lr = Lk; pk.row_map = row_map;
    pk.n_seg = n_seg_t; pk.row_stride = common_row_stride(segs_t, n_seg_t);
    pk.n_row_blocks = count_row_blocks(Lk, kPlanBM, pk.row_stride);
    pk.plan = static_cast<const PlanRec*>(plan_t);
    return pk;
}

}  // namespace splat

using namespace splat;

static int bwd_impl(const char* who, bool f32, const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* k, int64_t k_sb,
                                   int64_t k_sh, int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl,
                                   const void* out, int64_t o_sb, int64_t o_sh, int64_t o_sl, const void* dout, int64_t g_sb,
                                   int64_t g_sh, int64_t g_sl, const float* lse, float* delta, void* dq, void* dk, void* dv,
                                   const splat_acsr_seg* segs, int32_t n_seg, const void* plan, int64_t plan_bytes,
                                   const splat_acsr_seg* segs_t, int32_t n_seg_t, const void* plan_t, int64_t plan_t_bytes,
                                   int32_t B, int32_t H, int32_t L, int32_t d, float scale, int32_t dtype, void* stream) {
    if (!q || !k || !v || !out || !dout || !lse || !delta || !dq || !dk || !dv || !segs || !segs_t || !plan || !plan_t)
        return fail(SPLAT_E_NULL, "%s: null pointer argument", who);
    const Rows3 rq{q, q_sb, q_sh, q_sl}, rk{k, k_sb, k_sh, k_sl}, rv{v, v_sb, v_sh, v_sl}, ro{out, o_sb, o_sh, o_sl}, rg{dout, g_sb, g_sh, g_sl};
    if (int rc = check_bwd_common(who, f32, B, H, L, d, scale, dtype, {rq, rk, rv, ro, rg}, {dq, dk, dv, plan, plan_t})) return rc;
    if ((reinterpret_cast<uintptr_t>(lse) & 3) != 0 || (reinterpret_cast<uintptr_t>(delta) & 3) != 0)
        return fail(SPLAT_E_ALIGN, "%s: lse and delta must be 4-byte aligned", who);
    SegPtrs tmp[SPLAT_MAX_SEGMENTS];
    if (int rc = fill_segs(who, segs, n_seg, tmp, -1)) return rc;
    if (int rc = fill_segs(who, segs_t, n_seg_t, tmp, -1)) return rc;
    if (plan_bytes < splat_attention_plan_bytes(segs, n_seg, L) || plan_t_bytes < splat_attention_plan_bytes(segs_t, n_seg_t, L))
        return fail(SPLAT_E_SHAPE, "%s: a plan is smaller than its mask needs (%lld and %lld bytes given)", who, (long long)plan_bytes,
                    (long long)plan_t_bytes);
    if (too_many_blocks(B, H, std::max(count_row_blocks(L, kPlanBM, common_row_stride(segs, n_seg)),
                                       count_row_blocks(L, kPlanBM, common_row_stride(segs_t, n_seg_t)))))
        return fail(SPLAT_E_SHAPE, "%s: too many row blocks", who);
    hipStream_t st = (hipStream_t)stream;

    const BwdParams base = bwd_base(lse, delta, B, H, L, scale);
    // dQ: rows = queries, the mask's own plan
    BwdParams pq = base;
    pq.a = q; pq.a_sb = q_sb; pq.a_sh = q_sh; pq.a_sl = q_sl;
    pq.b = dout; pq.b_sb = g_sb; pq.b_sh = g_sh; pq.b_sl = g_sl;
    pq.x = k; pq.x_sb = k_sb; pq.x_sh = k_sh; pq.x_sl = k_sl;
    pq.y = v; pq.y_sb = v_sb; pq.y_sh = v_sh; pq.y_sl = v_sl;
    pq.out = dq; pq.o_sb = (int64_t)H * L * d; pq.o_sh = (int64_t)L * d; pq.o_sl = d;  // the gradients are contiguous [B, H, L, d]
    pq.n_seg = n_seg; pq.row_stride = common_row_stride(segs, n_seg);
    pq.n_row_blocks = count_row_blocks(L, kPlanBM, pq.row_stride);
    pq.plan = static_cast<const PlanRec*>(plan);
    pq.o = out; pq.oo_sb = o_sb; pq.oo_sh = o_sh; pq.oo_sl = o_sl; pq.delta_w = delta;  // D = rowsum(dO * O): computed and stored by this launch
    // dK, dV: rows = keys, the transposed mask's plan
    const BwdParams pk = bwd_keys_params(base, rq, rk, rv, rg, dk, dv, segs_t, n_seg_t, plan_t, L, nullptr, d);
    if (f32) {
        if (int rc = launch_bwd_dq_f32(pq, d, st)) return rc;
        return launch_bwd_dkv_f32(pk, d, st);
    }
    return dtype == SPLAT_F16 ? run_bwd<f16>(pq, pk, d, st) : run_bwd<bf16>(pq, pk, d, st);
}


static int bwd_keys_impl(const char* who, bool f32, const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* k, int64_t k_sb,
                                        int64_t k_sh, int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl,
                                        const void* dout, int64_t g_sb, int64_t g_sh, int64_t g_sl, const float* lse,
                                        const float* delta, const int32_t* key_of_row, void* dk_rows, void* dv_rows,
                                        const splat_acsr_seg* segs_t, int32_t n_seg_t, const void* plan_t, int64_t plan_t_bytes,
                                        int32_t B, int32_t H, int32_t L, int32_t n_rows, int32_t d, float scale, int32_t dtype,
                                        void* dk, void* dv, int32_t rows_per_stretch, void* stream) {
    if (!q || !k || !v || !dout || !lse || !delta || !key_of_row || !dk_rows || !dv_rows || !segs_t || !plan_t)
        return fail(SPLAT_E_NULL, "%s: null pointer argument", who);
    const Rows3 rq{q, q_sb, q_sh, q_sl}, rk{k, k_sb, k_sh, k_sl}, rv{v, v_sb, v_sh, v_sl}, rg{dout, g_sb, g_sh, g_sl};
    if (int rc = check_bwd_common(who, f32, B, H, L, d, scale, dtype, {rq, rk, rv, rg}, {dk_rows, dv_rows, plan_t})) return rc;
    if (n_rows <= 0 || n_rows > (1 << 23)) return fail(SPLAT_E_SHAPE, "%s: need 0 < n_rows <= 2^23 (got %d)", who, n_rows);
    if ((dk == nullptr) != (dv == nullptr)) return fail(SPLAT_E_NULL, "%s: dk and dv go together (both or neither)", who);
    if (dk) {
        if ((reinterpret_cast<uintptr_t>(dk) & 15) != 0 || (reinterpret_cast<uintptr_t>(dv) & 15) != 0)
            return fail(SPLAT_E_ALIGN, "%s: dk and dv must be 16-byte aligned", who);
        if (rows_per_stretch <= 0 || n_rows % rows_per_stretch != 0)
            return fail(SPLAT_E_SHAPE, "%s: n_rows (%d) must be a multiple of rows_per_stretch (%d)", who, n_rows, rows_per_stretch);
    }
    if ((reinterpret_cast<uintptr_t>(lse) & 3) != 0 || (reinterpret_cast<uintptr_t>(delta) & 3) != 0 ||
        (reinterpret_cast<uintptr_t>(key_of_row) & 3) != 0)
        return fail(SPLAT_E_ALIGN, "%s: lse, delta and key_of_row must be 4-byte aligned", who);
    SegPtrs tmp[SPLAT_MAX_SEGMENTS];
    if (int rc = fill_segs(who, segs_t, n_seg_t, tmp, -1)) return rc;
    if (plan_t_bytes < splat_attention_plan_bytes(segs_t, n_seg_t, n_rows))
        return fail(SPLAT_E_SHAPE, "%s: the plan is smaller than %d rows of this mask need (%lld bytes given)", who, n_rows,
                    (long long)plan_t_bytes);
    if (too_many_blocks(B, H, count_row_blocks(n_rows, kPlanBM, common_row_stride(segs_t, n_seg_t))))
        return fail(SPLAT_E_SHAPE, "%s: too many row blocks", who);
    const BwdParams base = bwd_base(lse, delta, B, H, L, scale);
    const BwdParams pk = bwd_keys_params(base, rq, rk, rv, rg, dk_rows, dv_rows, segs_t, n_seg_t, plan_t, n_rows, key_of_row, d);
    hipStream_t st = (hipStream_t)stream;
    if (f32) {
        if (int rc = launch_bwd_dkv_f32(pk, d, st)) return rc;
        return dk ? launch_rows_add<float>(dk_rows, dv_rows, dk, dv, key_of_row, B, H, L, n_rows, rows_per_stretch, d, st) : 0;
    }
    if (int rc = dtype == SPLAT_F16 ? launch_bwd_pair<f16>(pk, d, st) : launch_bwd_pair<bf16>(pk, d, st)) return rc;
    if (!dk) return 0;
    return dtype == SPLAT_F16 ? launch_rows_add<f16>(dk_rows, dv_rows, dk, dv, key_of_row, B, H, L, n_rows, rows_per_stretch, d, st)
                              : launch_rows_add<bf16>(dk_rows, dv_rows, dk, dv, key_of_row, B, H, L, n_rows, rows_per_stretch, d, st);
}

extern "C" int splat_attention_bwd(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* k, int64_t k_sb,
                                   int64_t k_sh, int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl,
                                   const void* out, int64_t o_sb, int64_t o_sh, int64_t o_sl, const void* dout, int64_t g_sb,
                                   int64_t g_sh, int64_t g_sl, const float* lse, float* delta, void* dq, void* dk, void* dv,
                                   const splat_acsr_seg* segs, int32_t n_seg, const void* plan, int64_t plan_bytes,
                                   const splat_acsr_seg* segs_t, int32_t n_seg_t, const void* plan_t, int64_t plan_t_bytes,
                                   int32_t B, int32_t H, int32_t L, int32_t d, float scale, int32_t dtype, void* stream) {
    return bwd_impl("splat_attention_bwd", false, q, q_sb, q_sh, q_sl, k, k_sb, k_sh, k_sl, v, v_sb, v_sh, v_sl, out, o_sb, o_sh, o_sl,
        dout, g_sb, g_sh, g_sl, lse, delta, dq, dk, dv, segs, n_seg, plan, plan_bytes, segs_t, n_seg_t, plan_t, plan_t_bytes, B, H, L,
        d, scale, dtype, stream);
}

extern "C" int splat_attention_bwd_f32(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* k, int64_t k_sb,
                                   int64_t k_sh, int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl,
                                   const void* out, int64_t o_sb, int64_t o_sh, int64_t o_sl, const void* dout, int64_t g_sb,
                                   int64_t g_sh, int64_t g_sl, const float* lse, float* delta, void* dq, void* dk, void* dv,
                                   const splat_acsr_seg* segs, int32_t n_seg, const void* plan, int64_t plan_bytes,
                                   const splat_acsr_seg* segs_t, int32_t n_seg_t, const void* plan_t, int64_t plan_t_bytes,
                                   int32_t B, int32_t H, int32_t L, int32_t d, float scale, void* stream) {
    return bwd_impl("splat_attention_bwd_f32", true, q, q_sb, q_sh, q_sl, k, k_sb, k_sh, k_sl, v, v_sb, v_sh, v_sl, out, o_sb, o_sh,
        o_sl, dout, g_sb, g_sh, g_sl, lse, delta, dq, dk, dv, segs, n_seg, plan, plan_bytes, segs_t, n_seg_t, plan_t, plan_t_bytes, B,
        H, L, d, scale, SPLAT_F32, stream);
}

extern "C" int splat_attention_bwd_keys(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* k, int64_t k_sb,
                                        int64_t k_sh, int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl,
                                        const void* dout, int64_t g_sb, int64_t g_sh, int64_t g_sl, const float* lse,
                                        const float* delta, const int32_t* key_of_row, void* dk_rows, void* dv_rows,
                                        const splat_acsr_seg* segs_t, int32_t n_seg_t, const void* plan_t, int64_t plan_t_bytes,
                                        int32_t B, int32_t H, int32_t L, int32_t n_rows, int32_t d, float scale, int32_t dtype,
                                        void* dk, void* dv, int32_t rows_per_stretch, void* stream) {
    return bwd_keys_impl("splat_attention_bwd_keys", false, q, q_sb, q_sh, q_sl, k, k_sb, k_sh, k_sl, v, v_sb, v_sh, v_sl, dout, g_sb,
        g_sh, g_sl, lse, delta, key_of_row, dk_rows, dv_rows, segs_t, n_seg_t, plan_t, plan_t_bytes, B, H, L, n_rows, d, scale, dtype,
        dk, dv, rows_per_stretch, stream);
}

extern "C" int splat_attention_bwd_keys_f32(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* k, int64_t k_sb,
                                        int64_t k_sh, int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl,
                                        const void* dout, int64_t g_sb, int64_t g_sh, int64_t g_sl, const float* lse,
                                        const float* delta, const int32_t* key_of_row, void* dk_rows, void* dv_rows,
                                        const splat_acsr_seg* segs_t, int32_t n_seg_t, const void* plan_t, int64_t plan_t_bytes,
                                        int32_t B, int32_t H, int32_t L, int32_t n_rows, int32_t d, float scale, void* dk, void* dv,
                                   int32_t rows_per_stretch, void* stream) {
    return bwd_keys_impl("splat_attention_bwd_keys_f32", true, q, q_sb, q_sh, q_sl, k, k_sb, k_sh, k_sl, v, v_sb, v_sh, v_sl, dout,
        g_sb, g_sh, g_sl, lse, delta, key_of_row, dk_rows, dv_rows, segs_t, n_seg_t, plan_t, plan_t_bytes, B, H, L, n_rows, d, scale,
        SPLAT_F32, dk, dv, rows_per_stretch, stream);
}

// Fused ACSR sparse-attention forward (online softmax), gfx950.
//
// A workgroup of 4 wavefronts owns 128 query rows of one (batch, head).  It walks the key range its
// rows' affine spans cover in tiles of BN keys.  Per tile:
//   * the K and V tiles are copied global -> LDS without passing through registers (LDS-DMA), into a
//     ring of NSTAGE stages: the copy of tile t + NSTAGE - 1 is issued while tile t is computed, piecewise
//     between its score MFMAs;
//   * every wavefront computes the TRANSPOSED score tile S^T = K . Q^T for its 32 rows with
//     32x32x16 MFMA (A = K fragment from LDS, B = Q fragment held in registers for the whole kernel).
//     In the transposed product one lane owns one query row, so masking, the running max and the
//     running sum need no cross-lane traffic beyond one exchange with the lane that holds the other
//     half of the row;
//   * P^T (the exponentials, converted to the input type) is already laid out as the B operand of
//     O^T += V^T . P^T, whose A operand (V^T fragments) is read from the row-major V tile in LDS with
//     the transposing LDS read (ds_read_b64_tr_b16); K^T tiles ([d, keys] input layout) use the same read.
// The compressed score matrix never exists in memory: traffic is Q + K + V + O.
//
// Which keys a tile holds is decided per workgroup from the rows' (a, lin, cnt) maps: if all rows
// share the column step and phase, tiles enumerate exactly those columns (key index c0 + cs*j,
// gathered rows of K/V) and validity is a per-row range test in j; otherwise tiles are dense columns
// and validity is the full affine test (offset, step divisibility, count).  Each wavefront skips tiles (d = 64: halves of tiles)
// that lie outside all of its rows' spans and drops the mask on tiles inside all of them.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "attn_tile.hpp"

namespace splat {

template <typename T, int D, bool KT, int BN, int NSTAGE, bool PLANNED>
__global__ __launch_bounds__(256, 2) void attn_fwd_kernel(const AttnParams p) {
    using G = TileGeom<T, D, KT, BN>;
    constexpr int ES = G::ES;
    static_assert(ES == 2, "16-bit element types (float32: attention_f32.hip)");
    constexpr int BM = 128;
    constexpr int KS = D / 16;  // contraction steps of the score product
    constexpr int DT = D / 32;  // 32-row tiles of O^T
    constexpr int NT = BN / 32;
    constexpr int PD = NSTAGE - 1;  // tiles whose copies run ahead of the tile being computed
    static_assert(NT == 1 || NT == 2, "tiles of 32 or 64 keys");
    static_assert(PD == 1 || PD == 3, "the wait ladder below covers 2 and 4 stages");

    extern __shared__ __attribute__((aligned(1024))) char smem[];
    __shared__ SegPlan s_plan[SPLAT_MAX_SEGMENTS];
    __shared__ PlanScratch<BM> s_ps;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 31, g = lane >> 5;

    load_args(p.total, p.n_row_blocks, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.H, p.row_stride, p.L, p.n_seg, p.plan, p.scale_log2e,
              p.q, p.q_sb, p.q_sh, p.q_sl, p.k, p.k_sb, p.k_sh, p.k_sd, p.k_sl, p.v, p.v_sb, p.v_sh, p.v_sl);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int bh = quotient(logical, p.by_blocks);
    // later row blocks of causal patterns carry the most keys: hand them out first
    const int rb = p.n_row_blocks - 1 - (logical - bh * p.n_row_blocks);
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride;
    const int r0 = block_first_row(rb, BM, rs);
    const int L = p.L;

    const T* qb = (const T*)p.q + b * p.q_sb + h * p.q_sh;
    const T* kb = (const T*)p.k + b * p.k_sb + h * p.k_sh;
    const T* vb = (const T*)p.v + b * p.v_sb + h * p.v_sh;
    T* ob = (T*)p.o + b * p.o_sb + h * p.o_sh;

    // ---- Q fragments (B operand of S^T), resident for the whole kernel; requested before the plan so that
    // their latency overlaps the metadata loads (the plan's barriers wait for both) ------------------------
    Frag<T> qf[KS];
    {
        const int my_row = r0 + rs * (wave * 32 + lm);
        const T* qr = qb + (int64_t)min(my_row, L - 1) * p.q_sl;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[ks] = global_frag<T>(qr + 16 * ks + 8 * g);
    }
    // ---- plan: per segment, the column range and step of this row block; computed here from the rows' maps or
    // taken from the mask's plan table (scalar loads: no LDS, no barrier) ------------------------
    static_assert(!PLANNED || (BM == kPlanBM && PD == 1), "the plan table is laid out for 128-row blocks");
    const PlanRec* const pt = p.plan;
    const int n_rb = p.n_row_blocks;
    auto seg_plan_of = [&](int sg) {
        SegPlan t;
        if constexpr (PLANNED) {
            const PlanRec r = plan_uniform_load(pt + plan_seg_at(p.n_seg, rb, sg));
            t.c0 = r.x, t.cs = r.y, t.n_tiles = r.z, t.uniform = r.w;
        } else {
            const SegPlan l = s_plan[sg];  // the same for every lane: keep it in scalar registers
            t.c0 = __builtin_amdgcn_readfirstlane(l.c0);
            t.cs = __builtin_amdgcn_readfirstlane(l.cs);
            t.n_tiles = __builtin_amdgcn_readfirstlane(l.n_tiles);
            t.uniform = __builtin_amdgcn_readfirstlane(l.uniform);
        }
        return t;
    };
    if constexpr (!PLANNED) plan_segments<BM, BN>(p.seg, p.n_seg, r0, rs, L, !KT, s_plan, &s_ps, tid);

    int total_tiles = 0;
    for (int sg = 0; sg < p.n_seg; ++sg) total_tiles += seg_plan_of(sg).n_tiles;
    total_tiles = __builtin_amdgcn_readfirstlane(total_tiles);

    // ---- tile walker: asynchronous global -> LDS copies of a tile into a stage -------------------------
    // A tile is copied as 1 KiB blocks, one wavefront instruction each; block q holds tile rows q*RPI.. and
    // wavefront w issues blocks w, w+4, ...  Lane i of a block supplies physical chunk i, i.e. (row i / CPR,
    // chunk position i % CPR), and loads the logical chunk the tile's swizzle assigns to that position.  That
    // assignment does not depend on the block, so a lane's source offset within a block is a per-segment
    // constant and the block's base is wavefront-uniform.
    constexpr int V_CPR = G::V_ROWB / 16, V_RPI = 1024 / G::V_ROWB;
    constexpr int K_CPR = G::K_ROWB / 16, K_RPI = 1024 / G::K_ROWB;
    constexpr int V_NI = BN * G::V_ROWB / 4096, K_NI = G::K_ROWS * G::K_ROWB / 4096;  // blocks per wavefront
    constexpr int NDMA = V_NI + K_NI;  // copy instructions per wavefront and tile, on every path
    static_assert(V_NI >= 1 && K_NI >= 1 && NDMA * (PD - 1) < 64, "tile shape");
    auto issue_tile_general = [&](const SegPlan& pl, int tile, int stage) {
        const int j0 = tile * BN;
        char* ks_w = smem + stage * G::STAGE;
        char* vs_w = ks_w + G::K_BYTES;
        auto key_row = [&](int row) { return min(max(pl.c0 + pl.cs * (j0 + row), 0), L - 1); };
        dma_tile<T, G::V_ROWB, BN, 2>(vs_w, wave, lane, [&](int row) { return vb + (int64_t)key_row(row) * p.v_sl; });
        if constexpr (KT) {
            // rows = contraction index, BN consecutive keys per row (dense walk); a chunk that would run past
            // the last key is replaced by the last whole chunk (those positions are never live)
#pragma unroll
            for (int i = 0; i < K_NI; ++i) {
                const int q = wave + 4 * i;
                const int flat = q * 64 + lane;
                const int row = flat / K_CPR, pc = flat % K_CPR;
                const int lc = logical_chunk<G::K_ROWB, 2>(row, pc);
                const int c = min(pl.c0 + j0 + lc * G::EPC, L - G::EPC);
                dma16(kb + (int64_t)row * p.k_sd + c, ks_w + q * 1024);
            }
        } else {
            dma_tile<T, G::K_ROWB, BN, 1>(ks_w, wave, lane, [&](int row) { return kb + (int64_t)key_row(row) * p.k_sl; });
        }
    };
    // State of the fast copies for the segment being fetched: per-lane byte offsets inside a block, wavefront-uniform
    // running pointers to block `wave` of the next tile, and the byte distance between tile positions.
    uint32_t v_lane_off = 0, k_lane_off = 0;
    bool lane_off_fits = true;  // the copy instruction takes a 32-bit per-lane offset: wider ones go the general way
    const char* v_next = nullptr;
    const char* k_next = nullptr;
    int64_t v_key = 0, k_key = 0;  // bytes from one tile position to the next (K^T layout: from one d row to the next)
    auto set_lane_offsets = [&](const SegPlan& pl) {
        const int vr = lane / V_CPR, vpc = lane % V_CPR;
        // the largest offsets of the segment: the last row of a block, with gathered rows pl.cs keys apart
        const int64_t v_far = (int64_t)pl.cs * (V_RPI - 1) * p.v_sl * ES + G::V_ROWB;
        const int64_t k_far = KT ? (int64_t)(K_RPI - 1) * p.k_sd * ES + G::K_ROWB : (int64_t)pl.cs * (K_RPI - 1) * p.k_sl * ES + G::K_ROWB;
        lane_off_fits = v_far < ((int64_t)1 << 32) && k_far < ((int64_t)1 << 32);
        v_lane_off = (uint32_t)((int64_t)pl.cs * vr * p.v_sl * ES) + logical_chunk<G::V_ROWB, 2>(vr, vpc) * 16;
        v_key = (int64_t)p.v_sl * ES * pl.cs;
        v_next = reinterpret_cast<const char*>(vb) + (int64_t)pl.c0 * p.v_sl * ES + (int64_t)wave * V_RPI * v_key;
        const int kr = lane / K_CPR, kpc = lane % K_CPR;
        if constexpr (KT) {
            k_lane_off = (uint32_t)((int64_t)kr * p.k_sd * ES) + logical_chunk<G::K_ROWB, 2>(kr, kpc) * 16;
            k_key = (int64_t)p.k_sd * ES;
            k_next = reinterpret_cast<const char*>(kb) + (int64_t)pl.c0 * ES + (int64_t)wave * K_RPI * k_key;
        } else {
            k_lane_off = (uint32_t)((int64_t)pl.cs * kr * p.k_sl * ES) +
                         logical_chunk<G::K_ROWB, 1>(wave * K_RPI + kr, kpc) * 16;
            k_key = (int64_t)p.k_sl * ES * pl.cs;
            k_next = reinterpret_cast<const char*>(kb) + (int64_t)pl.c0 * p.k_sl * ES + (int64_t)wave * K_RPI * k_key;
        }
    };
    // whether every key of the tile exists, so that the running pointers can be used as they are
    auto tile_is_fast = [&](const SegPlan& pl, int tile) {
        const int j0 = tile * BN;
        const int key_first = pl.c0 + pl.cs * j0, key_last = pl.c0 + pl.cs * (j0 + BN - 1);
        bool fast = lane_off_fits && key_last < L;
        if constexpr (KT) fast = fast && (key_first + BN <= L);
        return fast;
    };
    // copy instruction i (0 .. NDMA-1) of the tile the running pointers stand at
    auto issue_step = [&](int i, int stage) {
        char* ks_w = smem + stage * G::STAGE;
        char* vs_w = ks_w + G::K_BYTES;
        if (i < V_NI)
            dma16_uniform(v_next + (int64_t)(4 * V_RPI * i) * v_key, v_lane_off, vs_w + (wave + 4 * i) * 1024);
        else
            dma16_uniform(k_next + (int64_t)(4 * K_RPI * (i - V_NI)) * k_key, k_lane_off, ks_w + (wave + 4 * (i - V_NI)) * 1024);
    };

    int pf_seg = 0, pf_tile = 0;  // position of the next tile to fetch
    SegPlan ppl = {0, 1, 0, 1};
    // move on to the first segment at or after pf_seg that has tiles and take its plan into scalar registers
    auto pf_enter_segment = [&]() {
        pf_tile = 0;
        while (pf_seg < p.n_seg) {
            ppl = seg_plan_of(pf_seg);
            if (ppl.n_tiles > 0) break;
            ++pf_seg;
        }
        if (pf_seg < p.n_seg) set_lane_offsets(ppl);
    };
    // Tiles of a segment are fetched in order, so the running pointers advance by one tile per fetch; LDS is
    // only consulted at the end of a segment.
    auto advance_fetch = [&]() {
        v_next += BN * v_key;
        k_next += KT ? (int64_t)(BN * ES) : BN * k_key;
        if (++pf_tile >= ppl.n_tiles) {
            ++pf_seg;
            pf_enter_segment();
        }
    };
    f32x16 o_acc[DT];
    float m_ref = kNegBigA, l_run = 0.f;

    // ---- LDS read addresses: lane-dependent part + current stage; tile constants go into the instruction's
    // immediate offset; the stage offset is added once per tile -------------------------------------------
    const uint32_t smem_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    // transposing reads: lane s of a 16-lane block addresses row s/4, 8 bytes at element column 16*(block%2) + 4*(s%4)
    const int tr_row = (lane & 15) >> 2;
    const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    uint32_t k_addr[KT ? NT : KS];  // K tile: row-major: (row lm, swizzled chunk of step ks); K^T: (row 8g + tr_row, block nt)
    uint32_t v_addr[DT];            // V tile: (row 4g + tr_row, swizzled 64-byte block dt, column tr_col)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        v_addr[dt] = smem_base + G::K_BYTES + (4 * g + tr_row) * G::V_ROWB +
                     ((dt ^ swz64<G::V_ROWB>(4 * g + tr_row)) * 64) + tr_col * 2;
    if constexpr (KT) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            k_addr[nt] = smem_base + (8 * g + tr_row) * G::K_ROWB + ((nt ^ swz64<G::K_ROWB>(8 * g + tr_row)) * 64) + tr_col * 2;
    } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) k_addr[ks] = smem_base + lds_off<G::K_ROWB, true>(lm, (16 * ks + 8 * g) * ES);
    }

    // Two ways to take a tile's exponentials.  The careful one tracks the row maxima and moves the reference (with a
    // rescale of O and l) when they outrun it.  Once every row of the wavefront has a reference, the fast one leaves the
    // references where they are: no maxima, no exchange between the half rows, no data-dependent branch between the
    // score MFMAs and the exponentials.  That is exact as long as nothing overflows (float range for 32-bit and bf16
    // probabilities, 65504 for fp16 ones); if a later score outruns a row's reference by more than that, the row's sum
    // or output turns infinite or NaN and stays so, which is checked after the last tile, and the workgroup then
    // repeats its tiles on the careful path alone.
    bool careful_only = false;
    int stage_it = 0;  // stage that holds the tile being computed (the LDS read addresses stand at it)
    for (;;) {
        pf_seg = 0;
        pf_enter_segment();
        // the row windows of the first segment with tiles: requested here, long before the loop needs them
        PlanRec win_rec = {0, 0, 1, 0};
        if constexpr (PLANNED) {
            if (pf_seg < p.n_seg) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, pf_seg, wave * 32 + lm)];
        }
#pragma unroll
        for (int i = 0; i < PD; ++i) {
            if (i < total_tiles) {
                if (tile_is_fast(ppl, pf_tile)) {
#pragma unroll
                    for (int s = 0; s < NDMA; ++s) issue_step(s, (stage_it + i) % NSTAGE);
                } else {
                    issue_tile_general(ppl, pf_tile, (stage_it + i) % NSTAGE);
                }
                advance_fetch();
            }
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int j = 0; j < 16; ++j) o_acc[dt][j] = 0.f;
        m_ref = kNegBigA;
        l_run = 0.f;

        // per-lane row map of the segment being computed
        int cur_seg = -1, cur_tile = 0;
        RowWin win = {0, 0, 1};
        int first = 0, dec = 0;  // periodic part of the row mask of dense plans: see row_live_bits
        uint64_t pat = ~0ull;
        int w_lo_min = 0, w_lo_max = 0, w_hi_min = 0, w_hi_max = 0;
        SegPlan cpl = {0, 1, 0, 1};
        const float c2 = p.scale_log2e;
        bool settled = false;         // every row of this wavefront has a reference
        int stage_pf = (stage_it + PD) % NSTAGE;  // stage the next fetch goes to
        // The Q fragments have to be in their registers before the loop: otherwise the compiler puts its waits for them
        // in front of the first score MFMAs of every tile, counted against the loads it knows of, and those waits would
        // then hold for the copies of the next tile that are in flight at that point.
#if defined(__HIP_DEVICE_COMPILE__)  // the register constraint means something else to the host pass
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(qf[ks].v));
#endif

        for (int it = 0; it < total_tiles; ++it) {
            // advance the compute position; reload the row map on a segment change
            if (cur_seg < 0 || cur_tile >= cpl.n_tiles) {
                do {
                    ++cur_seg;
                    cpl = seg_plan_of(cur_seg);
                } while (cpl.n_tiles == 0);
                cur_tile = 0;
                WaveSpan sp;
                if constexpr (PLANNED) {
                    if (it > 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur_seg, wave * 32 + lm)];
                    win.lo = win_rec.x, win.cnt = win_rec.y, win.lin = win_rec.z;
                    first = win_rec.w;
                    const PlanRec r = plan_uniform_load(pt + plan_span_at(n_rb, p.n_seg, rb, cur_seg, wave));
                    sp.lo_min = r.x, sp.lo_max = r.y, sp.hi_min = r.z, sp.hi_max = r.w;
                } else {
                    win = make_row_win(cached_row_map<BM>(&s_ps, cur_seg, wave * 32 + lm), cpl);
                    first = cpl.uniform ? 0 : win_phase(win);
                    sp = wave_span(win, cpl.uniform != 0);
                }
                if (!cpl.uniform) {
                    // periodic part of the row's live positions (position 0 of the walk is column c0)
                    dec = BN % win.lin;
                    uint64_t pt_bits = 0;
                    for (int q = 0; q < 64; q += win.lin) pt_bits |= 1ull << q;
                    pat = pt_bits;
                } else {  // unit step: every position of the span
                    pat = ~0ull;
                }
                w_lo_min = sp.lo_min, w_lo_max = sp.lo_max, w_hi_min = sp.hi_min, w_hi_max = sp.hi_max;
                if constexpr (PLANNED) {
                    // keep the spans in vector registers, as the reductions of the other path leave them
                    asm volatile("v_mov_b32 %0, %0" : "+v"(w_lo_min));
                    asm volatile("v_mov_b32 %0, %0" : "+v"(w_lo_max));
                    asm volatile("v_mov_b32 %0, %0" : "+v"(w_hi_min));
                    asm volatile("v_mov_b32 %0, %0" : "+v"(w_hi_max));
                }
            }
            const int j0 = cur_tile * BN;
            ++cur_tile;

            // This wavefront's part of tile `it` has landed once at most the copies of the later tiles in flight
            // are outstanding; after the barrier every part has, and every wavefront is done with tile it - 1,
            // whose stage the next fetch overwrites.
            {
                const int later = total_tiles - 1 - it;
                if (PD == 1 || later == 0)
                    wait_loads<0>();
                else if (later == 1)
                    wait_loads<NDMA>();
                else
                    wait_loads<NDMA*(PD > 1 ? PD - 1 : 1)>();
            }
            __builtin_amdgcn_s_barrier();

            const bool fetch = (it + PD < total_tiles);
            bool spread = false;  // the fetch is issued piecewise between the matrix instructions below
            if (fetch) {
                spread = tile_is_fast(ppl, pf_tile);
                if (!spread) issue_tile_general(ppl, pf_tile, stage_pf);
            }

            // NP 32-key halves of the tile, from half `half` on
            auto compute = [&](auto parts, int half) __attribute__((always_inline)) {
                constexpr int NP = decltype(parts)::value;
                const bool full = (j0 >= w_lo_max) && (j0 + BN <= w_hi_min);
                const uint32_t k_half = NP < NT ? half * 32 * G::K_ROWB : 0, v_half = NP < NT ? half * 32 * G::V_ROWB : 0;
                // ---- S^T = K . Q^T ----
                // K fragments are requested from LDS a few MFMAs ahead of their use, never more than 12 read
                // instructions at a time: the counter that tracks them holds 15, and the compiler falls back to
                // waiting for every outstanding read once it could overflow.
                f32x16 s_acc[NP];
#pragma unroll
                for (int nt = 0; nt < NP; ++nt)
#pragma unroll
                    for (int j = 0; j < 16; ++j) s_acc[nt][j] = 0.f;
                Frag<T> kfr[NP][KS];
                auto load_k = [&](int nt, int ks) {
                    Frag<T> kf;
                    if constexpr (KT) {
                        // rows 16ks + 8g + {0..3} and +4: multiples of 4 rows leave the lane's swizzle term alone
                        const uint32_t a0 = (NP < NT && half ? k_addr[NT - 1] : k_addr[nt]) + 16 * ks * G::K_ROWB;
                        kf = frag_from_tr<T>(lds_load_tr16(a0), lds_load_tr16(a0 + 4 * G::K_ROWB));
                    } else {
                        kf.v = __builtin_bit_cast(typename Frag<T>::vec, lds_load128(k_addr[ks] + k_half + 32 * nt * G::K_ROWB));
                    }
                    return kf;
                };
                constexpr int NMMA = NP * KS;
                constexpr int K_AHEAD = (KT ? 6 : 12) < NMMA ? (KT ? 6 : 12) : NMMA;  // fragments
#pragma unroll
                for (int i = 0; i < K_AHEAD; ++i) kfr[i / KS][i % KS] = load_k(i / KS, i % KS);
                __builtin_amdgcn_sched_barrier(0);  // keep the requests above the matrix work
                // the copy instructions of the fetch go between the MFMAs, so that the address path sees them at
                // the rate it can take instead of as one burst that stalls the wavefront
                constexpr int MMA_PER_DMA = (NMMA / NDMA) > 0 ? NMMA / NDMA : 1;
#pragma unroll
                for (int i = 0; i < NMMA; ++i) {
                    mma32(s_acc[i / KS], kfr[i / KS][i % KS], qf[i % KS]);
                    if (i + K_AHEAD < NMMA) {
                        kfr[(i + K_AHEAD) / KS][(i + K_AHEAD) % KS] = load_k((i + K_AHEAD) / KS, (i + K_AHEAD) % KS);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if ((i + 1) % MMA_PER_DMA == 0 && (i + 1) / MMA_PER_DMA <= NDMA) {
                        if (spread) issue_step((i + 1) / MMA_PER_DMA - 1, stage_pf);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                if constexpr (NMMA / MMA_PER_DMA < NDMA) {
                    if (spread) {
#pragma unroll
                        for (int s = NMMA / MMA_PER_DMA; s < NDMA; ++s) issue_step(s, stage_pf);
                    }
                }
                // ---- mask, online softmax against a lazily updated reference ----
                Frag<T> pf[NP][2];
                if (!full) {
                    const uint64_t live = row_live_bits(win, j0, first, pat);
#pragma unroll
                    for (int nt = 0; nt < NP; ++nt) mask_half(s_acc[nt], (uint32_t)(live >> (32 * (half + nt))) >> (4 * g));
                }
                if (settled && !careful_only)
                    l_run += exp_tile<NP, T>(s_acc, pf, m_ref * c2, c2);
                else
                    settled = softmax_tile<NP, T, DT>(s_acc, pf, m_ref, l_run, o_acc, c2);

                // ---- O^T += V^T . P^T ----
                // V fragments are requested one 16-key step (DT fragments) ahead of the MFMAs that consume them.
                auto load_v = [&](int nt, int t, int dt) {
                    Frag<T> vf;
                    const uint32_t a0 = v_addr[dt] + v_half + (32 * nt + 16 * t) * G::V_ROWB;
                    vf = frag_from_tr<T>(lds_load_tr16(a0), lds_load_tr16(a0 + 8 * G::V_ROWB));
                    return vf;
                };
                Frag<T> vfr[2][DT];
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) vfr[0][dt] = load_v(0, 0, dt);
                __builtin_amdgcn_sched_barrier(0);  // keep the requests above the matrix work
#pragma unroll
                for (int step = 0; step < 2 * NP; ++step) {
                    const int nt = step >> 1, t = step & 1;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) {
                        mma32(o_acc[dt], vfr[step & 1][dt], pf[nt][t]);
                        if (step + 1 < 2 * NP) {
                            vfr[(step + 1) & 1][dt] = load_v((step + 1) >> 1, (step + 1) & 1, dt);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
            };
            // A wavefront of 32 rows ends its span in the middle of a tile as often as not.  Where half of a tile holds nothing
            // for it, that half is left out: 64 heads of 4096, d = 64, window 256, 44.6 -> 43.7 us, 256 keys with step 3
            // 39.1 -> 38.3, two segments 39.3 -> 38.3; a walk without such tiles takes no more tests than before.  Not at d = 128: the
            // second path's code costs its first fetch, 1 us of 50 at windows up to 64, against 1 % gained at 512.
            constexpr bool BY_HALVES = D == 64 && NT == 2;
            constexpr int NEAR = BY_HALVES ? BN / 2 : BN, FAR = BN - NEAR;
            if (j0 + NEAR > w_lo_min && j0 + FAR < w_hi_max) {
                compute(std::integral_constant<int, NT>{}, 0);
            } else if (BY_HALVES && j0 + BN > w_lo_min && j0 < w_hi_max) {
                if constexpr (BY_HALVES) compute(std::integral_constant<int, 1>{}, j0 + BN / 2 > w_lo_min ? 0 : 1);
            } else if (spread) {
#pragma unroll
                for (int s = 0; s < NDMA; ++s) issue_step(s, stage_pf);
            }

            if (fetch) {
                advance_fetch();
                stage_pf = (stage_pf + 1 == NSTAGE) ? 0 : stage_pf + 1;
            }
            if (!cpl.uniform) {  // phase of the periodic mask at the next tile
                const int f = first - dec;
                first = f < 0 ? f + win.lin : f;
            }
            // the next stage becomes current
            stage_it = (stage_it + 1 == NSTAGE) ? 0 : stage_it + 1;
            const int delta = (stage_it == 0) ? -(NSTAGE - 1) * G::STAGE : G::STAGE;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) v_addr[dt] += delta;
#pragma unroll
            for (int i = 0; i < (KT ? NT : KS); ++i) k_addr[i] += delta;
        }
        // Every copy has been waited for (the last tile waits for all).  The barrier in here also makes the stages free
        // for the epilogue (or the second pass): every wavefront has finished reading the last tile.
        const bool bad = !careful_only && (!(l_run < 1.0e30f) || !(fabsf(o_acc[0][0]) < 1.0e30f));
        if (!__syncthreads_or(bad ? 1 : 0)) break;
        careful_only = true;  // the ring goes on from the stage it stands at
    }

    // ---- epilogue: O = O^T / l, transposed through LDS so that every global store is a contiguous run --------
    {
        constexpr int OROW = D * ES + 16;  // padded row of the staging tile
        static_assert(4 * 32 * OROW <= NSTAGE * G::STAGE, "staging space");
        char* stg = smem + wave * (32 * OROW);
        const float l_tot = with_lane_xor<32, 64>(l_run, [](float a, float b) { return a + b; });
        const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
        if (p.lse != nullptr && g == 0) {
            // probabilities are exp(scale * score - lse); a row without live columns gets +inf (every probability 0)
            const int my_row = r0 + rs * (wave * 32 + lm);
            const float lse = l_tot > 0.f ? (m_ref * p.scale_log2e + __log2f(l_tot)) * 0.6931471805599453f : __builtin_inff();
            if (my_row < L) p.lse[(int64_t)bh * L + my_row] = lse;
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                typedef T vec4 __attribute__((ext_vector_type(4)));
                vec4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = (T)(o_acc[dt][4 * jj + i] * inv);
                *reinterpret_cast<vec4*>(stg + lm * OROW + (32 * dt + 8 * jj + 4 * g) * ES) = o;
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wavefront's LDS writes are visible to its own reads
        constexpr int CPR = D * ES / 16;                    // 16-byte chunks per output row
#pragma unroll
        for (int i = 0; i < 32 * CPR / 64; ++i) {
            const int flat = i * 64 + lane;
            const int row = flat / CPR, c = flat % CPR;
            const int r = r0 + rs * (wave * 32 + row);
            const u32x4 val = *reinterpret_cast<const u32x4*>(stg + row * OROW + c * 16);
            // non-temporal: whole aligned rows that this kernel never reads back, so they need not pass through the L2
            if (r < L) __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(reinterpret_cast<char*>(ob + (int64_t)r * p.o_sl) + c * 16));
        }
    }
}

template <typename T, int D, bool KT, int BN, int NSTAGE, bool PLANNED>
static int launch_attn(const AttnParams& p0, hipStream_t st) {
    begin_launch();
    using G = TileGeom<T, D, KT, BN>;
    AttnParams p = p0;
    constexpr int BM = 128;
    p.n_row_blocks = count_row_blocks(p.L, BM, p.row_stride);
    p.total = p.B * p.H * p.n_row_blocks;
    p.by_blocks = divisor(p.n_row_blocks), p.by_h = divisor(p.H);
    if (PLANNED && KT) p.plan += plan_variant_recs(p.n_row_blocks, p.n_seg);  // the dense-walk variant
    const int grid = ((p.total + 7) / 8) * 8;
    const size_t lds = NSTAGE * (size_t)G::STAGE;
    auto kern = attn_fwd_kernel<T, D, KT, BN, NSTAGE, PLANNED>;
    static uint64_t lds_reserved = 0;  // per instantiation: devices whose copy of this kernel has the limit raised
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), lds, "splat_attention_fwd")) return rc;
    kern<<<grid, 256, lds, st>>>(p);
    return check_launch("splat_attention_fwd");
}

// One 32-row tile per wavefront (128 rows per workgroup): 16-bit kernels then fit two workgroups per CU, whose
// wavefronts hide part of each other's LDS, barrier and prologue latency.  Tiles of 64 keys, double buffered (the
// kernel also supports 32-key tiles in a ring of 4 stages; it measured slower at d = 128 and equal at d = 64).
template <typename T>
static int dispatch_attn(const AttnParams& p, int d, bool kt, hipStream_t st) {
    // Few row blocks: the kernel whose wavefronts share the keys of 32 rows (attention_shared.hip), eight of them where every workgroup
    // has a CU to itself anyway, else four, two or four workgroups a CU.  It wins as long as its workgroups are on the chip together: 128
    // blocks at d = 128 (at 192 and window 200 11.9 -> 13.0 us), at d = 64 some 256, less for K^T and for walks that are live throughout.  bf16,
    // causal windows of 40 / 200 / 800, before -> with it: d = 64, 64 blocks 5.6 -> 4.6, 8.0 -> 5.1, 15.5 -> 6.7, 128 blocks 5.6 -> 4.9, 8.0 -> 5.7,
    // 15.5 -> 9.6, 192 blocks 6.7 -> 5.7, 9.9 -> 7.0, 17.6 -> 12.5, 256 blocks 6.8 -> 6.4, 10.1 -> 8.2, 17.7 -> 15.6 (blocks of 256 keys 7.8 -> 8.1, K^T and
    // window 101 8.0 -> 9.3); d = 128, 64 blocks 6.5 -> 5.2, 9.7 -> 6.4, 19.6 -> 8.9, 128 blocks 6.8 -> 6.3, 10.0 -> 7.9, 19.9 -> 13.7.  Eight
    // against four wavefronts, 64 blocks, windows 200 / 400 / 800: d = 64 5.1 / 5.9 / 6.7 against 4.9 / 6.2 / 8.0, d = 128 6.4 / 7.3 / 8.9 against
    // 6.3 / 8.1 / 10.5.
    const int64_t blocks = (int64_t)p.B * p.H * count_row_blocks(p.L, kPlanBM, p.row_stride);
    const bool narrow = std::max(p.v_sl, kt ? 0 : p.k_sl) * 2 < (1 << 24) && std::max(p.v_sl, kt ? 0 : p.k_sl) * 2 * p.L < ((int64_t)1 << 32);
    if (narrow && (blocks <= 128 || (d == 64 && p.live_percent > 0 && p.live_percent <= 90 && blocks <= (kt ? 192 : 224))))
        return launch_attn_shared<T>(p, d, kt, blocks <= 64 ? 8 : 4, st);
    // Some more: the kernel of 16 rows a wavefront (attention_rows16.hip), two workgroups per row block, which reads every operand from
    // LDS for half the rows: it wins where it skips masked positions and loses where there are none.  The line lies at three quarters of the
    // walked positions live and 320 (192 at d = 128) blocks: at 192 blocks, d = 64, windows 128 / 320 (half, 72 % live) 8.5 -> 7.7, 11.1 -> 10.5
    // us, window 512 (80 %) 13.9 -> 13.4, blocks of 256 (all) 11.4 -> 12.4; d = 128 10.4 -> 9.4, 13.9 -> 13.6, 17.5 -> 17.7, 14.4 -> 16.9; at 384
    // blocks, d = 64, window 256 with K^T along the keys 12.1 -> 12.4.  (Up to 128 blocks it is the faster one of the two whatever the mask,
    // for rows too far apart for the other's offsets.)
    if (blocks <= 128 || (p.live_percent > 0 && p.live_percent <= 75 && blocks <= (d == 64 ? 320 : 192)))
        return launch_attn_rows16<T>(p, d, kt, st);
    if (p.keys_anywhere) return fail(SPLAT_E_UNSUPPORTED, "splat_attention_fwd_keys: this launch copies K in whole 16-byte pieces");
    if (p.plan) {
        if (d == 64) return kt ? launch_attn<T, 64, true, 64, 2, true>(p, st) : launch_attn<T, 64, false, 64, 2, true>(p, st);
        return kt ? launch_attn<T, 128, true, 64, 2, true>(p, st) : launch_attn<T, 128, false, 64, 2, true>(p, st);
    }
    if (d == 64) return kt ? launch_attn<T, 64, true, 64, 2, false>(p, st) : launch_attn<T, 64, false, 64, 2, false>(p, st);
    return kt ? launch_attn<T, 128, true, 64, 2, false>(p, st) : launch_attn<T, 128, false, 64, 2, false>(p, st);
}

// One workgroup per (row block, variant): the same planning code the unplanned kernel runs in its prologue, with
// the results written to the table.
struct PlanParams {
    PlanRec* table;
    int4* report;  // may be null
    SegPtrs seg[SPLAT_MAX_SEGMENTS];
    int n_seg, L, rs, n_rb;
};
__global__ __launch_bounds__(256) void attn_plan_kernel(const PlanParams p) {
    constexpr int BM = kPlanBM, BN = 64;
    __shared__ SegPlan s_plan[SPLAT_MAX_SEGMENTS];
    __shared__ PlanScratch<BM> s_ps;
    __shared__ int s_misaligned, s_live;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lm = lane & 31;
    const int rb = blockIdx.x, variant = blockIdx.y;
    const int n_seg = p.n_seg, n_rb = p.n_rb;
    if (tid == 0) s_misaligned = 0, s_live = 0;  // (plan_segments has the barriers)
    PlanRec* const pt = p.table + variant * plan_variant_recs(n_rb, n_seg);
    plan_segments<BM, BN>(p.seg, n_seg, block_first_row(rb, BM, p.rs), p.rs, p.L, variant == 0, s_plan, &s_ps, tid);
    for (int sg = 0; sg < n_seg; ++sg) {
        const SegPlan pl = s_plan[sg];
        const RowWin win = make_row_win(cached_row_map<BM>(&s_ps, sg, wave * 32 + lm), pl);
        const WaveSpan sp = wave_span(win, pl.uniform != 0);
        if (tid == 0) pt[plan_seg_at(n_seg, rb, sg)] = PlanRec{pl.c0, pl.cs, pl.n_tiles, pl.uniform};
        if (lane == 0) pt[plan_span_at(n_rb, n_seg, rb, sg, wave)] = PlanRec{sp.lo_min, sp.lo_max, sp.hi_min, sp.hi_max};
        if (lane < 32)
            pt[plan_row_at(n_rb, n_seg, rb, sg, wave * 32 + lm)] = PlanRec{win.lo, win.cnt, win.lin, pl.uniform ? 0 : win_phase(win)};
        if (lane < 32 && win.cnt > 0) {
            if ((win.lo & 7) != 0) s_misaligned = 1;
            atomicAdd(&s_live, cached_row_map<BM>(&s_ps, sg, wave * 32 + lm).cnt);
        }
    }
    // what a host that waits for the plan learns with it, from the walks of the first variant
    if (p.report != nullptr && variant == 0) {
        __syncthreads();
        if (tid == 0) {
            int tiles = 0, stepping = 0;
            for (int sg = 0; sg < n_seg; ++sg) tiles += s_plan[sg].n_tiles, stepping |= s_plan[sg].uniform == 0;
            p.report[rb] = make_int4(s_misaligned, tiles, s_live, stepping);
        }
    }
}

}  // namespace splat

using namespace splat;

static int attention_fwd_common(const char* who, const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* kT,
                                int64_t k_sb, int64_t k_sh, int64_t k_sd, int64_t k_sl, const void* v, int64_t v_sb,
                                int64_t v_sh, int64_t v_sl, void* out, int64_t o_sb, int64_t o_sh, int64_t o_sl,
                                const splat_acsr_seg* segs, int32_t n_seg, int32_t B, int32_t H, int32_t L, int32_t d,
                                float scale, int32_t dtype, const void* plan, int64_t plan_bytes, bool planned,
                                float* lse, void* stream, int32_t live_percent = 0, bool keys_anywhere = false) {
    if (!q || !kT || !v || !out || !segs) return fail(SPLAT_E_NULL, "%s: null pointer argument", who);
    if (B <= 0 || H <= 0 || L <= 0) return fail(SPLAT_E_SHAPE, "%s: need B, H, L > 0 (got %d, %d, %d)", who, B, H, L);
    if (L > (1 << 23)) return fail(SPLAT_E_SHAPE, "%s: L is limited to 2^23 (got %d)", who, L);
    if (d != 64 && d != 128) return fail(SPLAT_E_UNSUPPORTED, "%s: head dim must be 64 or 128 (got %d)", who, d);
    if (dtype != SPLAT_F32 && dtype != SPLAT_F16 && dtype != SPLAT_BF16)
        return fail(SPLAT_E_DTYPE, "%s: unknown dtype %d", who, dtype);
    // the running max is taken over unscaled scores (needs scale >= 0) and masked scores are zeroed through
    // the underflow of exp2(-1e30 * scale) (needs scale > 0)
    if (!(scale > 0.f)) return fail(SPLAT_E_UNSUPPORTED, "%s: scale must be > 0 (got %g)", who, (double)scale);
    const int es = dtype == SPLAT_F32 ? 4 : 2;
    const int epc = 16 / es;
    bool kt;
    if (k_sd == 1 && (k_sl % epc) == 0 && k_sl >= d)
        kt = false;  // rows of K are contiguous: [.., L, d] memory viewed as [.., d, L]
    else if (k_sl == 1)
        kt = true;  // K^T contiguous: [.., d, L] memory
    else
        return fail(SPLAT_E_ALIGN, "%s: kT needs unit stride along d (k_sd == 1) or along keys (k_sl == 1); got k_sd=%lld k_sl=%lld", who,
                    (long long)k_sd, (long long)k_sl);
    if (keys_anywhere) {
        if (!kt || !planned || L < 8 || k_sd < L) return fail(SPLAT_E_UNSUPPORTED, "%s: needs a plan, at least 8 keys and rows of them", who);
        if ((reinterpret_cast<uintptr_t>(kT) & (es - 1)) != 0) return fail(SPLAT_E_ALIGN, "%s: kT is not aligned to its element size", who);
    }
    if (!keys_anywhere && kt && ((L % epc) != 0 || (k_sd % epc) != 0 || L < epc))
        return fail(SPLAT_E_ALIGN, "%s: with K^T contiguous along keys, L and the d-stride must be multiples of %d (got L=%d, k_sd=%lld)", who,
                    epc, L, (long long)k_sd);
    auto mis = [&](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) != 0; };
    auto bad = [&](int64_t s) { return (s % epc) != 0; };
    if (mis(q) || (mis(kT) && !keys_anywhere) || mis(v) || mis(out)) return fail(SPLAT_E_ALIGN, "%s: q, kT, v and out must be 16-byte aligned", who);
    if (bad(q_sb) || bad(q_sh) || bad(q_sl) || (!keys_anywhere && (bad(k_sb) || bad(k_sh))) || bad(v_sb) || bad(v_sh) || bad(v_sl) || bad(o_sb) || bad(o_sh) || bad(o_sl))
        return fail(SPLAT_E_ALIGN, "%s: every batch/head/row stride must be a multiple of %d elements (16 bytes)", who, epc);
    if (q_sl < d || v_sl < d || o_sl < d) return fail(SPLAT_E_SHAPE, "%s: row strides must be >= d", who);

    AttnParams p;
    p.q = q; p.k = kT; p.v = v; p.o = out;
    p.q_sb = q_sb; p.q_sh = q_sh; p.q_sl = q_sl;
    p.k_sb = k_sb; p.k_sh = k_sh; p.k_sd = k_sd; p.k_sl = k_sl;
    p.v_sb = v_sb; p.v_sh = v_sh; p.v_sl = v_sl;
    p.o_sb = o_sb; p.o_sh = o_sh; p.o_sl = o_sl;
    p.B = B; p.H = H; p.L = L;
    p.scale_log2e = scale * 1.4426950408889634f;
    p.n_seg = n_seg;
    if (int rc = fill_segs(who, segs, n_seg, p.seg, -1)) return rc;
    p.row_stride = common_row_stride(segs, n_seg);
    p.plan = nullptr;
    p.lse = lse;
    p.live_percent = live_percent, p.keys_anywhere = keys_anywhere;
    if (planned) {
        if (!plan) return fail(SPLAT_E_NULL, "%s: null plan", who);
        if ((reinterpret_cast<uintptr_t>(plan) & 15) != 0) return fail(SPLAT_E_ALIGN, "%s: the plan must be 16-byte aligned", who);
        const int64_t need = splat_attention_plan_bytes(segs, n_seg, L);
        if (plan_bytes < need)
            return fail(SPLAT_E_SHAPE, "%s: the plan holds %lld bytes, this mask needs %lld", who, (long long)plan_bytes, (long long)need);
        p.plan = static_cast<const PlanRec*>(plan);
    }
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case SPLAT_F32: return launch_attn_f32(p, d, kt, st);
        case SPLAT_F16: return dispatch_attn<f16>(p, d, kt, st);
        default: return dispatch_attn<bf16>(p, d, kt, st);
    }
}

extern "C" int splat_attention_fwd(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* kT, int64_t k_sb,
                                   int64_t k_sh, int64_t k_sd, int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh,
                                   int64_t v_sl, void* out, int64_t o_sb, int64_t o_sh, int64_t o_sl,
                                   const splat_acsr_seg* segs, int32_t n_seg, int32_t B, int32_t H, int32_t L, int32_t d,
                                   float scale, int32_t dtype, void* stream) {
    return attention_fwd_common("splat_attention_fwd", q, q_sb, q_sh, q_sl, kT, k_sb, k_sh, k_sd, k_sl, v, v_sb, v_sh, v_sl, out,
                                o_sb, o_sh, o_sl, segs, n_seg, B, H, L, d, scale, dtype, nullptr, 0, false, nullptr, stream);
}

extern "C" int splat_attention_fwd_planned(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* kT,
                                           int64_t k_sb, int64_t k_sh, int64_t k_sd, int64_t k_sl, const void* v,
                                           int64_t v_sb, int64_t v_sh, int64_t v_sl, void* out, int64_t o_sb, int64_t o_sh,
                                           int64_t o_sl, const splat_acsr_seg* segs, int32_t n_seg, int32_t B, int32_t H,
                                           int32_t L, int32_t d, float scale, int32_t dtype, const void* plan,
                                           int64_t plan_bytes, void* stream) {
    return attention_fwd_common("splat_attention_fwd_planned", q, q_sb, q_sh, q_sl, kT, k_sb, k_sh, k_sd, k_sl, v, v_sb, v_sh,
                                v_sl, out, o_sb, o_sh, o_sl, segs, n_seg, B, H, L, d, scale, dtype, plan, plan_bytes, true,
                                nullptr, stream);
}

extern "C" int splat_attention_fwd_stats(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* kT,
                                         int64_t k_sb, int64_t k_sh, int64_t k_sd, int64_t k_sl, const void* v,
                                         int64_t v_sb, int64_t v_sh, int64_t v_sl, void* out, int64_t o_sb, int64_t o_sh,
                                         int64_t o_sl, const splat_acsr_seg* segs, int32_t n_seg, int32_t B, int32_t H,
                                         int32_t L, int32_t d, float scale, int32_t dtype, const void* plan,
                                         int64_t plan_bytes, float* lse, void* stream) {
    const char* who = "splat_attention_fwd_stats";
    if (!lse) return fail(SPLAT_E_NULL, "%s: null lse", who);
    if ((reinterpret_cast<uintptr_t>(lse) & 3) != 0) return fail(SPLAT_E_ALIGN, "%s: lse must be 4-byte aligned", who);
    return attention_fwd_common(who, q, q_sb, q_sh, q_sl, kT, k_sb, k_sh, k_sd, k_sl, v, v_sb, v_sh, v_sl, out, o_sb, o_sh,
                                o_sl, segs, n_seg, B, H, L, d, scale, dtype, plan, plan_bytes, plan != nullptr, lse, stream);
}

extern "C" int splat_attention_fwd_hinted(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* kT,
                                          int64_t k_sb, int64_t k_sh, int64_t k_sd, int64_t k_sl, const void* v,
                                          int64_t v_sb, int64_t v_sh, int64_t v_sl, void* out, int64_t o_sb,
                                          int64_t o_sh, int64_t o_sl, const splat_acsr_seg* segs, int32_t n_seg, int32_t B,
                                          int32_t H, int32_t L, int32_t d, float scale, int32_t dtype, const void* plan,
                                          int64_t plan_bytes, float* lse, int32_t live_percent, void* stream) {
    const char* who = "splat_attention_fwd_hinted";
    if ((reinterpret_cast<uintptr_t>(lse) & 3) != 0) return fail(SPLAT_E_ALIGN, "%s: lse must be 4-byte aligned", who);
    if (live_percent < 0 || live_percent > 100) return fail(SPLAT_E_SHAPE, "%s: live_percent is %d", who, live_percent);
    return attention_fwd_common(who, q, q_sb, q_sh, q_sl, kT, k_sb, k_sh, k_sd, k_sl, v, v_sb, v_sh, v_sl, out, o_sb, o_sh,
                                o_sl, segs, n_seg, B, H, L, d, scale, dtype, plan, plan_bytes, plan != nullptr, lse, stream,
                                live_percent);
}

extern "C" int splat_attention_fwd_keys(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* kT,
                                        int64_t k_sb, int64_t k_sh, int64_t k_sd, const void* v,
                                        int64_t v_sb, int64_t v_sh, int64_t v_sl, void* out, int64_t o_sb,
                                        int64_t o_sh, int64_t o_sl, const splat_acsr_seg* segs, int32_t n_seg, int32_t B,
                                        int32_t H, int32_t L, int32_t d, float scale, int32_t dtype, const void* plan,
                                        int64_t plan_bytes, float* lse, int32_t live_percent, void* stream) {
    const char* who = "splat_attention_fwd_keys";
    if ((reinterpret_cast<uintptr_t>(lse) & 3) != 0) return fail(SPLAT_E_ALIGN, "%s: lse must be 4-byte aligned", who);
    if (live_percent < 0 || live_percent > 100) return fail(SPLAT_E_SHAPE, "%s: live_percent is %d", who, live_percent);
    return attention_fwd_common(who, q, q_sb, q_sh, q_sl, kT, k_sb, k_sh, k_sd, 1, v, v_sb, v_sh, v_sl, out, o_sb, o_sh,
                                o_sl, segs, n_seg, B, H, L, d, scale, dtype, plan, plan_bytes, plan != nullptr, lse, stream,
                                live_percent, true);
}

// ---- the forward for callers that cannot allocate: the plan lives in a file-scope device array ----------------
constexpr int64_t kStaticPlanBytes = SPLAT_STATIC_PLAN_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticPlanBytes];
// Host code must not use the array's name as an address: each device holds its own copy, whose address the runtime
// hands out.  Resolved once per device, with that device current.
static std::mutex g_scratch_lock;
static void* g_scratch_ptr[64] = {};
static int static_plan_buffer(const char* who, void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail((int)e, "%s: hipGetDevice: %s", who, hipGetErrorString(e));
    if (dev < 0 || dev >= 64) return fail(SPLAT_E_UNSUPPORTED, "%s: device ordinal %d is beyond the 64 this table holds", who, dev);
    std::lock_guard<std::mutex> guard(g_scratch_lock);
    if (g_scratch_ptr[dev] == nullptr) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || ptr == nullptr)
            return fail(e != hipSuccess ? (int)e : SPLAT_E_NULL, "%s: cannot resolve the plan buffer on device %d: %s", who, dev,
                        hipGetErrorString(e));
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

extern "C" int64_t splat_attention_plan_bytes(const splat_acsr_seg* segs, int32_t n_seg, int32_t L) {
    if (!segs || n_seg < 1 || n_seg > SPLAT_MAX_SEGMENTS || L <= 0) return 0;
    const int n_rb = count_row_blocks(L, kPlanBM, common_row_stride(segs, n_seg));
    return 2 * plan_variant_recs(n_rb, n_seg) * (int64_t)sizeof(PlanRec);
}

static int attention_plan_common(const char* who, const splat_acsr_seg* segs, int32_t n_seg, int32_t L, void* plan, int64_t plan_bytes,
                                 int32_t* report, void* stream) {
    begin_launch();
    if (!segs || !plan) return fail(SPLAT_E_NULL, "%s: null pointer argument", who);
    if (L <= 0 || L > (1 << 23)) return fail(SPLAT_E_SHAPE, "%s: need 0 < L <= 2^23 (got %d)", who, L);
    if ((reinterpret_cast<uintptr_t>(plan) & 15) != 0) return fail(SPLAT_E_ALIGN, "%s: the plan must be 16-byte aligned", who);
    PlanParams p;
    if (int rc = fill_segs(who, segs, n_seg, p.seg, -1)) return rc;
    const int64_t need = splat_attention_plan_bytes(segs, n_seg, L);
    if (plan_bytes < need)
        return fail(SPLAT_E_SHAPE, "%s: the plan needs %lld bytes for this mask, got %lld", who, (long long)need, (long long)plan_bytes);
    p.table = static_cast<PlanRec*>(plan);
    p.report = reinterpret_cast<int4*>(report);
    p.n_seg = n_seg;
    p.L = L;
    p.rs = common_row_stride(segs, n_seg);
    p.n_rb = count_row_blocks(L, kPlanBM, p.rs);
    attn_plan_kernel<<<dim3(p.n_rb, 2), 256, 0, (hipStream_t)stream>>>(p);
    return check_launch(who);
}

extern "C" int splat_attention_plan(const splat_acsr_seg* segs, int32_t n_seg, int32_t L, void* plan, int64_t plan_bytes,
                                    void* stream) {
    return attention_plan_common("splat_attention_plan", segs, n_seg, L, plan, plan_bytes, nullptr, stream);
}

extern "C" int splat_attention_plan_report(const splat_acsr_seg* segs, int32_t n_seg, int32_t L, void* plan, int64_t plan_bytes,
                                           int32_t* report, int64_t report_bytes, void* stream) {
    const char* who = "splat_attention_plan_report";
    if (!report) return fail(SPLAT_E_NULL, "%s: null report", who);
    if ((reinterpret_cast<uintptr_t>(report) & 15) != 0) return fail(SPLAT_E_ALIGN, "%s: the report must be 16-byte aligned", who);
    if (segs && n_seg >= 1 && n_seg <= SPLAT_MAX_SEGMENTS && L > 0 && L <= (1 << 23)) {  // (else refused below)
        const int64_t need = 16 * (int64_t)count_row_blocks(L, kPlanBM, common_row_stride(segs, n_seg));
        if (report_bytes < need)
            return fail(SPLAT_E_SHAPE, "%s: the report needs %lld bytes for this mask, got %lld", who, (long long)need, (long long)report_bytes);
    }
    return attention_plan_common(who, segs, n_seg, L, plan, plan_bytes, report, stream);
}

extern "C" int splat_attention_fwd_noalloc(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* kT,
                                           int64_t k_sb, int64_t k_sh, int64_t k_sd, int64_t k_sl, const void* v,
                                           int64_t v_sb, int64_t v_sh, int64_t v_sl, void* out, int64_t o_sb, int64_t o_sh,
                                           int64_t o_sl, const splat_acsr_seg* segs, int32_t n_seg, int32_t B, int32_t H,
                                           int32_t L, int32_t d, float scale, int32_t dtype, void* stream) {
    const char* who = "splat_attention_fwd_noalloc";
    if (!segs) return fail(SPLAT_E_NULL, "%s: null pointer argument", who);
    if (L <= 0 || L > (1 << 23)) return fail(SPLAT_E_SHAPE, "%s: need 0 < L <= 2^23 (got %d)", who, L);
    int64_t need = splat_attention_plan_bytes(segs, n_seg, L);
    if (need <= 0) return fail(SPLAT_E_SHAPE, "%s: no plan for n_seg=%d, L=%d", who, n_seg, L);
    // (rows grouped by phase round the row blocks up to a multiple of the stride: a mask that fits only without the hint goes without)
    splat_acsr_seg plain[SPLAT_MAX_SEGMENTS];
    if (need > kStaticPlanBytes && common_row_stride(segs, n_seg) > 1) {
        for (int k = 0; k < n_seg; ++k) plain[k] = segs[k], plain[k].row_stride_hint = 1;
        segs = plain;
        need = splat_attention_plan_bytes(segs, n_seg, L);
    }
    if (need > kStaticPlanBytes)
        return fail(SPLAT_E_SHAPE,
                    "%s: this mask's plan needs %lld bytes, the built-in buffer holds %lld (about %lld row blocks of 128 rows "
                    "times segments); use splat_attention_plan + splat_attention_fwd_planned with a buffer of your own",
                    who, (long long)need, (long long)kStaticPlanBytes,
                    (long long)(kStaticPlanBytes / (2 * plan_variant_recs(1, 1) * (int64_t)sizeof(PlanRec))));
    void* plan = nullptr;
    if (int rc = static_plan_buffer(who, &plan)) return rc;
    // the plan kernel rewrites every record this mask's forward reads, so nothing of an earlier call's plan is seen;
    // the forward follows on the same stream
    if (int rc = splat_attention_plan(segs, n_seg, L, plan, kStaticPlanBytes, stream)) return rc;
    return attention_fwd_common(who, q, q_sb, q_sh, q_sl, kT, k_sb, k_sh, k_sd, k_sl, v, v_sb, v_sh, v_sl, out, o_sb, o_sh, o_sl,
                                segs, n_seg, B, H, L, d, scale, dtype, plan, kStaticPlanBytes, true, nullptr, stream);
}

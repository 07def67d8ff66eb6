// The three operators of a forward in one kernel: 16-bit types, rows of at most 512 slots, inner dimension a multiple of 8 up to 128, with the mask's
// plan table.  Scores and probabilities are written as the separate operators write them, and read by nobody.
//
// Bound: the latency of dependent requests in small launches, the dense operands and the stores of the two compressed matrices in large ones.  As
// three launches (or two, where the sampled product's wavefronts take the softmax) scores are read once and probabilities twice; here a workgroup
// keeps its rows in LDS from the first product to the last.  bfloat16, causal masks, the separate launches -> this kernel, us: 64 heads of 4096 rows,
// d = 64, 64 slots 59 -> 45, 128 80 -> 62, 256 145 -> 96; d = 128, 256 slots 195 -> 130; 128 heads of 8192, d = 64, 256 slots 574 -> 416; 16 heads of
// 1024, d = 64, 40 slots 11.8 -> 9.1, 512 slots 35.6 -> 22.2; float16, 16 heads of 2000, 129 slots, d = 80 20.3 -> 17.2.
//
// A workgroup is 64 rows of one (batch, head) in two halves of 32, four wavefronts or, in launches of few workgroups, eight (16 heads of 1024
// rows, 200 slots, d = 64: 18.0 -> 14.2 us; 64 of 4096 119 -> 139).
//   Scores: S^T = K Q^T by 16x16x32 matrix instructions, the wavefronts of a half take turns at subtiles of 16 positions.  K goes through registers
//     into LDS a tile at a time, two tiles ahead, in the place of V's tiles, which is free until then; or from memory straight into the operands'
//     registers (kDirect): no barrier, but 16 lines a request and each of them twice.  That is faster for rows of up to 64 slots (64 heads of 4096 rows, 40
//     slots, d = 64 51.5 -> 47.0) and where eight wavefronts share few rows (16 heads of 1024, 16 slots 7.9 -> 7.5), slower for longer rows (128 heads of 8192, 200 slots
//     412 -> 438).  K stored along the keys is turned on its way into LDS.
//   Softmax: a wavefront's share of the rows, in the order of addition of softmax_rows; scores and probabilities leave from here in whole 16-byte
//     pieces.  (Held back until the output is there, so that no wait for V is a wait for them: no faster, and the registers are missed.)
//   Output: O^T = V^T P^T, V through registers into two stages, three tiles ahead, one barrier a tile; a wavefront has
//     32 rows and its share of the features (the operands, their order and so the bits of spmm_tile.hip).
//
// A row of LDS has room for PS slots, a power of two.  Blocks whose rows share the column step (a uniform plan) and are one segment keep a row by
// POSITION modulo PS, so that both products meet it in whole aligned pieces, and it is shifted to slots only for the softmax.  Other blocks
// (several segments, rows of different steps) keep it by slot; the products then write element by element and read shifted pieces.
// The pieces of 16 bytes are permuted by the row, so that 16 rows at one place cover all banks.
#include <algorithm>

#include "operators16.hpp"
#include "rows16.hpp"
#include "softmax_rows.hpp"
#include "spmm_params.hpp"

namespace splat {

namespace {

static_assert(kPlanBM == 2 * kHalfRows, "half a row block of the plan per workgroup");

// How K comes: from memory into operands, in rows through LDS, along the keys through LDS
enum { kDirect, kStaged, kAlongKeys };

// PS: slots that a row of LDS has room for; NW: wavefronts
template <int D, int PS, int NW>
struct Ops16Geom {
    static constexpr int VK = NW == 8 && D == 64 ? 64 : 32;      // keys of a tile of V
    static constexpr int STAGES = PS == 256 && D == 128 && NW == 4 ? 1 : 2;  // (one: four workgroups a CU)
    static constexpr int ROWB = D * 2, V_STAGE = VK * ROWB, P_ROWB = PS * 2;
    static constexpr int V_AT = kHalfRows * P_ROWB, LDS_BYTES = V_AT + STAGES * V_STAGE;
    static constexpr int O_ROW = ROWB + 16;
    // tiles of K take the place of V's: of 64 keys where that has room for them, two where it has room for two
    static constexpr int ROOM = STAGES * V_STAGE / ROWB, KK = ROOM < 64 ? ROOM : 64, K_STAGE = KK * ROWB, K_STAGES = ROOM / KK;
    static_assert(K_STAGES == 1 || K_STAGES == 2, "stages of K");
    static_assert(kHalfRows * O_ROW <= LDS_BYTES, "the output's turn-around");
};

// elements sh .. sh + 7 of the sixteen in a and b
__device__ __forceinline__ u32x4 window8(u32x4 a, u32x4 b, int sh) {
    const bool d2 = (sh & 4) != 0, d1 = (sh & 2) != 0;
    const uint32_t x0 = d2 ? a[2] : a[0], x1 = d2 ? a[3] : a[1], x2 = d2 ? b[0] : a[2], x3 = d2 ? b[1] : a[3], x4 = d2 ? b[2] : b[0], x5 = d2 ? b[3] : b[1];
    const uint32_t y0 = d1 ? x1 : x0, y1 = d1 ? x2 : x1, y2 = d1 ? x3 : x2, y3 = d1 ? x4 : x3, y4 = d1 ? x5 : x4;
    const uint32_t s = (sh & 1) * 16u;
    return u32x4{__builtin_amdgcn_alignbit(y1, y0, s), __builtin_amdgcn_alignbit(y2, y1, s), __builtin_amdgcn_alignbit(y3, y2, s),
                 __builtin_amdgcn_alignbit(y4, y3, s)};
}

// all ones in the 16-bit elements whose bit is set
__device__ __forceinline__ u32x4 spread8(uint32_t bits) {
    u32x4 m;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t lo = (uint32_t)((int32_t)(bits << (31 - 2 * i)) >> 31), hi = (uint32_t)((int32_t)(bits << (30 - 2 * i)) >> 31);
        m[i] = (lo & 0xffffu) | (hi & 0xffff0000u);
    }
    return m;
}

// minus infinity in both halves of a register
template <typename T>
constexpr uint32_t kMinusInf = std::is_same_v<T, f16> ? 0xfc00fc00u : 0xff80ff80u;

// bits of the elements u .. u + 7 that lie in [0, cnt)
__device__ __forceinline__ uint32_t inside8(int u, int cnt) {
    const int a = min(max(-u, 0), 8), b = min(max(cnt - u, 0), 8);
    return ((1u << b) - 1u) & ~((1u << a) - 1u);
}

// x of the lane before, of each group of LPR lanes in a ring
template <int LPR>
__device__ __forceinline__ uint32_t from_lane_before(uint32_t x, int lane) {
    if constexpr (LPR == 16) return __builtin_amdgcn_update_dpp(0, (int)x, 0x121, 0xf, 0xf, true);  // rotated by one among 16
    const int before = __builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, true);               // lane - 1
    const int last = __builtin_amdgcn_update_dpp(0, (int)x, 0x107, 0xf, 0xf, true);                 // lane + 7
    return (uint32_t)((lane & 7) == 0 ? last : before);
}

}  // namespace

template <typename T, int D, int PS, int KEYS, int NW>
__global__ __launch_bounds__(NW * 64, 4) void operators16_kernel(const Operators16Params p) {
    using G = Ops16Geom<D, PS, NW>;
    constexpr int VK = G::VK, GW = NW / 2, NT = NW * 64, ROWS_PW = kHalfRows / NW;  // GW: wavefronts that share 32 rows
    constexpr int ROWB = G::ROWB, V_STAGE = G::V_STAGE, P_ROWB = G::P_ROWB, O_ROW = G::O_ROW;
    constexpr int KS = D / 32, CPR = ROWB / 16, NI = VK * CPR / NT, FD = D / 16 / GW;
    constexpr int NC = PS / 8, LPR = PS == 64 ? 8 : 16, NCH = NC / LPR, RPW = 64 / LPR;  // chunks of a row, lanes a row, chunks a lane, rows at a time
    typedef T vec4 __attribute__((ext_vector_type(4)));
    typedef T vec8 __attribute__((ext_vector_type(8)));

    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, g = lane >> 4;
    const int pr = wave / GW, hw = wave % GW;  // which 32 rows, and the place among those that share them

    load_args(p.total, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.n_row_blocks, p.H, p.row_stride, p.L, p.n_keys, p.d, p.T, p.n_seg, p.plan,
              p.q, p.q_sb, p.q_sh, p.q_sl, p.k, p.k_sb, p.k_sh, p.k_sd, p.k_sl, p.v, p.v_sb, p.v_sh, p.v_sl, p.scale);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int per_head = 2 * p.n_row_blocks;
    const int bh = quotient(logical, p.by_blocks);
    const int at_block = per_head - 1 - (logical - bh * per_head);
    const int rb = at_block >> 1, half = at_block & 1;
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride, L = p.L, d = p.d, n_rb = p.n_row_blocks, n_seg = p.n_seg;
    const int r0 = block_first_row(rb, kPlanBM, rs) + rs * half * kHalfRows;
    if (r0 >= L) return;

    const T* const kb = (const T*)p.k + b * p.k_sb + h * p.k_sh;
    const char* const vbytes = reinterpret_cast<const char*>((const T*)p.v + b * p.v_sb + h * p.v_sh);
    const PlanRec* const pt = p.plan;
    const u32x4 zero = {0u, 0u, 0u, 0u};

    Frag<T> q[2][KS];  // B operands: rows 32 pr + 16 cb + li
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        const T* const qr = (const T*)p.q + b * p.q_sb + h * p.q_sh + (int64_t)min(r0 + rs * (32 * pr + 16 * cb + li), L - 1) * p.q_sl;
#pragma unroll
        for (int t = 0; t < KS; ++t) {
            q[cb][t].v = __builtin_bit_cast(typename Frag<T>::vec, zero);
            if (32 * t + 8 * g < d) q[cb][t] = global_frag<T>(qr + 32 * t + 8 * g);
        }
    }

    // ---- the rows of a pair in one segment ----
    struct Seg {
        int sg, off;
        SegPlan pl;
        RowWin win[2];
        WaveSpan span;
        bool by_position;  // how the rows lie in LDS
        bool apart;        // no two positions that the pair walks share a place there
    };
    struct Recs {  // of the plan table
        PlanRec seg, span0, span1;
    };
    auto recs_of = [&](int sg) {
        return Recs{plan_uniform_load(pt + plan_seg_at(n_seg, rb, sg)), plan_uniform_load(pt + plan_span_at(n_rb, n_seg, rb, sg, 2 * half)),
                    plan_uniform_load(pt + plan_span_at(n_rb, n_seg, rb, sg, 2 * half + 1))};
    };
    auto enter = [&](int sg, const Recs& rec) {
        Seg s;
        s.sg = sg;
        s.off = p.seg[sg].slot_offset;
        const PlanRec r = rec.seg, sp = pr ? rec.span1 : rec.span0;
        s.pl = SegPlan{r[0], r[1], r[2], r[3]};
        s.span = WaveSpan{sp[0], sp[1], sp[2], sp[3]};
        s.by_position = n_seg == 1 && s.pl.uniform != 0;
        s.apart = s.by_position && ((max(s.span.hi_max, 0) + 31) & ~31) - (s.span.lo_min & ~31) <= PS;
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const int k = 32 * pr + 16 * cb + li;
            const PlanRec w = pt[plan_row_at(n_rb, n_seg, rb, sg, half * kHalfRows + k)];
            // (the table knows the mask alone: a row's slots are bounded by the buffer's here, as load_row_map does)
            const int64_t most = s.pl.uniform ? (int64_t)p.seg[sg].max_cnt : (int64_t)w[2] * (p.seg[sg].max_cnt - 1) + 1;
            s.win[cb] = RowWin{w[0], r0 + rs * k < L ? (int)min((int64_t)w[1], most) : 0, w[2]};
        }
        return s;
    };
    auto place = [&](int row, int chunk) { return row * P_ROWB + (((chunk & (NC - 1)) ^ swz<P_ROWB>(row)) << 4); };

    // ---- scores ----
    auto put = [&](const Seg& s, int u, const f32x4(&acc)[2]) {
        const int j = 16 * u + 4 * g;  // the lane's first position
        const bool whole = s.apart || (s.by_position && 16 * u >= s.span.lo_max && 16 * u + 16 <= s.span.hi_min);
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const int row = 32 * pr + 16 * cb + li;
            vec4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = rounded<T>(acc[cb][e] * p.scale);
            if (s.by_position) {
                char* const to = smem + place(row, j >> 3) + (j & 4) * 2;
                if (whole) {
                    *reinterpret_cast<vec4*>(to) = x;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if ((unsigned)(j + e - s.win[cb].lo) < (unsigned)s.win[cb].cnt) *reinterpret_cast<T*>(to + 2 * e) = x[e];
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bool live = s.pl.uniform ? (unsigned)(j + e - s.win[cb].lo) < (unsigned)s.win[cb].cnt : win_live(s.win[cb], j + e);
                    if (live) {
                        const int slot = s.off + (s.pl.uniform ? j + e - s.win[cb].lo : win_slot(s.win[cb], j + e));
                        *reinterpret_cast<T*>(smem + place(row, slot >> 3) + (slot & 7) * 2) = x[e];
                    }
                }
            }
        }
    };
    auto products = [&](const Frag<T>(&k)[KS], f32x4(&acc)[2]) {
        acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < KS; ++t)
            if (D == 64 || 32 * t < d) mma16(acc[0], k[t], q[0][t]), mma16(acc[1], k[t], q[1][t]);
    };

    // position of a walk over tiles of VK positions, and the one after it
    auto walk_in = [&](auto keys, int sg, const Recs& rec) {
        constexpr int BN = decltype(keys)::value;
        HalfWalk w;
        w.seg = sg;
        w.pl = SegPlan{rec.seg[0], rec.seg[1], rec.seg[2], rec.seg[3]};
        w.tile = max(min(rec.span0[0], rec.span1[0]), 0) / BN;
        w.end = max(min((max(max(rec.span0[3], rec.span1[3]), 0) + BN - 1) / BN, w.pl.n_tiles * kBN / BN), w.tile);
        return w;
    };
    auto walk_from = [&](auto keys, int sg) {
        HalfWalk w;
        for (; sg < n_seg; ++sg) {
            w = walk_in(keys, sg, recs_of(sg));
            if (w.tile < w.end) return w;
        }
        w.seg = n_seg, w.tile = w.end = 0;
        return w;
    };
    auto first_walk = [&](auto keys, const Recs& rec) {
        const HalfWalk w = walk_in(keys, 0, rec);
        return w.tile < w.end ? w : walk_from(keys, 1);
    };
    auto advance = [&](auto keys, HalfWalk& w) {
        if (++w.tile >= w.end) w = walk_from(keys, w.seg + 1);
    };
    constexpr std::integral_constant<int, VK> v_keys{};
    constexpr std::integral_constant<int, G::KK> k_keys{};

    const Recs rec0 = recs_of(0);
    Seg s = enter(0, rec0);

    // ---- V: a thread's pieces of a tile, of which the first two are requested before the softmax ----
    int v_row[NI], v_col[NI], v_to[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int id = tid + NT * i;
        v_row[i] = id / CPR;
        v_col[i] = min(id % CPR, d / 8 - 1) * 16;  // (chunks past the last repeat it: what they add lands in columns that are not stored)
        v_to[i] = G::V_AT + v_row[i] * ROWB + v_chunk<ROWB>(v_row[i], id % CPR) * 16;
    }
    const int64_t v_rowb = p.v_sl * 2;
    auto load_v = [&](const HalfWalk& w, u32x4(&reg)[NI]) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int key = min(max(w.pl.c0 + w.pl.cs * (w.tile * VK + v_row[i]), 0), p.n_keys - 1);
            reg[i] = *reinterpret_cast<const u32x4*>(vbytes + key * v_rowb + v_col[i]);
        }
    };
    auto write_v = [&](int stage, const u32x4(&reg)[NI]) {
#pragma unroll
        for (int i = 0; i < NI; ++i) *reinterpret_cast<u32x4*>(smem + stage + v_to[i]) = reg[i];
    };
    const HalfWalk v_first = first_walk(v_keys, rec0);
    HalfWalk v_ahead = v_first;
    u32x4 va[NI], vb[NI];
    auto request_v = [&] {
        if (v_ahead.seg < n_seg) {
            load_v(v_ahead, va);
            advance(v_keys, v_ahead);
            if (v_ahead.seg < n_seg) load_v(v_ahead, vb);
        }
    };

    // ---- this wavefront's share of the rows in the softmax ----
    SoftmaxSegs segs;
    segs.n = n_seg;
#pragma unroll
    for (int k = 0; k < SPLAT_MAX_SEGMENTS; ++k) segs.nnz[k] = k < n_seg ? p.seg[k].nnz : p.seg[0].nnz, segs.off[k] = p.seg[k].slot_offset;
    const bool by_position = n_seg == 1 && rec0.seg[3] != 0;
    const int my = lane & (LPR - 1);
    LiveRanges lr;
    float cnt[ROWS_PW / RPW][SPLAT_MAX_SEGMENTS];
    int base[ROWS_PW / RPW];  // of slot 0, where rows lie by position
    auto request_counts = [&] {
#pragma unroll
        for (int it = 0; it < ROWS_PW / RPW; ++it) {
            const int k = ROWS_PW * wave + RPW * it + lane / LPR, r = r0 + rs * k;
            lr.request(segs, r < L ? r : r0);
#pragma unroll
            for (int i = 0; i < SPLAT_MAX_SEGMENTS; ++i) cnt[it][i] = lr.cnt[i];
            base[it] = by_position ? pt[plan_row_at(n_rb, n_seg, rb, 0, half * kHalfRows + k)][0] - segs.off[0] : 0;
        }
    };

    if constexpr (KEYS != kDirect) {
        // A thread's piece is 8 values of one key; lanes = pieces of a row, or keys
        constexpr int KK = G::KK, NP = KK * CPR / NT;
        int pc_key[NP], pc_c[NP], pc_to[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int f = tid + NT * i;
            pc_key[i] = KEYS == kAlongKeys ? f % KK : f / CPR, pc_c[i] = KEYS == kAlongKeys ? f / KK : f % CPR;
            pc_to[i] = G::V_AT + lds_off<ROWB, true>(pc_key[i], pc_c[i] * 16);
        }
        auto load_tile = [&](const HalfWalk& w, u32x4(&raw)[NP]) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int key = min(max(w.pl.c0 + w.pl.cs * (w.tile * KK + pc_key[i]), 0), p.n_keys - 1);
                raw[i] = zero;
                if (8 * pc_c[i] < d) {
                    if constexpr (KEYS == kAlongKeys) {
                        const T* const src = kb + (int64_t)(8 * pc_c[i]) * p.k_sd + (int64_t)key * p.k_sl;
                        Frag<T> f;
#pragma unroll
                        for (int e = 0; e < 8; ++e) f.v[e] = src[e * p.k_sd];
                        raw[i] = __builtin_bit_cast(u32x4, f.v);
                    } else {
                        raw[i] = *reinterpret_cast<const u32x4*>(kb + (int64_t)key * p.k_sl + 8 * pc_c[i]);
                    }
                }
            }
        };
        HalfWalk ahead = first_walk(k_keys, rec0), cur = ahead;
        u32x4 ra[NP], rb_[NP];
        if (ahead.seg < n_seg) {
            load_tile(ahead, ra);
            advance(k_keys, ahead);
            if (ahead.seg < n_seg) load_tile(ahead, rb_);
        }
        auto tile = [&](int stage, u32x4(&raw)[NP]) {
            if (cur.seg != s.sg) s = enter(cur.seg, recs_of(cur.seg));
#pragma unroll
            for (int i = 0; i < NP; ++i) *reinterpret_cast<u32x4*>(smem + stage + pc_to[i]) = raw[i];
            if (ahead.seg < n_seg) advance(k_keys, ahead);
            if (ahead.seg < n_seg) load_tile(ahead, raw);
            lds_barrier();  // the tile is there; of two stages, everybody is done with the one before it, whose stage comes next
#pragma unroll
            for (int i = 0; i < (KK / 16 + GW - 1) / GW; ++i) {
                const int in_tile = hw + GW * i, u = KK / 16 * cur.tile + in_tile;
                if (in_tile < KK / 16 && 16 * u + 16 > s.span.lo_min && 16 * u < s.span.hi_max) {
                    Frag<T> k[KS];
#pragma unroll
                    for (int t = 0; t < KS; ++t) k[t].v = __builtin_bit_cast(typename Frag<T>::vec,
                        *reinterpret_cast<const u32x4*>(smem + G::V_AT + stage + lds_off<ROWB, true>(16 * in_tile + li, (4 * t + g) * 16)));
                    f32x4 acc[2];
                    products(k, acc);
                    put(s, u, acc);
                }
            }
            if constexpr (G::K_STAGES == 1) lds_barrier();
            advance(k_keys, cur);
        };
        while (cur.seg < n_seg) {
            tile(0, ra);
            if (cur.seg < n_seg) tile(G::K_STAGES == 1 ? 0 : G::K_STAGE, rb_);
        }
    } else {
        for (int sg = 0; sg < n_seg; ++sg) {
            if (sg != s.sg) s = enter(sg, recs_of(sg));
            auto load_k = [&](int u, Frag<T>(&k)[KS]) {
                const int key = min(max(s.pl.c0 + s.pl.cs * (16 * u + li), 0), p.n_keys - 1);
                const T* const src = kb + (int64_t)key * p.k_sl + 8 * g;
#pragma unroll
                for (int t = 0; t < KS; ++t) {
                    k[t].v = __builtin_bit_cast(typename Frag<T>::vec, zero);
                    if (32 * t + 8 * g < d) k[t] = global_frag<T>(src + 32 * t);
                }
            };
            const int u_first = max(s.span.lo_min, 0) >> 4, u_end = min((max(s.span.hi_max, 0) + 15) >> 4, s.pl.n_tiles * (kBN / 16));
            int u = u_first + ((hw - u_first) & (GW - 1));
            Frag<T> k[KS];
            f32x4 acc[2];
            if (u < u_end) load_k(u, k);
            for (; u < u_end; u += GW) {
                products(k, acc);
                if (u + GW < u_end) load_k(u + GW, k);
                put(s, u, acc);
            }
        }
    }

    request_v();
    request_counts();

    // ---- softmax ----
    // which of the 8 slots of the lane's chunk c live, of the row of group `it`
    auto live_of = [&](int it, uint32_t(&live)[NCH]) {
#pragma unroll
        for (int i = 0; i < SPLAT_MAX_SEGMENTS; ++i) lr.cnt[i] = cnt[it][i];
        lr.set(segs, p.T);
#pragma unroll
        for (int c = 0; c < NCH; ++c) live[c] = lr.live8(8 * (my + LPR * c));
    };
    // a row of scores or probabilities: whole pieces, the beginning of one, or what lives in it
    auto store_row = [&](void* matrix, int it, const uint32_t(&live)[NCH], const u32x4(&row)[NCH]) {
        const int r = r0 + rs * (ROWS_PW * wave + RPW * it + lane / LPR);
        if (r >= L) return;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            T* const to = (T*)matrix + ((int64_t)bh * L + r) * p.T + 8 * (my + LPR * c);
            const u32x4 x = row[c];
            if (live[c] == 0xffu) {
                if (p.stream)
                    __builtin_nontemporal_store(x, reinterpret_cast<u32x4*>(to));
                else
                    __builtin_memcpy(to, &x, 16);
            } else if ((live[c] & (live[c] + 1u)) == 0u) {
                const uint32_t n = live[c];  // 1, 3, 7, ... 127
                if (n & 8u) __builtin_memcpy(to, &x, 8);
                const bool four = (n & 8u) != 0;
                const uint32_t y0 = four ? x[2] : x[0], y1 = four ? x[3] : x[1], rest = four ? n >> 4 : n;
                if (rest & 2u) __builtin_memcpy(to + (four ? 4 : 0), &y0, 4);
                const uint16_t z = (uint16_t)((rest & 2u) ? y1 : y0);
                if (rest == 1u || rest == 7u) __builtin_memcpy(to + (four ? 4 : 0) + ((rest & 2u) ? 2 : 0), &z, 2);
            } else {
                const vec8 v = __builtin_bit_cast(vec8, x);
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if ((live[c] >> e) & 1u) to[e] = v[e];
            }
        }
    };
    lds_barrier();  // the scores of all wavefronts are there
#pragma unroll
    for (int it = 0; it < ROWS_PW / RPW; ++it) {
        const int k = ROWS_PW * wave + RPW * it + lane / LPR;
        const int m = base[it] & 7, c0 = base[it] >> 3;
        u32x4 raw[NCH];
        uint32_t live[NCH];
        live_of(it, live);
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int ch = my + LPR * c;
            const u32x4 x = *reinterpret_cast<const u32x4*>(smem + place(k, c0 + ch));
            raw[c] = by_position ? window8(x, *reinterpret_cast<const u32x4*>(smem + place(k, c0 + ch + 1)), m) : x;
        }
        store_row(p.scores, it, live, raw);
        // (dead slots hold -inf, whose exponential is exactly 0 against a maximum of at least -1e30.  The common case, decided for the whole wavefront,
        // has none.)
        bool whole = true;
#pragma unroll
        for (int c = 0; c < NCH; ++c) whole = whole && live[c] == 0xffu;
        const bool all_whole = !__any(!whole);
        if (!all_whole) {
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                const u32x4 keep = spread8(live[c]);
                raw[c] = (raw[c] & keep) | (kMinusInf<T> & ~keep);
            }
        }
        float v[NCH][8], part[NCH], mx = kNegBig;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const vec8 t = __builtin_bit_cast(vec8, raw[c]);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[c][e] = (float)t[e];
                mx = fmaxf(mx, v[c][e]);
            }
        }
        mx = wave_max<LPR>(mx);
        const float mb = mx * kLog2e;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[c][e] = fast_exp2(fmaf(v[c][e], kLog2e, -mb));
            part[c] = add_chunk<false, true>(0.f, v[c], 0);
        }
        float sum = part[0];
        if constexpr (NCH > 2)
            sum = (part[0] + part[2]) + (part[1] + part[3]);
        else if constexpr (NCH > 1)
            sum = part[0] + part[1];
        sum = wave_sum<LPR>(sum);
        const float inv = sum > 0.f ? 1.0f / sum : 0.f;
        u32x4 o[NCH];
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            vec8 t;
#pragma unroll
            for (int e = 0; e < 8; ++e) t[e] = rounded<T>(v[c][e] * inv);
            o[c] = __builtin_bit_cast(u32x4, t);
        }
        store_row(p.probs, it, live, o);
        // back into LDS, zeros where the row has no slot; by position the slots of a piece come from two
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            u32x4 x = o[c];
            if (by_position) {
                u32x4 before = my == LPR - 1 ? o[(c + NCH - 1) % NCH] : o[c];
#pragma unroll
                for (int i = 0; i < 4; ++i) before[i] = from_lane_before<LPR>(before[i], lane);
                if (m != 0) x = window8(before, o[c], 8 - m);
            }
            *reinterpret_cast<u32x4*>(smem + place(k, c0 + my + LPR * c)) = x;
        }
    }

    // ---- output ----
    int v_off[FD];
    {
        const int sq = li >> 2, in_half = 16 * ((li & 3) >> 1) + 8 * (li & 1), blk = ROWB >= 256 ? sq : (sq >> 1);
#pragma unroll
        for (int fd = 0; fd < FD; ++fd) {
            const int dt = GW * fd + hw;
            v_off[fd] = G::V_AT + (8 * g + sq) * ROWB + in_half + 64 * ((dt >> 1) ^ blk) + 32 * ((dt & 1) ^ (g & 1));
        }
    }
    f32x4v acc[FD][2];
#pragma unroll
    for (int fd = 0; fd < FD; ++fd) acc[fd][0] = acc[fd][1] = f32x4v{0.f, 0.f, 0.f, 0.f};
    HalfWalk cur = v_first;
    if (cur.seg < n_seg) {
        write_v(0, va);
        if (v_ahead.seg < n_seg) advance(v_keys, v_ahead);
        if (v_ahead.seg < n_seg) load_v(v_ahead, va);
    }
    lds_barrier();
    // one tile: the next one goes from registers into the other stage (which everybody has left at the last barrier), the one two after that is requested
    auto step = [&](int stage, u32x4 (&next)[NI]) {
        const HalfWalk w = cur;
        advance(v_keys, cur);
        if (G::STAGES == 2 && cur.seg < n_seg) {
            write_v(stage ^ V_STAGE, next);
            if (v_ahead.seg < n_seg) advance(v_keys, v_ahead);
            if (v_ahead.seg < n_seg) load_v(v_ahead, next);
        }
        if (w.seg != s.sg) s = enter(w.seg, recs_of(w.seg));
#pragma unroll
        for (int hf = 0; hf < VK / 32; ++hf) {
            const int pos0 = w.tile * VK + 32 * hf;
            if (pos0 + 32 <= s.span.lo_min || pos0 >= s.span.hi_max) continue;
            Frag<T> pf[2];
#pragma unroll
            for (int cb = 0; cb < 2; ++cb) {
                const int row = 32 * pr + 16 * cb + li, j = pos0 + 8 * g;
                u32x4 x;
                if (s.by_position) {
                    x = *reinterpret_cast<const u32x4*>(smem + place(row, j >> 3));
                    // (a place that two positions share holds the live one's value)
                    if (!s.apart && !(pos0 >= s.span.lo_max && pos0 + 32 <= s.span.hi_min)) x &= spread8(inside8(j - s.win[cb].lo, s.win[cb].cnt));
                } else if (s.pl.uniform) {
                    const int slot = s.off + j - s.win[cb].lo;
                    x = window8(*reinterpret_cast<const u32x4*>(smem + place(row, slot >> 3)), *reinterpret_cast<const u32x4*>(smem + place(row, (slot >> 3) + 1)), slot & 7);
                    x &= spread8(inside8(j - s.win[cb].lo, s.win[cb].cnt));
                } else {
                    vec8 v;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        v[e] = (T)0.f;
                        if (win_live(s.win[cb], j + e)) {
                            const int slot = s.off + win_slot(s.win[cb], j + e);
                            v[e] = *reinterpret_cast<const T*>(smem + place(row, slot >> 3) + (slot & 7) * 2);
                        }
                    }
                    x = __builtin_bit_cast(u32x4, v);
                }
                pf[cb].v = __builtin_bit_cast(typename Frag<T>::vec, x);
            }
#pragma unroll
            for (int fd = 0; fd < FD; ++fd) {
                if (16 * (GW * fd + hw) >= d) break;  // wavefront-uniform
                const char* const a = smem + stage + 32 * hf * ROWB + v_off[fd];
                const Frag<T> vf = frag_from_tr<T>(lds_tr16(a), lds_tr16(a + 4 * ROWB));
                mma16(acc[fd][0], vf, pf[0]);
                mma16(acc[fd][1], vf, pf[1]);
            }
        }
        if constexpr (G::STAGES == 1) {
            lds_barrier();
            if (cur.seg < n_seg) {
                write_v(0, next);
                if (v_ahead.seg < n_seg) advance(v_keys, v_ahead);
                if (v_ahead.seg < n_seg) load_v(v_ahead, next);
            }
        }
        lds_barrier();
    };
    while (cur.seg < n_seg) {
        step(0, vb);
        if (cur.seg < n_seg) step(G::STAGES == 1 ? 0 : V_STAGE, va);
    }

    // ---- O^T (lane: row 32 pr + 16 cb + li, features 16 (GW fd + hw) + 4 g .. + 3) turned around in LDS, rows stored whole ----
#pragma unroll
    for (int fd = 0; fd < FD; ++fd)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            vec4 t;
#pragma unroll
            for (int e = 0; e < 4; ++e) t[e] = (T)acc[fd][cb][e];
            *reinterpret_cast<vec4*>(smem + (32 * pr + 16 * cb + li) * O_ROW + (16 * (GW * fd + hw) + 4 * g) * 2) = t;
        }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < ROWS_PW * CPR / 64; ++i) {
        const int flat = i * 64 + lane, row = ROWS_PW * wave + flat / CPR, c = flat % CPR, r = r0 + rs * row;
        const u32x4 x = *reinterpret_cast<const u32x4*>(smem + row * O_ROW + c * 16);
        if (r < L && c < d / 8) __builtin_nontemporal_store(x, reinterpret_cast<u32x4*>(reinterpret_cast<char*>(p.out) + ((int64_t)bh * L + r) * d * 2 + c * 16));
    }
}

template <typename T, int D, int PS, int KEYS, int NW>
static int launch_ops16(Operators16Params p, hipStream_t st) {
    using G = Ops16Geom<D, PS, NW>;
    p.n_row_blocks = count_row_blocks(p.L, kPlanBM, p.row_stride);
    p.total = (int)(2 * (int64_t)p.B * p.H * p.n_row_blocks);
    p.by_blocks = divisor(2 * p.n_row_blocks), p.by_h = divisor(p.H);
    static uint64_t reserved = 0;
    auto kern = operators16_kernel<T, D, PS, KEYS, NW>;
    if (const int rc = reserve_dynamic_lds(&reserved, reinterpret_cast<const void*>(kern), G::LDS_BYTES, "splat_operators")) return rc;
    kern<<<((p.total + 7) / 8) * 8, NW * 64, G::LDS_BYTES, st>>>(p);
    return check_launch("splat_operators");
}

static int launch_operators16(const Operators16Params& p, int64_t blocks, int dtype, bool kt, hipStream_t st) {
    auto by_layout = [&](auto t, auto dd, auto ps, auto nw) {
        using T = decltype(t);
        constexpr int D = decltype(dd)::value, PS = decltype(ps)::value, NW = decltype(nw)::value;
        return kt ? launch_ops16<T, D, PS, kAlongKeys, NW>(p, st) : launch_ops16<T, D, PS, (NW == 4 && PS > 64) ? kStaged : kDirect, NW>(p, st);
    };
    auto by_waves = [&](auto t, auto dd, auto ps) {  // (up to two workgroups a CU; of short rows one: 320 to 512, 64 slots, d = 128 0.94 to 0.99 of the time)
        return blocks <= (p.T <= 64 ? 256 : 512) ? by_layout(t, dd, ps, std::integral_constant<int, 8>{}) : by_layout(t, dd, ps, std::integral_constant<int, 4>{});
    };
    auto by_slots = [&](auto t, auto dd) {
        if (p.T <= 64) return by_waves(t, dd, std::integral_constant<int, 64>{});
        if (p.T <= 128) return by_waves(t, dd, std::integral_constant<int, 128>{});
        if (p.T <= 256) return by_waves(t, dd, std::integral_constant<int, 256>{});
        return by_layout(t, dd, std::integral_constant<int, 512>{}, std::integral_constant<int, 8>{});
    };
    auto by_d = [&](auto t) { return p.d <= 64 ? by_slots(t, std::integral_constant<int, 64>{}) : by_slots(t, std::integral_constant<int, 128>{}); };
    return dtype == SPLAT_BF16 ? by_d(bf16{}) : by_d(f16{});
}

}  // namespace splat

using namespace splat;

extern "C" int splat_operators(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* kT, int64_t k_sb, int64_t k_sh, int64_t k_sd,
                               int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl, void* scores, void* probs, void* out,
                               const splat_acsr_seg* segs, int32_t n_seg, int32_t B, int32_t H, int32_t L, int32_t n_keys, int32_t d, int32_t T,
                               float scale, int32_t dtype, const void* plan, int64_t plan_bytes, void* stream) {
    const char* who = "splat_operators";
    if (!q || !kT || !v || !scores || !probs || !out || !segs || !plan) return fail(SPLAT_E_NULL, "%s: null pointer argument", who);
    if (B <= 0 || H <= 0 || L <= 0 || n_keys <= 0 || d <= 0 || T <= 0)
        return fail(SPLAT_E_SHAPE, "%s: need B, H, L, n_keys, d, T > 0 (got %d, %d, %d, %d, %d, %d)", who, B, H, L, n_keys, d, T);
    if (L > (1 << 23) || n_keys > (1 << 23)) return fail(SPLAT_E_SHAPE, "%s: L and n_keys are limited to 2^23", who);
    if (dtype != SPLAT_F32 && dtype != SPLAT_F16 && dtype != SPLAT_BF16) return fail(SPLAT_E_DTYPE, "%s: unknown dtype %d", who, dtype);
    if (k_sd != 1 && k_sl != 1)
        return fail(SPLAT_E_ALIGN, "%s: kT needs unit stride along d (k_sd == 1) or along keys (k_sl == 1); got k_sd=%lld k_sl=%lld", who, (long long)k_sd,
                    (long long)k_sl);
    if (v_sl < d) return fail(SPLAT_E_SHAPE, "%s: v row stride %lld < d %d", who, (long long)v_sl, d);
    if (scores == probs) return fail(SPLAT_E_SHAPE, "%s: scores and probabilities need buffers of their own", who);
    if ((reinterpret_cast<uintptr_t>(plan) & 15) != 0) return fail(SPLAT_E_ALIGN, "%s: the plan must be 16-byte aligned", who);
    Operators16Params p;
    if (const int rc = fill_segs(who, segs, n_seg, p.seg, T)) return rc;
    const int64_t need = splat_attention_plan_bytes(segs, n_seg, L);
    if (need <= 0 || plan_bytes < need)
        return fail(SPLAT_E_SHAPE, "%s: the plan holds %lld bytes, this mask needs %lld", who, (long long)plan_bytes, (long long)need);
    auto whole = [](const void* ptr, std::initializer_list<int64_t> strides) {
        return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0 && std::all_of(strides.begin(), strides.end(), [](int64_t s) { return s % 8 == 0; });
    };
    const bool kt = k_sd != 1;
    p.row_stride = common_row_stride(segs, n_seg);
    const int64_t blocks = 2 * (int64_t)B * H * count_row_blocks(L, kPlanBM, p.row_stride);
    // Where the separate launches are as fast or faster, as shares of their time.  Several segments: 0.77 to 0.91 for 55 slots, but 0.94 to 1.17 for
    // 158 and 0.86 to 1.44 for 315, whose scores go into LDS one by one.  65 to 128 slots with d = 128: 0.79 to 0.98, and 1.01 to 1.13 at 320 to 448
    // workgroups.  More than 256 slots, two workgroups of eight wavefronts a CU: up to 512 workgroups 0.58 to 0.98 (64 of d = 80 to 128 1.02 to 1.10); beyond,
    // d = 64 0.76 to 0.92 from 384 slots and 1536 workgroups on, with fewer of either 0.90 to 1.13, d = 128 0.88 to 1.28.
    const bool pays = n_seg > 1 ? T <= 64
                      : T <= 64 ? true
                      : T <= 128 ? !(d > 96 && blocks > 256 && blocks <= 448)
                      : T <= 256 ? true
                      : blocks <= 512 ? d <= 64 || blocks >= 128 : d <= 64 && T >= 384 && blocks >= 1536;
    if (!pays || dtype == SPLAT_F32 || d % 8 != 0 || d > 128 || T > 512 || blocks > 0x7ffffff0 || !whole(q, {q_sb, q_sh, q_sl}) || !whole(v, {v_sb, v_sh, v_sl}) ||
        !whole(out, {}) || (!kt && !whole(kT, {k_sb, k_sh, k_sl})))
        return SPLAT_E_UNSUPPORTED;
    p.q = q, p.k = kT, p.v = v, p.scores = scores, p.probs = probs, p.out = out;
    p.q_sb = q_sb, p.q_sh = q_sh, p.q_sl = q_sl;
    p.k_sb = k_sb, p.k_sh = k_sh, p.k_sd = k_sd, p.k_sl = k_sl;
    p.v_sb = v_sb, p.v_sh = v_sh, p.v_sl = v_sl;
    p.B = B, p.H = H, p.L = L, p.n_keys = n_keys, p.d = d, p.T = T, p.n_seg = n_seg;
    p.scale = scale;
    p.plan = static_cast<const PlanRec*>(plan);  // the variant with gathered walks comes first
    p.stream = whole(scores, {T}) && whole(probs, {}) && T % 32 == 0 && (int64_t)B * H * L * T * 2 > kCachedBytes;
    begin_launch();
    return launch_operators16(p, blocks, dtype, kt, (hipStream_t)stream);
}

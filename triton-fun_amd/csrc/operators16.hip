// The three operators of a forward in one kernel: 16-bit types, rows of at most 512 slots, inner dimension a multiple of 8 up to 128, with the mask's
// plan table.  Scores and probabilities are written as the separate operators write them, and read by nobody.
//
// Bound: instructions and the latency of dependent requests, the stores of the two compressed matrices in large launches.  As
// three launches (or two, where the sampled product's wavefronts take the softmax) scores are read once and probabilities twice; here a workgroup
// keeps its rows in LDS from the first product to the last.  bfloat16, causal masks, the separate launches -> this kernel, us: 128 heads of 2048 rows,
// d = 64, 64 slots 58 -> 36, 128 78 -> 49, 256 148 -> 80, 512 224 -> 146; d = 128, 256 slots 195 -> 109, 512 274 -> 230; 8 heads of 2048, d = 64, 48 slots 11.8 -> 7.8,
// 512 35.3 -> 18.0; float16, 16 heads of 2000, 129 slots, d = 80 20.2 -> 15.4; 64 heads of 8192, 512 slots with step 2, d = 128 551 -> 466.
// (A first version had the general case of every place, rows whose steps differ among them, beside the common one: 300 vector and 200 scalar
// instructions for 8 slots of a lane, 128 registers and spills, 1.1 to 1.4 times the time.)
//
// A workgroup is 64 rows of one (batch, head) in two halves of 32, four wavefronts or eight.
//   Q: whole rows, once a workgroup, into the place of the scores and from there into every wavefront's operands.  Loaded straight into operands, by
//     every wavefront for itself and 64 bytes of 16 rows an instruction, it takes more of the address path than K: 64 heads of 8192, 512 slots with step 2, d = 128
//     495 -> 466 us, 128 heads of 2048, 512 slots 219 -> 209; 8 heads of 2048, d = 128, 48 slots 9.9 -> 8.9, 256 slots 16.0 -> 14.8 (and 13.8 with
//     tiles of 64 keys of V); d = 64 0 to 4 %.
//   Scores: S^T = K Q^T by 16x16x32 matrix instructions, the wavefronts of a half take turns at subtiles of 16 positions.  K goes through registers
//     into LDS a tile at a time, two tiles ahead, in the place of V's tiles, which is free until then; or from memory straight into the operands'
//     registers (kDirect): no barrier, but 16 lines a request and each of them twice.  That is faster for rows of up to 64 slots where eight
//     wavefronts share few rows (8 heads of 2048, 20 slots, d = 64 6.5 -> 6.3 us) and slower elsewhere (128 heads of 2048, 256 slots, d = 128 109 for 123).
//     K stored along the keys is turned on its way into LDS.
//   Softmax: a wavefront's share of the rows, in the order of addition of softmax_rows; scores and probabilities leave from here in whole 16-byte
//     pieces.  (Held back until the output is there, so that no wait for V is a wait for them: no faster, and the registers are missed.)
//   Output: O^T = V^T P^T, V through registers into two stages, three tiles ahead, one barrier a tile; a wavefront has
//     32 rows and its share of the features (the operands, their order and so the bits of spmm_tile.hip).
//
// A row of LDS has room for PS slots, a power of two.  One segment keeps a row by POSITION modulo PS, so that both products meet it in whole aligned
// pieces, and it is shifted to slots only for the softmax.  Several segments keep it by slot: scores are written one by one, and the last product reads
// shifted pieces.  The pieces of 16 bytes are permuted by the row, so that 16 rows at one place cover all banks.
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
    static constexpr int VK = NW == 8 && (D == 64 || PS <= 256) ? 64 : 32;  // keys of a tile of V (launches of eight wavefronts have LDS for it)
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

// x where it lies in [0, last], else the nearer end, in one instruction as with one bound (of two 512 slots with step 2, 64 heads of 8192, d = 128 465 -> 467 us,
// 129 slots, 16 heads of 2000, d = 80 15.30 -> 15.39)
__device__ __forceinline__ int clamped(int x, int last) {
#if defined(__HIP_DEVICE_COMPILE__)
    int r;
    asm("v_med3_i32 %0, %1, 0, %2" : "=v"(r) : "v"(x), "s"(last));
    return r;
#else
    return x < 0 ? 0 : x < last ? x : last;
#endif
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

// MULTI: several segments, rows by slot; else one, rows by position
template <typename T, int D, int PS, int KEYS, int NW, bool MULTI>
__global__ __launch_bounds__(NW * 64, 4) void operators16_kernel(const Operators16Params p) {
    using G = Ops16Geom<D, PS, NW>;
    constexpr int VK = G::VK, GW = NW / 2, NT = NW * 64, ROWS_PW = kHalfRows / NW;  // GW: wavefronts that share 32 rows
    constexpr int ROWB = G::ROWB, V_STAGE = G::V_STAGE, P_ROWB = G::P_ROWB, O_ROW = G::O_ROW;
    constexpr int KS = D / 32, CPR = ROWB / 16, NI = VK * CPR / NT, FD = D / 16 / GW;
    constexpr int NC = PS / 8, LPR = PS == 64 ? 8 : 16, NCH = NC / LPR, RPW = 64 / LPR;  // chunks of a row, lanes a row, chunks a lane, rows at a time
    constexpr int ITS = ROWS_PW / RPW;
    typedef T vec4 __attribute__((ext_vector_type(4)));
    typedef T vec8 __attribute__((ext_vector_type(8)));

    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, g = lane >> 4;
    const int pr = wave / GW, hw = wave % GW;  // which 32 rows, and the place among those that share them

    load_args(p.total, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.n_row_blocks, p.H, p.row_stride, p.L, p.n_keys, p.d, p.n_seg, p.plan,
              p.q, p.q_sb, p.q_sh, p.q_sl, p.k, p.k_sb, p.k_sh, p.k_sd, p.k_sl);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int per_head = 2 * p.n_row_blocks;
    const int bh = quotient(logical, p.by_blocks);
    const int at_block = per_head - 1 - (logical - bh * per_head);
    const int rb = at_block >> 1, half = at_block & 1;
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride, L = p.L, d = p.d, n_rb = p.n_row_blocks, n_seg = MULTI ? p.n_seg : 1;
    const int r0 = block_first_row(rb, kPlanBM, rs) + rs * half * kHalfRows;
    if (r0 >= L) return;

    const T* const kb = (const T*)p.k + b * p.k_sb + h * p.k_sh;
    const char* const vbytes = reinterpret_cast<const char*>((const T*)p.v + b * p.v_sb + h * p.v_sh);
    const PlanRec* const pt = p.plan;
    const u32x4 zero = {0u, 0u, 0u, 0u};

    // Q: whole rows into LDS, where the scores will be, and from there into the B operands; a thread's pieces are requested before anything else
    constexpr int NQ = kHalfRows * CPR / NT;
    u32x4 q_raw[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        const int f = tid + NT * i, row = f / CPR, c = f % CPR;
        q_raw[i] = zero;
        if (8 * c < d) q_raw[i] = *reinterpret_cast<const u32x4*>((const T*)p.q + b * p.q_sb + h * p.q_sh + (int64_t)min(r0 + rs * row, L - 1) * p.q_sl + 8 * c);
    }

    // ---- a segment: its walk, and where the 32 rows lie in it ----
    struct Seg {
        int sg, first, end;  // first, end: positions that one of the workgroup's rows sees
        int c0, cs;
        int lo[2], cnt[2];   // of rows 32 pr + 16 cb + li; slot 0 of the buffer's row is `off` positions before lo
        WaveSpan span;
        bool apart;          // by position: no two positions that the 32 rows' wavefronts walk share a place in LDS
    };
    auto row_rec = [&](int sg, int k) { return pt[plan_row_at(n_rb, n_seg, rb, sg, half * kHalfRows + k)]; };
    // (the table knows the mask alone: a row's slots are bounded by the buffer's here, as load_row_map does)
    auto count_of = [&](int sg, int k, const PlanRec& w) { return r0 + rs * k < L ? min(w[1], p.seg[sg].max_cnt) : 0; };
    auto enter = [&](int sg) {
        Seg s;
        const PlanRec r = plan_uniform_load(pt + plan_seg_at(n_seg, rb, sg));
        const PlanRec s0 = plan_uniform_load(pt + plan_span_at(n_rb, n_seg, rb, sg, 2 * half)), s1 = plan_uniform_load(pt + plan_span_at(n_rb, n_seg, rb, sg, 2 * half + 1));
        const PlanRec sp = pr ? s1 : s0;
        s.sg = sg, s.c0 = r[0], s.cs = r[1];
        s.span = planned_span(sp, p.seg[sg].max_cnt);
        s.first = max(min(s0[0], s1[0]), 0), s.end = min(max(max(s0[3], s1[3]), 0), r[2] * kBN);
        s.apart = ((max(s.span.hi_max, 0) + 31) & ~31) - (sp[0] & ~31) <= PS;
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const PlanRec w = row_rec(sg, 32 * pr + 16 * cb + li);
            s.lo[cb] = w[0], s.cnt[cb] = count_of(sg, 32 * pr + 16 * cb + li, w);
        }
        return s;
    };
    // A walk over the tiles of N positions that one of the workgroup's rows sees
    struct Walk {
        int sg, tile, end, c0, cs;
    };
    auto walk_of = [&](auto n, const Seg& s) {
        constexpr int N = decltype(n)::value;
        Walk w{s.sg, s.first / N, (s.end + N - 1) / N, s.c0, s.cs};
        w.tile = min(w.tile, w.end);
        return w;
    };
    auto settle = [&](auto n, Walk& w) {  // on to the next segment that has tiles
        if constexpr (MULTI) {
            while (w.tile >= w.end && w.sg + 1 < n_seg) w = walk_of(n, enter(w.sg + 1));
        }
        (void)n;
    };
    auto advance = [&](auto n, Walk& w) {
        ++w.tile;
        settle(n, w);
    };
    auto more = [](const Walk& w) { return w.tile < w.end; };
    auto place = [&](int row, int chunk) { return row * P_ROWB + (((chunk & (NC - 1)) ^ swz<P_ROWB>(row)) << 4); };
    constexpr std::integral_constant<int, VK> v_keys{};
    constexpr std::integral_constant<int, G::KK> k_keys{};
    Seg s = enter(0);
    Walk v_first = walk_of(v_keys, s);
    settle(v_keys, v_first);

    // ---- scores ----
    const int my_rows = (32 * pr + li) * P_ROWB, my_swz = swz<P_ROWB>(li) << 4;  // (rows 16 apart are permuted alike)
    auto put = [&](int u, const f32x4(&acc)[2]) {
        const int j = 16 * u + 4 * g;  // the lane's first position
        const bool whole = s.apart || (16 * u >= s.span.lo_max && 16 * u + 16 <= s.span.hi_min);
        char* const to = smem + my_rows + ((((2 * u + (g >> 1)) & (NC - 1)) << 4) ^ my_swz) + 8 * (g & 1);
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            vec4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = rounded<T>(acc[cb][e] * p.scale);
            if constexpr (MULTI) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int at = j + e - s.lo[cb], slot = p.seg[s.sg].slot_offset + at;
                    if ((unsigned)at < (unsigned)s.cnt[cb]) *reinterpret_cast<T*>(smem + place(32 * pr + 16 * cb + li, slot >> 3) + (slot & 7) * 2) = x[e];
                }
            } else if (whole) {
                *reinterpret_cast<vec4*>(to + 16 * P_ROWB * cb) = x;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if ((unsigned)(j + e - s.lo[cb]) < (unsigned)s.cnt[cb]) *reinterpret_cast<T*>(to + 16 * P_ROWB * cb + 2 * e) = x[e];
            }
        }
    };
    Frag<T> q[2][KS];  // B operands: rows 32 pr + 16 cb + li
    auto q_through_lds = [&]() {
#pragma unroll
        for (int i = 0; i < NQ; ++i) *reinterpret_cast<u32x4*>(smem + lds_off<ROWB, true>((tid + NT * i) / CPR, (tid + NT * i) % CPR * 16)) = q_raw[i];
        lds_barrier();
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int t = 0; t < KS; ++t)
                q[cb][t].v = __builtin_bit_cast(typename Frag<T>::vec, *reinterpret_cast<const u32x4*>(smem + lds_off<ROWB, true>(32 * pr + 16 * cb + li, (4 * t + g) * 16)));
        // (tiles of K lie behind the scores' place, and scores come after a tile's barrier)
        if constexpr (KEYS == kDirect || PS < D) lds_barrier();
    };
    auto products = [&](const Frag<T>(&k)[KS], f32x4(&acc)[2]) {
        acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < KS; ++t)
            if (D == 64 || 32 * t < d) mma16(acc[0], k[t], q[0][t]), mma16(acc[1], k[t], q[1][t]);
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
        auto load_tile = [&](const Walk& w, u32x4(&raw)[NP]) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int key = clamped(w.c0 + w.cs * (w.tile * KK + pc_key[i]), p.n_keys - 1);
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
        Walk cur = walk_of(k_keys, s);
        settle(k_keys, cur);
        Walk ahead = cur;
        u32x4 ra[NP], rb_[NP];
        if (more(ahead)) {
            load_tile(ahead, ra);
            advance(k_keys, ahead);
            if (more(ahead)) load_tile(ahead, rb_);
        }
        q_through_lds();
        auto tile = [&](int stage, u32x4(&raw)[NP]) {
            if (MULTI && cur.sg != s.sg) s = enter(cur.sg);
#pragma unroll
            for (int i = 0; i < NP; ++i) *reinterpret_cast<u32x4*>(smem + stage + pc_to[i]) = raw[i];
            if (more(ahead)) advance(k_keys, ahead);
            if (more(ahead)) load_tile(ahead, raw);
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
                    put(u, acc);
                }
            }
            if constexpr (G::K_STAGES == 1) lds_barrier();
            advance(k_keys, cur);
        };
        while (more(cur)) {
            tile(0, ra);
            if (more(cur)) tile(G::K_STAGES == 1 ? 0 : G::K_STAGE, rb_);
        }
    } else {
        q_through_lds();
        for (int sg = 0; sg < n_seg; ++sg) {
            if (MULTI && sg != s.sg) s = enter(sg);
            auto load_k = [&](int u, Frag<T>(&k)[KS]) {
                const int key = clamped(s.c0 + s.cs * (16 * u + li), p.n_keys - 1);
                const T* const src = kb + (int64_t)key * p.k_sl + 8 * g;
#pragma unroll
                for (int t = 0; t < KS; ++t) {
                    k[t].v = __builtin_bit_cast(typename Frag<T>::vec, zero);
                    if (32 * t + 8 * g < d) k[t] = global_frag<T>(src + 32 * t);
                }
            };
            const int u_first = max(s.span.lo_min, 0) >> 4, u_end = (min(s.span.hi_max, s.end) + 15) >> 4;
            int u = u_first + ((hw - u_first) & (GW - 1));
            Frag<T> k[KS];
            f32x4 acc[2];
            if (u < u_end) load_k(u, k);
            for (; u < u_end; u += GW) {
                products(k, acc);
                if (u + GW < u_end) load_k(u + GW, k);
                put(u, acc);
            }
        }
    }

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
    auto load_v = [&](const Walk& w, u32x4(&reg)[NI]) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int key = clamped(w.c0 + w.cs * (w.tile * VK + v_row[i]), p.n_keys - 1);
            reg[i] = *reinterpret_cast<const u32x4*>(vbytes + key * v_rowb + v_col[i]);
        }
    };
    auto write_v = [&](int stage, const u32x4(&reg)[NI]) {
#pragma unroll
        for (int i = 0; i < NI; ++i) *reinterpret_cast<u32x4*>(smem + stage + v_to[i]) = reg[i];
    };
    Walk cur = v_first, ahead = v_first;
    u32x4 va[NI], vb[NI];
    if (more(ahead)) {
        load_v(ahead, va);
        advance(v_keys, ahead);
        if (more(ahead)) load_v(ahead, vb);
    }

    // ---- softmax of this wavefront's share of the rows ----
    const int my = lane & (LPR - 1);
    int base[ITS], cnt[ITS][MULTI ? SPLAT_MAX_SEGMENTS : 1];  // position of slot 0 where rows lie by position; live slots
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
        const int k = ROWS_PW * wave + RPW * it + lane / LPR;
        base[it] = 0;
        if constexpr (MULTI) {
#pragma unroll
            for (int i = 0; i < SPLAT_MAX_SEGMENTS; ++i) cnt[it][i] = i < n_seg ? count_of(i, k, row_rec(i, k)) : 0;
        } else {
            const PlanRec w = row_rec(0, k);
            base[it] = w[0] - p.seg[0].slot_offset, cnt[it][0] = count_of(0, k, w);
        }
    }
    lds_barrier();  // the scores of all wavefronts are there
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
        const int k = ROWS_PW * wave + RPW * it + lane / LPR, r = r0 + rs * k;
        const int m = base[it] & 7, c0 = base[it] >> 3;
        u32x4 raw[NCH];
        uint32_t live[NCH];  // of the 8 slots of each chunk; none beyond L
        bool whole = true;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int ch = my + LPR * c;
            const u32x4 x = *reinterpret_cast<const u32x4*>(smem + place(k, c0 + ch));
            if constexpr (MULTI) {
                raw[c] = x, live[c] = 0;
#pragma unroll
                for (int i = 0; i < SPLAT_MAX_SEGMENTS; ++i) live[c] |= inside8(8 * ch - p.seg[i].slot_offset, cnt[it][i]);
            } else {
                raw[c] = window8(x, *reinterpret_cast<const u32x4*>(smem + place(k, c0 + ch + 1)), m);
                live[c] = inside8(8 * ch - p.seg[0].slot_offset, cnt[it][0]);
            }
            whole = whole && live[c] == 0xffu;
        }
        // the common case, decided for the whole wavefront, has no dead slot
        const bool all_whole = !__any(!whole);
        const int64_t to = ((int64_t)bh * L + r) * p.T + 8 * my;
        auto store_row = [&](void* matrix, const u32x4(&row)[NCH]) {
            T* const first = (T*)matrix + to;
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                const u32x4 x = row[c];
                T* const at = first + 8 * LPR * c;
                if (all_whole || live[c] == 0xffu) {
                    if (p.stream)
                        __builtin_nontemporal_store(x, reinterpret_cast<u32x4*>(at));
                    else
                        __builtin_memcpy(at, &x, 16);
                } else if ((live[c] & (live[c] + 1u)) == 0u) {  // the beginning of a piece: 1, 3, 7, ... 127
                    const uint32_t n = live[c];
                    const bool four = (n & 8u) != 0;
                    if (four) __builtin_memcpy(at, &x, 8);
                    const uint32_t y0 = four ? x[2] : x[0], y1 = four ? x[3] : x[1], rest = four ? n >> 4 : n;
                    if (rest & 2u) __builtin_memcpy(at + (four ? 4 : 0), &y0, 4);
                    const uint16_t z = (uint16_t)((rest & 2u) ? y1 : y0);
                    if (rest == 1u || rest == 7u) __builtin_memcpy(at + (four ? 4 : 0) + ((rest & 2u) ? 2 : 0), &z, 2);
                } else {
                    const vec8 v = __builtin_bit_cast(vec8, x);
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if ((live[c] >> e) & 1u) at[e] = v[e];
                }
            }
        };
        store_row(p.scores, raw);
        if (!all_whole) {  // dead slots hold -inf, whose exponential is exactly 0 against a maximum of at least -1e30
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
        store_row(p.probs, o);
        // back into LDS, zeros where the row has no slot; by position the slots of a piece come from two
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            u32x4 x = o[c];
            if constexpr (!MULTI) {
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
    if (more(cur)) {
        write_v(0, va);
        if (more(ahead)) advance(v_keys, ahead);
        if (more(ahead)) load_v(ahead, va);
    }
    lds_barrier();
    // one tile: the next one goes from registers into the other stage (which everybody has left at the last barrier), the one two after that is requested
    auto step = [&](int stage, u32x4(&next)[NI]) {
        const Walk w = cur;
        advance(v_keys, cur);
        auto put_next = [&](int to) {
            if (!more(cur)) return;
            write_v(to, next);
            if (more(ahead)) advance(v_keys, ahead);
            if (more(ahead)) load_v(ahead, next);
        };
        if constexpr (G::STAGES == 2) put_next(stage ^ V_STAGE);
        if (MULTI && w.sg != s.sg) s = enter(w.sg);
#pragma unroll
        for (int hf = 0; hf < VK / 32; ++hf) {
            const int pos0 = w.tile * VK + 32 * hf;
            if (pos0 + 32 <= s.span.lo_min || pos0 >= s.span.hi_max) continue;
            Frag<T> pf[2];
#pragma unroll
            for (int cb = 0; cb < 2; ++cb) {
                u32x4 x;
                if constexpr (MULTI) {
                    const int row = 32 * pr + 16 * cb + li, at = pos0 + 8 * g - s.lo[cb], slot = p.seg[s.sg].slot_offset + at;
                    x = window8(*reinterpret_cast<const u32x4*>(smem + place(row, slot >> 3)), *reinterpret_cast<const u32x4*>(smem + place(row, (slot >> 3) + 1)), slot & 7);
                    x &= spread8(inside8(at, s.cnt[cb]));
                } else {
                    x = *reinterpret_cast<const u32x4*>(smem + my_rows + 16 * P_ROWB * cb + (((((pos0 >> 3) + g) & (NC - 1)) << 4) ^ my_swz));
                    // (a place that two positions share holds the live one's value)
                    if (!s.apart && !(pos0 >= s.span.lo_max && pos0 + 32 <= s.span.hi_min)) x &= spread8(inside8(pos0 + 8 * g - s.lo[cb], s.cnt[cb]));
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
            put_next(0);
        }
        lds_barrier();
    };
    while (more(cur)) {
        step(0, vb);
        if (more(cur)) step(G::STAGES == 1 ? 0 : V_STAGE, va);
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

template <typename T, int D, int PS, int KEYS, int NW, bool MULTI>
static int launch_ops16(Operators16Params p, hipStream_t st) {
    using G = Ops16Geom<D, PS, NW>;
    p.n_row_blocks = count_row_blocks(p.L, kPlanBM, p.row_stride);
    p.total = (int)(2 * (int64_t)p.B * p.H * p.n_row_blocks);
    p.by_blocks = divisor(2 * p.n_row_blocks), p.by_h = divisor(p.H);
    static uint64_t reserved = 0;
    auto kern = operators16_kernel<T, D, PS, KEYS, NW, MULTI>;
    if (const int rc = reserve_dynamic_lds(&reserved, reinterpret_cast<const void*>(kern), G::LDS_BYTES, "splat_operators")) return rc;
    kern<<<((p.total + 7) / 8) * 8, NW * 64, G::LDS_BYTES, st>>>(p);
    return check_launch("splat_operators");
}

static int launch_operators16(const Operators16Params& p, int64_t blocks, int dtype, bool kt, hipStream_t st) {
    auto by_layout = [&](auto t, auto dd, auto ps, auto nw, auto multi) {
        using T = decltype(t);
        constexpr int D = decltype(dd)::value, PS = decltype(ps)::value, NW = decltype(nw)::value;
        constexpr bool MULTI = decltype(multi)::value;
        return kt ? launch_ops16<T, D, PS, kAlongKeys, NW, MULTI>(p, st)
                  : launch_ops16<T, D, PS, (MULTI || (NW == 8 && PS == 64)) ? kDirect : kStaged, NW, MULTI>(p, st);
    };
    auto by_segments = [&](auto t, auto dd, auto ps, auto nw) {
        return p.n_seg > 1 ? by_layout(t, dd, ps, nw, std::true_type{}) : by_layout(t, dd, ps, nw, std::false_type{});
    };
    // Eight wavefronts up to two workgroups a CU, of short rows one.  bfloat16, as shares of the separate launches' time, four and eight: 40 to
    // 64 slots, d = 64, 256 workgroups 0.71 and 0.63, 384 0.73 and 0.77; 256 slots, d = 64, 256 workgroups 0.77 and 0.61, 512 0.68 and 0.62, 1024
    // 0.71 and 0.76, d = 128, 1024 0.76 and 0.90; two segments of 10 to 64 slots together 288 to 512 workgroups 0.79 to 0.88 and 0.81 to 0.90; of 83 to 256 (17 masks,
    // d = 32 to 128, rows of K and K along the keys) 288 to 512 0.84 to 1.09 and 0.83 to 1.01, 576 and 640 0.84 to 1.02 and 0.89 to 1.15, beyond 0.67 to 1.09 and
    // 0.78 to 1.29.  Longer rows have two workgroups a CU in any case: 512 slots, d = 128, 4096 workgroups 0.94 and 0.84.
    auto by_waves = [&](auto t, auto dd, auto ps) {
        return blocks <= (p.T <= 64 ? 256 : 512) ? by_segments(t, dd, ps, std::integral_constant<int, 8>{})
                                                                : by_segments(t, dd, ps, std::integral_constant<int, 4>{});
    };
    auto by_slots = [&](auto t, auto dd) {
        if (p.T <= 64) return by_waves(t, dd, std::integral_constant<int, 64>{});
        if (p.T <= 128) return by_waves(t, dd, std::integral_constant<int, 128>{});
        if (p.T <= 256) return by_waves(t, dd, std::integral_constant<int, 256>{});
        return by_segments(t, dd, std::integral_constant<int, 512>{}, std::integral_constant<int, 8>{});
    };
    auto by_d = [&](auto t) { return p.d <= 64 ? by_slots(t, std::integral_constant<int, 64>{}) : by_slots(t, std::integral_constant<int, 128>{}); };
    return dtype == SPLAT_BF16 ? by_d(bf16{}) : by_d(f16{});
}

// The separate launches are faster on some masks of several segments, whose scores go into LDS one by one.  Shares of their time, bfloat16, two segments
// (23 masks, heads of 1024 and 4096 rows, graphs of the forwards):
// More than 256 slots together: rows of K, d = 32 and 64, 16 and 32 workgroups 0.97 to 1.10, 80 to 448 0.72 to 0.99, 512 at d = 64 0.90 to 0.99, at d = 32
// 0.93 to 1.03, beyond 1.06 to 1.21; K along the keys, which is turned tile by tile, 16 to 96 workgroups 0.94 to 1.17, 128 to 448 0.70 to 1.01; d = 128, rows 64
// workgroups 1.09, 128 to 256 0.77 to 0.97, beyond 1.10 to 1.28, keys 128 0.91 to 1.10, 192 and 256 0.76 to 0.95.
// 129 to 256 slots, more than 512 workgroups, scores that the sampled product's wavefronts take the softmax of (own_rows_fit): d = 32 and 64 up to 2048
// workgroups 0.78 to 1.06, at 3072 and 4096 0.89 to 1.09; d = 96 0.82 to 1.04; d = 128 up to 768 0.90 to 0.96, 1024 and 1536 0.93 to 1.07, beyond 0.86 to 1.08 with
// a mean of 0.99.  Larger scores 0.69 to 1.01, fewer slots 0.67 to 1.01.
static bool one_launch_pays(int n_seg, int T, int d, bool kt, int64_t blocks, int64_t score_bytes) {
    if (n_seg == 1 || T <= 128) return true;
    if (T > 256) return d <= 64 ? blocks >= (kt ? 128 : 80) && blocks <= (d <= 32 ? 448 : 512) : blocks >= (kt ? 192 : 128) && blocks <= 256;
    if (score_bytes > kCachedBytes) return true;
    return d <= 64 ? blocks <= 2048 : d <= 96 || blocks <= 768 || blocks > 1536;
}

}  // namespace splat

using namespace splat;

extern "C" int splat_operators(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* kT, int64_t k_sb, int64_t k_sh, int64_t k_sd,
                               int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl, void* scores, void* probs, void* out,
                               const splat_acsr_seg* segs, int32_t n_seg, int32_t B, int32_t H, int32_t L, int32_t n_keys, int32_t d, int32_t T,
                               float scale, int32_t dtype, const void* plan, int64_t plan_bytes, int32_t one_step, void* stream) {
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
    // In separate launches an operand has been read before a later result takes its memory (K in the output of the call before, say); here workgroups
    // store results while others still read.
    const Extent results[] = {extent_of(scores, 2, {{B * (int64_t)H * L, T}, {T, 1}}), extent_of(probs, 2, {{B * (int64_t)H * L, T}, {T, 1}}),
                              extent_of(out, 2, {{B * (int64_t)H * L, d}, {d, 1}})};
    const Extent operands[] = {extent_of(q, 2, {{B, q_sb}, {H, q_sh}, {L, q_sl}, {d, 1}}), extent_of(kT, 2, {{B, k_sb}, {H, k_sh}, {d, k_sd}, {n_keys, k_sl}}),
                               extent_of(v, 2, {{B, v_sb}, {H, v_sh}, {n_keys, v_sl}, {d, 1}})};
    bool apart = !results[0].meets(results[1]) && !results[0].meets(results[2]) && !results[1].meets(results[2]);
    for (const Extent& r : results)
        for (const Extent& o : operands) apart = apart && !r.meets(o);
    const bool kt = k_sd != 1;
    p.row_stride = common_row_stride(segs, n_seg);
    const int64_t blocks = 2 * (int64_t)B * H * count_row_blocks(L, kPlanBM, p.row_stride);
    if (!apart || !one_launch_pays(n_seg, T, d, kt, blocks, (int64_t)B * H * L * T * 2) || !one_step || dtype == SPLAT_F32 || d % 8 != 0 || d > 128 || T > 512 || blocks > 0x7ffffff0 || !whole(q, {q_sb, q_sh, q_sl}) || !whole(v, {v_sb, v_sh, v_sl}) ||
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

// Fused backward of the ACSR attention in float32: dQ, and dK + dV, without any compressed [B, H, L, T] matrix in memory.
//
// The products, the roles of the operands and the plans are those of attention_bwd.hip (dQ: rows are queries, positions keys, X = K,
// Y = V; dK + dV: rows are keys, positions queries, X = Q, Y = dO):
//     S^T = X A^T;  P;  dP^T = Y B^T;  dS = P (dP - D);  acc^T += X^T dS^T;  dK + dV also acc2^T += Y^T P^T
// They run, as in attention_f32.hip, on the 16-bit matrix instructions, of operands split into three parts (split3.hpp): a wavefront
// owns 16 rows, four of them share tiles of 32 positions, whose pieces every thread loads a tile ahead, splits, and writes between two
// barriers.  A and B are split once and stay in registers.  dK + dV at d = 128 does not fit them and is a kernel of its own
// (attention_bwd_f32_keys.hip).
// Measured against the kernel on the float32 instructions, us: 64 heads of 2048 rows, d = 64, window 256: dQ 140 -> 97, dK + dV 181 ->
// 135; 128 heads, window 32: 99 -> 81 and 116 -> 104; 32 heads, d = 128, window 256 / 32: dQ 142 -> 110 and 59 -> 51; one head, window 32,
// d = 64: 11.0 -> 9.7 and 10.8 -> 9.6.  Two workgroups of dQ a CU instead of three at d = 64: 110.  Relative error of dq, dk, dv
// against float64 (norms), window 257: 5.1e-7, 5.1e-7, 4.9e-7 -> 4.3e-7, 4.3e-7, 4.2e-7.
#include "attn_bwd.hpp"
#include "rows16.hpp"
#include "split3.hpp"

namespace splat {

// PER_CU: workgroups a CU that registers are kept for
template <int D, bool KEYS, int PER_CU>
__global__ __launch_bounds__(256, PER_CU) void attn_bwd_f32_kernel(const BwdParams p) {
    constexpr int BN = 32, ROWB = 2 * D, PLANE = BN * ROWB, TILE = 3 * PLANE;  // positions a tile; bytes of a row, a plane, an operand
    constexpr int STATS = 2 * TILE;           // lse and D of the tile's positions (dK + dV)
    constexpr int KS = D / 32, DT = D / 16;
    constexpr int CPR = D / 8;                // 8-value pieces of a row
    constexpr int NP = 2 * BN * CPR / 256;    // pieces a thread: the first half of them X's, the others Y's
    constexpr int AHEAD = D == 64 && !(KEYS && PER_CU == 3) ? 2 : 1;  // parts of fragments requested ahead of their products (as many as registers are left)
    constexpr float kLog2e = 1.4426950408889634f;

    extern __shared__ __attribute__((aligned(1024))) char smem[];  // three planes of X, three of Y, the statistics

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;

    load_args(p.total, p.n_row_blocks, p.by_blocks.m, p.by_blocks.shift, p.by_h.m, p.by_h.shift, p.H, p.row_stride, p.L, p.n_seg, p.plan, p.scale_log2e,
              p.a, p.a_sb, p.a_sh, p.a_sl, p.b, p.b_sb, p.b_sh, p.b_sl, p.x, p.x_sb, p.x_sh, p.x_sl, p.y, p.y_sb, p.y_sh, p.y_sl, p.lse, p.delta);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int per_head = 2 * p.n_row_blocks;
    const int bh = quotient(logical, p.by_blocks);
    const int at = per_head - 1 - (logical - bh * per_head);
    const int rb = at >> 1, half = at & 1;
    const int b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int rs = p.row_stride, L = p.L, Lr = p.Lr;
    const int k0 = half * kHalfRows;
    const int r0 = block_first_row(rb, kPlanBM, rs) + rs * k0;
    if (r0 >= Lr) return;

    const float* ab = (const float*)p.a + b * p.a_sb + h * p.a_sh;
    const float* bb = (const float*)p.b + b * p.b_sb + h * p.b_sh;
    const float* xb = (const float*)p.x + b * p.x_sb + h * p.x_sh;
    const float* yb = (const float*)p.y + b * p.y_sb + h * p.y_sh;
    const float* lse_b = p.lse + (int64_t)bh * L;
    const float* del_b = p.delta + (int64_t)bh * L;

    // ---- the lane's share of its rows of A and B: B operands of the products over d ----
    const int out_row = r0 + rs * (wave * 16 + n);
    int my_row = min(out_row, Lr - 1);
    if constexpr (KEYS) {
        if (p.row_map) my_row = min(max(p.row_map[my_row], 0), L - 1);
    }
    const float* const a_row = ab + (int64_t)my_row * p.a_sl;
    const float* const b_row = bb + (int64_t)my_row * p.b_sl;
    f32x8 a_raw[KS], b_raw[KS], o_raw[KEYS ? 1 : KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        a_raw[ks] = global_frag<float>(a_row + 32 * ks + 8 * g).v;
        b_raw[ks] = global_frag<float>(b_row + 32 * ks + 8 * g).v;
        if constexpr (!KEYS)
            o_raw[ks] = global_frag<float>((const float*)p.o + b * p.oo_sb + h * p.oo_sh + (int64_t)my_row * p.oo_sl + 32 * ks + 8 * g).v;
    }
    float row_lse2 = 0.f, row_delta = 0.f;  // dQ: the lane's own query
    if constexpr (!KEYS) row_lse2 = lse_b[my_row] * kLog2e;

    // ---- plan: the row block's walk, cut down to the tiles that this half of it sees ----
    const PlanRec* const pt = p.plan;
    const int n_rb = p.n_row_blocks;
    auto walk_of = [&](int sg) { return half_walk<BN>(pt, n_rb, p.n_seg, rb, half, sg); };
    auto next_segment = [&](HalfWalk& w) {  // the first segment from w.seg on that has tiles
        for (int sg = w.seg; sg < p.n_seg; ++sg) {
            w = walk_of(sg);
            if (w.end > w.tile) return;
        }
        w.seg = p.n_seg, w.tile = 0, w.end = 0x7fffffff;
    };
    HalfWalk fetch;
    fetch.seg = 0;
    next_segment(fetch);
    int total = fetch.end - fetch.tile;
    for (int sg = fetch.seg + 1; sg < p.n_seg; ++sg) {
        const HalfWalk w = walk_of(sg);
        total += w.end - w.tile;
    }
    total = fetch.seg < p.n_seg ? __builtin_amdgcn_readfirstlane(total) : 0;

    // ---- a tile's way into LDS: pieces of 8 values, by their position in the tile's rows ----
    const uint32_t smem_base = lds_address(smem);
    int pc_row[NP], pc_c[NP];
    uint32_t pc_to[NP];  // LDS address of its first part
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int f = (tid + 256 * i) % (BN * CPR);
        pc_row[i] = f / CPR, pc_c[i] = f % CPR;
        pc_to[i] = smem_base + (i < NP / 2 ? 0 : TILE) + pc_row[i] * ROWB + ((pc_c[i] ^ swz_both16<ROWB>(pc_row[i])) << 4);
    }
    f32x8 raw[NP];
    float raw_stat = 0.f;  // dK + dV: wavefront 0 carries lse (lanes 0..31) and D
    // operands of one head within 32-bit offsets, and strides that 24-bit products take
    const bool narrow = max(p.x_sl, p.y_sl) * 4 * L < ((int64_t)1 << 32) && max(p.x_sl, p.y_sl) * 4 < (1 << 24);
    auto load_next = [&](HalfWalk& w) {  // the tile the walk stands at, which moves on
        const int c0 = w.pl.c0 + w.pl.cs * w.tile * BN;
        auto position = [&](int row) { return min(max(c0 + w.pl.cs * row, 0), L - 1); };
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const char* base = reinterpret_cast<const char*>(i < NP / 2 ? xb : yb);
            const int64_t sl = i < NP / 2 ? p.x_sl : p.y_sl;
            const int row = position(pc_row[i]);
            if (narrow)
                raw[i] = global_frag<float>(reinterpret_cast<const float*>(base + (__umul24(row, (uint32_t)sl * 4) + 32 * pc_c[i]))).v;
            else
                raw[i] = global_frag<float>(reinterpret_cast<const float*>(base) + row * sl + 8 * pc_c[i]).v;
        }
        if constexpr (KEYS) {
            if (wave == 0) raw_stat = (lane < BN ? lse_b : del_b)[position(lane & (BN - 1))];
        }
        if (++w.tile >= w.end) {
            ++w.seg;
            next_segment(w);
        }
    };

    // ---- LDS read addresses of X (Y: TILE further) ----
    const int tr_row = (lane & 15) >> 2, tr_chunk = (lane >> 1) & 1, tr_byte = 8 * (lane & 1);  // transposing reads: 4 rows x 32 bytes
    // (pieces of a row are permuted by an exclusive or, so that the addresses of one row differ by one)
    uint32_t r_base = smem_base + n * ROWB + ((g ^ swz_both16<ROWB>(n)) << 4);
    uint32_t c_base = smem_base + (4 * g + tr_row) * ROWB + ((tr_chunk ^ swz_both16<ROWB>(4 * g + tr_row)) << 4) + tr_byte;

    HalfWalk cur = fetch;
    PlanRec win_rec = {0, 0, 1, 0};
    if (total > 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + wave * 16 + n)];
    if (total > 0) load_next(fetch);

    // (one operand after the other: their raw and split forms together would not fit the registers at d = 128)
    Split3 af[KS], bf[KS];
    float a_most = 0.f, b_most = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        bf[ks] = split3(b_raw[ks]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            b_most = fmaxf(b_most, fabsf(b_raw[ks][e]));
            if constexpr (!KEYS) row_delta = fmaf(b_raw[ks][e], o_raw[ks][e], row_delta);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        af[ks] = split3(a_raw[ks]);
#pragma unroll
        for (int e = 0; e < 8; ++e) a_most = fmaxf(a_most, fabsf(a_raw[ks][e]));
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!KEYS) row_delta = over_groups(row_delta, [](float x, float y) { return x + y; });  // D = rowsum(dO * O)
    bool beyond = out_of_split(a_most) || out_of_split(b_most);  // something that the split operands do not hold

    f32x4 acc[DT], acc2[KEYS ? DT : 1];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (KEYS) acc2[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // X and Y are lifted, and with them S, dP and dS, so that what the kernel itself splits holds its parts as well: dS is small where
    // dO and V are so together.  P is lifted for its product with Y; the results are so twice.
    const float c2 = p.scale_log2e * (1.f / kSplitLift), lift_delta = row_delta * kSplitLift;
    RowState rows;
    bool entered = false;

    for (int it = 0; it < total; ++it) {
        if (!entered) {
            if (it > 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + wave * 16 + n)];
            const RowWin w = {win_rec.x, win_rec.y, win_rec.z};
            rows.template enter<BN>(w, win_rec.w, cur.pl.uniform != 0, cur.tile);
            entered = true;
        }
        const int j0 = cur.tile * BN;
        lds_barrier();  // everybody is done with tile it - 1
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const Split3 s = split3(raw[i] * kSplitLift);
#pragma unroll
            for (int k = 0; k < 3; ++k) lds_store128(pc_to[i] + k * PLANE, __builtin_bit_cast(u32x4, s.p[k].v));
        }
        if constexpr (KEYS) {
            if (wave == 0) reinterpret_cast<float*>(smem + STATS)[lane] = lane < BN ? raw_stat : raw_stat * kSplitLift;
        }
        if (it + 1 < total) load_next(fetch);
        lds_barrier();  // tile `it` is there

        if (j0 + BN > rows.lo_min && j0 < rows.hi_max) {
#if defined(__HIP_DEVICE_COMPILE__)
            asm volatile("" : "+v"(r_base), "+v"(c_base));  // (the addresses are made here: kept over the loop they would spill)
#endif
            auto r_addr = [&](int ks) { return r_base ^ (uint32_t)(ks << 6); };
            auto c_addr = [&](int dt) { return c_base ^ (uint32_t)(dt << 5); };
            // ---- S^T = X A^T, then dP^T = Y B^T, of two subtiles of 16 positions; fragments are requested ahead of their products, part k
            // of a step as the one of the step before is done with ----
            Frag<bf16> rf[2][3];
            auto load_rf = [&](int x) {  // part 2 - x % 3 of step x / 3
                const int st = x / 3, k = 2 - x % 3;
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    rf[u][k].v = __builtin_bit_cast(bf16x8, lds_load128(r_addr(st % KS) + (st / KS) * TILE + k * PLANE + 16 * u * ROWB));
            };
#pragma unroll
            for (int x = 0; x < AHEAD; ++x) load_rf(x);
            __builtin_amdgcn_sched_barrier(0);
            f32x4 s[2], ds[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) s[u] = ds[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m = 0; m < 24 * KS; ++m) {
                const int st = m / 12, i = (m % 12) / 2, u = m % 2, x = 3 * st + 2 - kSplitA[i];
                if (st < KS)
                    mma16(s[u], rf[u][kSplitA[i]], af[st % KS].p[kSplitB[i]]);
                else
                    mma16(ds[u], rf[u][kSplitA[i]], bf[st % KS].p[kSplitB[i]]);
                if (u == 1 && kSplitLast[kSplitA[i]] == i && x + AHEAD < 6 * KS) load_rf(x + AHEAD);
                __builtin_amdgcn_sched_barrier(0);
            }
            // ---- P = exp2(S * scale * log2e - lse * log2e); masked scores underflow to exactly 0.  dS = P (dP - D) ----
            if (!(j0 >= rows.lo_max && j0 + BN <= rows.hi_min)) rows.mask_tile(s, j0, g, cur.pl.uniform != 0, kNegBigA * kSplitLift);
            Frag<bf16> cf[2][3];
            auto load_cf = [&](int operand, int x) {
                const int d2 = x / 3, k = 2 - x % 3;
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    const uint32_t a0 = c_addr(2 * d2 + y) + operand * TILE + k * PLANE;
                    cf[y][k] = frag_from_tr<bf16>(lds_load_tr16(a0), lds_load_tr16(a0 + 16 * ROWB));
                }
            };
            f32x8 pr, dsv;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                f32x4 lse4, del4;
                if constexpr (KEYS) {
                    lse4 = __builtin_bit_cast(f32x4, lds_load128(smem_base + STATS + 64 * u + 16 * g));
                    del4 = __builtin_bit_cast(f32x4, lds_load128(smem_base + STATS + 128 + 64 * u + 16 * g));
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int e = 4 * u + j;
                    pr[e] = fast_exp2(fmaf(s[u][j], c2, KEYS ? -kLog2e * lse4[j] : -row_lse2));
                    dsv[e] = pr[e] * (ds[u][j] - (KEYS ? del4[j] : lift_delta));
                }
            }
            // ---- acc2^T += Y^T P^T, acc^T += X^T dS^T, of two tiles of 16 columns at a time ----
            auto accumulate = [&](f32x4 (&to)[DT], int operand, const f32x8& v) {
#pragma unroll
                for (int x = 0; x < AHEAD; ++x) load_cf(operand, x);
                __builtin_amdgcn_sched_barrier(0);
                const Split3 vf = split3(v);
#pragma unroll
                for (int m = 0; m < 6 * DT; ++m) {
                    const int d2 = m / 12, i = (m % 12) / 2, y = m % 2, x = 3 * d2 + 2 - kSplitA[i];
                    mma16(to[2 * d2 + y], cf[y][kSplitA[i]], vf.p[kSplitB[i]]);
                    if (y == 1 && kSplitLast[kSplitA[i]] == i && x + AHEAD < 3 * DT / 2) load_cf(operand, x + AHEAD);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            if constexpr (KEYS) accumulate(acc2, 1, pr * kSplitLift);
            accumulate(acc, 0, dsv);
        }
        if (!cur.pl.uniform) rows.next_tile();
        if (++cur.tile >= cur.end) {
            ++cur.seg;
            next_segment(cur);
            entered = false;
        }
    }

    // What is not finite anywhere, the lift's overflow included, stays so in a row's results (NaN compares unequal).
    float chk = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            chk = fmaf(acc[dt][j], 0.f, chk);
            if constexpr (KEYS) chk = fmaf(acc2[dt][j], 0.f, chk);
        }
    beyond |= chk != 0.f;
    auto out_at = [&](void* base) { return (float*)base + b * p.o_sb + h * p.o_sh + (int64_t)out_row * p.o_sl; };
    if constexpr (!KEYS) {
        if (out_row < Lr && g == 0) p.delta_w[(int64_t)bh * L + out_row] = row_delta;
    }
    if (__any(beyond)) {
        // ---- this wavefront's rows once more in float32 arithmetic, position by position, each lane a quarter of a row's columns,
        // live positions only (64 heads of 2048 rows, d = 64, window 256, every row: 1470 for 213 us) ----
        constexpr int QD = D / 4;
        float a[QD], bq[QD], r1[QD], r2[KEYS ? QD : 1];
#pragma unroll
        for (int i = 0; i < QD; ++i) {
            a[i] = a_row[g * QD + i], bq[i] = b_row[g * QD + i], r1[i] = 0.f;
            if constexpr (KEYS) r2[i] = 0.f;
        }
        for (int sg = 0; sg < p.n_seg; ++sg) {
            const HalfWalk w = walk_of(sg);
            const PlanRec wr = pt[plan_row_at(n_rb, p.n_seg, rb, sg, k0 + wave * 16 + n)];
            const RowWin win = {wr.x, wr.y, wr.z};
            for (int j = w.tile * BN; j < w.end * BN; ++j) {
                const bool live = win_live(win, j);
                if (!__any(live)) continue;
                const int64_t pos = min(max(w.pl.c0 + w.pl.cs * j, 0), L - 1);
                const float *xr = xb + pos * p.x_sl + g * QD, *yr = yb + pos * p.y_sl + g * QD;
                float s = 0.f, dp = 0.f;
#pragma unroll
                for (int i = 0; i < QD; ++i) s = fmaf(a[i], xr[i], s), dp = fmaf(bq[i], yr[i], dp);
                s = over_groups(s, [](float x, float y) { return x + y; });
                dp = over_groups(dp, [](float x, float y) { return x + y; });
                if (live) {
                    const float e = fast_exp2(fmaf(s, p.scale_log2e, KEYS ? -kLog2e * lse_b[pos] : -row_lse2));
                    const float d = e * (dp - (KEYS ? del_b[pos] : row_delta));
#pragma unroll
                    for (int i = 0; i < QD; ++i) {
                        r1[i] = fmaf(d, xr[i], r1[i]);
                        if constexpr (KEYS) r2[i] = fmaf(e, yr[i], r2[i]);
                    }
                }
            }
        }
        if (out_row < Lr) {
#pragma unroll
            for (int i = 0; i < QD; ++i) {
                out_at(p.out)[g * QD + i] = r1[i] * p.scale;
                if constexpr (KEYS) out_at(p.out2)[g * QD + i] = r2[i];
            }
        }
        return;
    }

    // ---- epilogue: a lane holds columns 16 dt + 4g .. + 3 of its row ----
    if (out_row < Lr) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            *reinterpret_cast<f32x4*>(out_at(p.out) + 16 * dt + 4 * g) = acc[dt] * (1.f / (kSplitLift * kSplitLift)) * p.scale;
            if constexpr (KEYS) *reinterpret_cast<f32x4*>(out_at(p.out2) + 16 * dt + 4 * g) = acc2[dt] * (1.f / (kSplitLift * kSplitLift));
        }
    }
}

template <int D, bool KEYS, int PER_CU>
static int launch(const BwdParams& p0, hipStream_t st) {
    begin_launch();
    BwdParams p = p0;
    p.total = p.B * p.H * 2 * p.n_row_blocks;
    p.by_blocks = divisor(2 * p.n_row_blocks), p.by_h = divisor(p.H);
    constexpr size_t lds = 6 * 32 * D * 2 + 256;
    auto kern = attn_bwd_f32_kernel<D, KEYS, PER_CU>;
    static uint64_t lds_reserved = 0;
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), lds, "splat_attention_bwd_f32")) return rc;
    kern<<<((p.total + 7) / 8) * 8, 256, lds, st>>>(p);
    return check_launch("splat_attention_bwd_f32");
}

int launch_bwd_dq_f32(const BwdParams& dq, int d, hipStream_t st) { return d == 64 ? launch<64, false, 3>(dq, st) : launch<128, false, 2>(dq, st); }
int launch_bwd_dkv_f32(const BwdParams& dkv, int d, hipStream_t st) {
    if (d != 64) return launch_bwd_dkv_f32_d128(dkv, st);
    // Beyond two workgroups a CU, three of them of 168 registers each (28 bytes of scratch, fragments one part ahead), us, two a CU -> three: 680 workgroups, window
    // 128 37.3 -> 33.0; 768, window 257 to both sides 60.0 -> 51.0; 1440, window 100 62.4 -> 60.7; 2048, window 256 139 -> 133 and 139; 4096, window 32 111 -> 104.
    // Up to that the third is of no use: 512, window 128 25.1 -> 26.6; 16, window 32 9.7 -> 9.9.
    return (int64_t)dkv.B * dkv.H * 2 * dkv.n_row_blocks > 2 * 256 ? launch<64, true, 3>(dkv, st) : launch<64, true, 2>(dkv, st);
}

}  // namespace splat

// dK + dV of the fused float32 backward at d = 128, on the float32 matrix instructions.
//
// The products and the plan are those of attention_bwd_f32.hip: rows are keys, positions queries, X = Q, Y = dO, A = K, B = V:
//     S^T = X A^T;  P;  dP^T = Y B^T;  dS = P (dP - D);  acc^T += X^T dS^T;  acc2^T += Y^T P^T
// Operands split into bfloat16 parts, as there, take 96 registers for A and B and 64 for the two results here and spill: 32 heads of
// 2048 rows, window 256 / 32, us: this kernel 179 / 68, split 249 / 95, and with eight wavefronts a workgroup 163 / 82.
// Bound: these instructions and the vector arithmetic that shares their units.  A wavefront owns 16 rows and takes positions in
// subtiles of 16, skipping those outside its rows' spans; four wavefronts share tiles of 16 positions.  A and B stay in registers, X
// and Y come through the asynchronous copy ring; their tiles are read row-wise for the products over d and column-wise for those
// over positions, both as 16-byte pieces without bank conflicts (pieces of a row are permuted among the row's own 256 bytes).
#include "attn_bwd.hpp"
#include "rows16.hpp"

namespace splat {

// Operand layouts of mma4 (acc[16x16] += A[16x4] * B[4x16], v_mfma_f32_16x16x4_f32): lane (n = lane % 16, g = lane / 16) feeds row n
// of A and column n of B at contraction slot g, and holds rows 4g .. 4g + 3 of column n of the result.  Which index of the
// contraction a slot stands for is free as long as A and B agree:
//   * products over d take d = 16t + 4g + j in instruction 4t + j, so that one 16-byte read of a row feeds four instructions;
//   * products over positions take position 4g + j in instruction j: register j of a score tile is then the B operand as it
//     stands, without any exchange between lanes;
//   * of the output of those, row m of tile dt stands for d = 4m + dt (+ 64h), so that one 16-byte read of a row of the other
//     operand feeds four tiles, and a lane's 16 results of one row are 16 consecutive columns.
constexpr int kF32D = 128, kF32Tile = 16;  // positions per tile: 8 KB an operand

__device__ __forceinline__ f32x4 lds_load_f32x4(uint32_t addr) { return __builtin_bit_cast(f32x4, lds_load128(addr)); }

__global__ __launch_bounds__(256, 2) void attn_bwd_keys_f32_kernel(const BwdParams p) {
    constexpr int D = kF32D, BN = kF32Tile;
    constexpr int KQ = D / 16, DH = D / 64;
    constexpr int ROWB = D * 4, TILE = BN * ROWB, STAGE = 2 * TILE;
    constexpr int STATS = 512;       // lse and D of a tile's positions: 64 floats each, the first BN in use
    constexpr int RING = 2 * STATS;  // both stages' statistics come first
    constexpr int NI = TILE / 4096;  // copy blocks per wavefront and operand
    constexpr int CPR = ROWB / 16, RPI = 1024 / ROWB;
    constexpr float kLog2e = 1.4426950408889634f;

    extern __shared__ __attribute__((aligned(1024))) char smem[];

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

    // ---- the lane's share of its rows of A and B, resident: B operands of the products over d ----
    const int out_row = r0 + rs * (wave * 16 + n);
    int my_row = min(out_row, Lr - 1);
    if (p.row_map) my_row = min(max(p.row_map[my_row], 0), L - 1);
    float ar[D / 4], br[D / 4];
    auto load_row = [&](const float* row, float (&to)[D / 4]) {
#pragma unroll
        for (int t = 0; t < KQ; ++t) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(row + 16 * t + 4 * g);
#pragma unroll
            for (int j = 0; j < 4; ++j) to[4 * t + j] = x[j];
        }
    };
    load_row(ab + (int64_t)my_row * p.a_sl, ar);
    load_row(bb + (int64_t)my_row * p.b_sl, br);

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
    int total = 0;
    for (int sg = 0; sg < p.n_seg; ++sg) {
        const HalfWalk w = walk_of(sg);
        total += w.end - w.tile;
    }
    total = __builtin_amdgcn_readfirstlane(total);

    // ---- asynchronous copies of one tile (see tile_copy.hpp) ----
    auto position_row = [&](const HalfWalk& w, int j) { return min(max(w.pl.c0 + w.pl.cs * j, 0), L - 1); };
    uint32_t x_off[NI], y_off[NI];
    const char *x_next = nullptr, *y_next = nullptr;
    int64_t x_row = 0, y_row = 0;  // bytes from one tile row to the next
    bool off_fits = true;
    auto set_offsets = [&](const HalfWalk& w) {
        x_row = (int64_t)p.x_sl * 4 * w.pl.cs;
        y_row = (int64_t)p.y_sl * 4 * w.pl.cs;
        off_fits = x_row * RPI < ((int64_t)1 << 31) && y_row * RPI < ((int64_t)1 << 31);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int c = logical_chunk<ROWB, 1>((wave + 4 * i) * RPI + lane / CPR, lane % CPR) * 16;
            x_off[i] = (uint32_t)(x_row * (lane / CPR)) + c;
            y_off[i] = (uint32_t)(y_row * (lane / CPR)) + c;
        }
        const int64_t first = w.pl.c0 + (int64_t)w.pl.cs * BN * w.tile;
        x_next = reinterpret_cast<const char*>(xb) + first * p.x_sl * 4 + wave * RPI * x_row;
        y_next = reinterpret_cast<const char*>(yb) + first * p.y_sl * 4 + wave * RPI * y_row;
    };
    auto issue_next = [&](HalfWalk& w, int stage) {
        char* xs_w = smem + RING + stage * STAGE;
        const int j0 = w.tile * BN;
        if (off_fits && w.pl.c0 + w.pl.cs * (j0 + BN - 1) < L && w.pl.c0 + w.pl.cs * j0 >= 0) {
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                dma16_uniform(x_next + 4 * i * RPI * x_row, x_off[i], xs_w + (wave + 4 * i) * 1024);
                dma16_uniform(y_next + 4 * i * RPI * y_row, y_off[i], xs_w + TILE + (wave + 4 * i) * 1024);
            }
        } else {
            dma_tile<float, ROWB, BN, 1>(xs_w, wave, lane, [&](int row) { return xb + (int64_t)position_row(w, j0 + row) * p.x_sl; });
            dma_tile<float, ROWB, BN, 1>(xs_w + TILE, wave, lane, [&](int row) { return yb + (int64_t)position_row(w, j0 + row) * p.y_sl; });
        }
        const int q = position_row(w, j0 + (lane & (BN - 1)));
        if (wave == 0) dma4(lse_b + q, smem + stage * STATS);
        if (wave == 1) dma4(del_b + q, smem + stage * STATS + 256);
        x_next += BN * x_row;
        y_next += BN * y_row;
        if (++w.tile >= w.end) {
            ++w.seg;
            next_segment(w);
            if (w.seg < p.n_seg) set_offsets(w);
        }
    };

    // ---- LDS read addresses: of stage 0, moved on once a tile ----
    const uint32_t smem_base = lds_address(smem);
    uint32_t x_addr[KQ];  // row-wise: row n of a subtile, piece 4t + g (Y: TILE further)
    uint32_t c_addr[4];   // column-wise: row 4g + j, piece n
#pragma unroll
    for (int t = 0; t < KQ; ++t) x_addr[t] = smem_base + RING + lds_off<ROWB, true>(n, (16 * t + 4 * g) * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) c_addr[j] = smem_base + RING + lds_off<ROWB, true>(4 * g + j, 16 * n);
    uint32_t st_addr = smem_base + 16 * g;

    HalfWalk fetch, cur;
    fetch.seg = 0;
    next_segment(fetch);
    if (fetch.seg < p.n_seg) set_offsets(fetch);
    cur = fetch;
    PlanRec win_rec = {0, 0, 1, 0};
    if (cur.seg < p.n_seg) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + wave * 16 + n)];
    if (total > 0) issue_next(fetch, 0);

    f32x4 acc[4 * DH], acc2[4 * DH];
#pragma unroll
    for (int i = 0; i < 4 * DH; ++i) {
        acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        acc2[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const float c2 = p.scale_log2e;
    RowState rows;
    bool entered = false;
    int stage = 0;
#if defined(__HIP_DEVICE_COMPILE__)
    // the register operands are in their registers before the loop, so that no wait of the compiler's for them holds up the
    // copies in flight there
#pragma unroll
    for (int i = 0; i < D / 4; ++i) asm volatile("" ::"v"(ar[i]), "v"(br[i]));
#endif

    for (int it = 0; it < total; ++it) {
        if (!entered) {
            if (it > 0) win_rec = pt[plan_row_at(n_rb, p.n_seg, rb, cur.seg, k0 + wave * 16 + n)];
            const RowWin w = {win_rec.x, win_rec.y, win_rec.z};
            rows.template enter<BN>(w, win_rec.w, cur.pl.uniform != 0, cur.tile);
            entered = true;
        }
        const int j0 = cur.tile * BN;
        // this wavefront's copies of tile `it` have landed; after the barrier everybody's have, and everybody is done with
        // tile it - 1, whose stage the next fetch overwrites
        wait_loads<0>();
        __builtin_amdgcn_s_barrier();
        if (it + 1 < total) issue_next(fetch, stage ^ 1);

        if (j0 + BN > rows.lo_min && j0 < rows.hi_max) {
            // fragments are requested a phase ahead of their use
            f32x4 xf[KQ], yf[KQ];
#pragma unroll
            for (int t = 0; t < KQ; ++t) xf[t] = lds_load_f32x4(x_addr[t]);
            __builtin_amdgcn_sched_barrier(0);
            f32x4 s[1] = {f32x4{0.f, 0.f, 0.f, 0.f}}, ds = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < KQ; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) mma4(s[0], xf[t][j], ar[4 * t + j]);
#pragma unroll
            for (int t = 0; t < KQ; ++t) yf[t] = lds_load_f32x4(x_addr[t] + TILE);
            __builtin_amdgcn_sched_barrier(0);
            const f32x4 lse4 = lds_load_f32x4(st_addr), del4 = lds_load_f32x4(st_addr + 256);
#pragma unroll
            for (int t = 0; t < KQ; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) mma4(ds, yf[t][j], br[4 * t + j]);
            // ---- P = exp2(S * scale * log2e - lse * log2e); masked scores underflow to exactly 0.  dS = P (dP - D) ----
            if (!(j0 >= rows.lo_max && j0 + BN <= rows.hi_min)) rows.mask_tile(s, j0, g, cur.pl.uniform != 0);
            f32x4 xc[4][DH], yc[4][DH];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int hh = 0; hh < DH; ++hh) {
                    xc[j][hh] = lds_load_f32x4(c_addr[j] + 256 * hh);
                    yc[j][hh] = lds_load_f32x4(c_addr[j] + TILE + 256 * hh);
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s[0][j] = fast_exp2(fmaf(s[0][j], c2, -kLog2e * lse4[j]));
                ds[j] = s[0][j] * (ds[j] - del4[j]);
            }
            // ---- acc^T += X^T dS^T, acc2^T += Y^T P^T ----
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int hh = 0; hh < DH; ++hh)
#pragma unroll
                    for (int dt = 0; dt < 4; ++dt) {
                        mma4(acc[4 * hh + dt], xc[j][hh][dt], ds[j]);
                        mma4(acc2[4 * hh + dt], yc[j][hh][dt], s[0][j]);
                    }
        }
        if (!cur.pl.uniform) rows.next_tile();
        stage ^= 1;
        const int delta = stage == 0 ? -STAGE : STAGE;
#pragma unroll
        for (int t = 0; t < KQ; ++t) x_addr[t] += delta;
#pragma unroll
        for (int j = 0; j < 4; ++j) c_addr[j] += delta;
        st_addr += stage == 0 ? -STATS : STATS;
        if (++cur.tile >= cur.end) {
            ++cur.seg;
            next_segment(cur);
            entered = false;
        }
    }

    // ---- epilogue: a lane holds 16 consecutive columns (per 64) of its row ----
    if (out_row < Lr) {
        auto store_row = [&](void* base, const f32x4 (&a)[4 * DH], float scale) {
            float* row = (float*)base + b * p.o_sb + h * p.o_sh + (int64_t)out_row * p.o_sl;
#pragma unroll
            for (int hh = 0; hh < DH; ++hh)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4 x = {a[4 * hh][i] * scale, a[4 * hh + 1][i] * scale, a[4 * hh + 2][i] * scale, a[4 * hh + 3][i] * scale};
                    *reinterpret_cast<f32x4*>(row + 64 * hh + 16 * g + 4 * i) = x;
                }
        };
        store_row(p.out, acc, p.scale);
        store_row(p.out2, acc2, 1.0f);
    }
}

int launch_bwd_dkv_f32_d128(const BwdParams& p0, hipStream_t st) {
    begin_launch();
    BwdParams p = p0;
    p.total = p.B * p.H * 2 * p.n_row_blocks;
    p.by_blocks = divisor(2 * p.n_row_blocks), p.by_h = divisor(p.H);
    constexpr size_t lds = 2 * 512 + 2 * 2 * kF32Tile * kF32D * 4;
    auto kern = attn_bwd_keys_f32_kernel;
    static uint64_t lds_reserved = 0;
    if (int rc = reserve_dynamic_lds(&lds_reserved, reinterpret_cast<const void*>(kern), lds, "splat_attention_bwd_f32")) return rc;
    kern<<<((p.total + 7) / 8) * 8, 256, lds, st>>>(p);
    return check_launch("splat_attention_bwd_f32");
}

}  // namespace splat

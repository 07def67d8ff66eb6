// Parameters of the fused backward kernels (attention_bwd.hip: 16-bit types, attention_bwd_f32.hip: float32).
#pragma once
#include "attn_tile.hpp"

namespace splat {

struct BwdParams {
    const void* a;  // register operand A, one row per lane: Q (dQ), K (dK + dV)
    const void* b;  // register operand B: dO (dQ), V (dK + dV)
    const void* x;  // tile operand X: K (dQ), Q (dK + dV)
    const void* y;  // tile operand Y: V (dQ), dO (dK + dV)
    void* out;      // dQ, dK
    void* out2;     // dV (same strides as out)
    int64_t a_sb, a_sh, a_sl, b_sb, b_sh, b_sl, x_sb, x_sh, x_sl, y_sb, y_sh, y_sl, o_sb, o_sh, o_sl;
    const float* lse;    // [B*H, L], natural log, per query
    const float* delta;  // [B*H, L], D per query (dK + dV: written by the dQ launch before it on the stream)
    const void* o;       // dQ only: the forward's output, from which that launch computes D = rowsum(dO * O) ...
    int64_t oo_sb, oo_sh, oo_sl;
    float* delta_w;      // ... and where it stores it
    int B, H, L;
    int Lr;               // rows of the launch: L, or the number of rows of a rectangular keys' side (dK + dV of selected keys)
    const int* row_map;   // [Lr] or null: the row of A / B that row r of the mask stands for (r itself when null)
    float scale, scale_log2e;
    int n_seg, n_row_blocks, row_stride;
    int total;                // workgroups; with by_blocks (workgroups per head) and by_h (H) filled in by the launch
    Divisor by_blocks, by_h;
    const PlanRec* plan;  // plan table of the mask (dQ) or of its transpose (dK + dV), first variant
};

// dK + dV, 16-bit types (attention_bwd_pair.hip)
template <typename T>
int launch_bwd_pair(const BwdParams& dkv, int d, hipStream_t st);

// float32: dQ (which also computes and stores D), and dK + dV of the rows that `dkv` describes
int launch_bwd_dq_f32(const BwdParams& dq, int d, hipStream_t st);
int launch_bwd_dkv_f32(const BwdParams& dkv, int d, hipStream_t st);
int launch_bwd_dkv_f32_d128(const BwdParams& dkv, hipStream_t st);  // attention_bwd_f32_keys.hip

}  // namespace splat

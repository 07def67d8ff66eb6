// Kernel arguments of operators16.hip.
#pragma once
#include "acsr_plan.hpp"

namespace splat {

struct Operators16Params {
    const void *q, *k, *v;
    void *scores, *probs, *out;  // compressed rows of T slots twice, [B, H, L, d] contiguous
    int64_t q_sb, q_sh, q_sl;
    int64_t k_sb, k_sh, k_sd, k_sl;
    int64_t v_sb, v_sh, v_sl;
    int B, H, L, n_keys, d, T;
    float scale;
    int n_seg;
    SegPtrs seg[SPLAT_MAX_SEGMENTS];
    int n_row_blocks, total, row_stride;
    Divisor by_blocks, by_h;  // halves of row blocks per head, H
    const PlanRec* plan;
    int stream;  // whole pieces of scores and probabilities are stored around the caches
};

}  // namespace splat

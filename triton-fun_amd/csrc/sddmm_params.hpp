// Kernel arguments of the SDDMM kernels (sddmm.hip: every shape; sddmm_lines.hip, sddmm_rows16.hip: 16-bit types, operators_f32.hip: float32,
// up to 128 inner values).
#pragma once
#include <algorithm>
#include <type_traits>

#include "acsr_plan.hpp"
#include "softmax_rows.hpp"

namespace splat {

struct SddmmParams {
    const void* q;
    const void* k;
    void* out;
    int64_t q_sb, q_sh, q_sl;
    int64_t k_sb, k_sh, k_sd, k_sl;
    int B, H, L, n_keys, d, T;
    float scale;
    const float* row_lse;  // optional [B*H, L]: the output is exp(scale * score - row_lse[row]) instead of scale * score
    int out_dtype;
    int n_seg;
    SegPtrs seg[SPLAT_MAX_SEGMENTS];
    int n_row_blocks, total;
    int q_vec, k_vec;  // 16-byte loads are legal for q / k
    int out_vec;       // 16-bit outputs: every row's segment starts on a 16-byte boundary
    int out_stream;    // they are stored around the caches, in whole lines
    int row_stride;
    Divisor by_split, by_blocks, by_h;  // key_split, row blocks (or halves) per head, H: filled in by the launches that read them
    int key_split;  // workgroups per row block: each takes a contiguous share of every segment's tiles
    const PlanRec* plan;  // optional: the mask's plan table for 128-row blocks (variant for row-major K), else nullptr
    void* probs;  // optional, like out: the softmax of its rows as well, by the wavefronts that have stored them
    int probs_vec;  // T % 8 == 0, and out and probs start on 32-byte boundaries
};

// Whether softmax_own_rows pays.  (The figures are of the three operators as two launches and three.  16-bit forwards whose masks step alike within a block and whose
// rows are whole 16-byte pieces are one launch since, operators16.hip, but for several segments where that does not pay; here come the others, rows of other
// addresses or strides, blocks whose rows step differently, and calls of these two operators alone.)
//  Float32: rows of up to 256 slots (of 300 1.05 of the time of a launch for each, of 512 1.03 to 1.13).  16-bit
// types: rows of up to 512 slots and scores that the caches hold: causal masks of 33 to 256 slots, d = 64 and 128, the three operators 0.68 to 0.99 of
// the time up to 80 MB of scores, the two alone 0.82 to 1.25 from 100 to 170 MB.  (Scores and probabilities are stored through the caches
// then: 4096 rows of 200 slots, 16 heads, d = 128 60 -> 41 us, of which 53 around them.)  Of rows of more than 256 slots the workgroups that have
// the chip to themselves at a launch's end take longer than the other kernel's, so that their round (512 row blocks) has to be filled, to nine
// sixteenths, or to three quarters where rows end inside pieces: 283 slots, 520 / 640 / 720 / 1024 row blocks 1.06 / 1.03 / 1.03 / 0.98 of the time
// at d = 64, 1.04 / 1.02 / 1.00 / 0.96 at 128; 384 slots, 480 / 528 / 576 / 768 blocks 0.91 / 1.00 / 0.97 / 0.91 and 0.87 / 0.97 / 0.95 / 0.92.
// Not where a stride between a block's rows leaves most of them empty (224 heads of 128 rows, 21 slots with step 3: 18.7 -> 20.6).
inline bool own_rows_fit(const SddmmParams& p) {
    if (!p.probs || p.row_lse || (p.row_stride > 1 && p.L < 128 * p.row_stride)) return false;
    if (p.out_dtype == SPLAT_F32) return p.T <= 256;
    if (p.T > 512 || (int64_t)p.B * p.H * p.L * p.T * 2 > kCachedBytes) return false;
    const int64_t blocks = (int64_t)p.B * p.H * count_row_blocks(p.L, 128, p.row_stride), room = (blocks + 511) / 512 * 512;
    return p.T <= 256 || blocks <= 512 || blocks * 16 >= room * (p.probs_vec ? 9 : 12);
}

// The splits of a row over lanes that softmax_own_rows has, by the longest row of each: a sampled product's kernel is compiled without softmax
// and with one of them, which its launch chooses.  With all of them in every kernel, chosen there, 128 registers and up to 24 bytes of scratch
// instead of 68 to 122 and none held back launches with and without a softmax: bfloat16, 128 heads of 4096 rows, d = 64, the sampled product alone at 33
// slots 37.7 -> 33.0 us, the three operators at 60 slots 157 -> 141; 256 heads of 8192, 40 slots, d = 32 514 -> 459.
enum { kNoSoftmax, kSoftmax32, kSoftmax64, kSoftmax128, kSoftmax256, kSoftmax384, kSoftmax512 };
inline int own_rows_split(int T) {
    return T <= 32 ? kSoftmax32 : T <= 64 ? kSoftmax64 : T <= 128 ? kSoftmax128 : T <= 256 ? kSoftmax256 : T <= 384 ? kSoftmax384 : kSoftmax512;
}

// f(integral_constant<int, split>) with the split of this launch, of those from LO to HI that its kernel comes with; without softmax where the
// rows are longer than HI's (p.probs says which).
template <int LO, int HI, typename F>
inline void by_split_of(SddmmParams& p, F f) {
    const int split = std::max<int>(own_rows_split(p.T), LO);
    if (split > HI) p.probs = nullptr;
    if (!p.probs) return f(std::integral_constant<int, kNoSoftmax>{});
    static_for<HI - LO + 1>([&](auto i) {
        constexpr int S = LO + decltype(i)::value;
        if (split == S) f(std::integral_constant<int, S>{});
    });
}

// The softmax of the 16 rows r0 + rs * k of head bh that this wavefront, and nobody else, has stored: they come from the cache, and a launch
// of their own is spared.  (The bits are launch_softmax's: see softmax_rows.)  ALIGNED: as there; rows of any length go through the other one.
// float16, 16 heads of 2000 rows, 129 slots, d = 80, the three operators: 26.7 -> 21 us; bfloat16, 208 heads of 128 rows, 64 slots: 16.7 -> 13.6.
template <typename T, int SPLIT, bool ALIGNED>
__device__ __forceinline__ void softmax_own_rows(const SddmmParams& p, int bh, int r0, int rs) {
    if (r0 >= p.L) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // stores and the loads that follow them are not ordered otherwise
    SoftmaxSegs segs;
    segs.n = p.n_seg;
#pragma unroll
    for (int k = 0; k < SPLAT_MAX_SEGMENTS; ++k) segs.nnz[k] = k < p.n_seg ? p.seg[k].nnz : p.seg[0].nnz, segs.off[k] = p.seg[k].slot_offset;
    // lanes a row and chunks a lane; float32 a lane for each chunk
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int LPR = SPLIT == kSoftmax32 ? 4 : F32 ? (SPLIT == kSoftmax64 ? 8 : SPLIT == kSoftmax128 ? 16 : 32) : SPLIT >= kSoftmax384 || (SPLIT == kSoftmax256 && ALIGNED) ? 16 : 8;
    constexpr int NCH = F32 || SPLIT <= kSoftmax64 ? 1 : SPLIT == kSoftmax128 || (SPLIT == kSoftmax256 && ALIGNED) ? 2 : SPLIT == kSoftmax384 ? 3 : 4;
    constexpr int RPW = 64 / LPR, RIF = std::min(16 / RPW, NCH == 1 ? 4 : SPLIT == kSoftmax512 ? 1 : 2);
    const int lane = threadIdx.x & 63;
    const int64_t first = (int64_t)bh * p.L;
    for (int k0 = 0; k0 < 16; k0 += RPW * RIF) {
        if (r0 + rs * k0 >= p.L) break;
        softmax_rows<T, T, NCH, LPR, RIF, ALIGNED, false>((const T*)p.out, (T*)p.probs, segs, p.T, [&](int i, int64_t& row, int& in_head) {
            const int at = r0 + rs * (k0 + RPW * i + lane / LPR);
            in_head = at < p.L ? at : r0;
            row = first + in_head;
            return at < p.L;
        });
    }
}

// Launches the line-wise kernel when the problem has its shape (see sddmm_lines.hip); returns 1 when it did, 2 when it took the
// softmax as well, 0 when the general kernel has to run, a negative code on errors.  `p` is complete except for key_split / total.
int launch_sddmm_lines(const char* who, const SddmmParams& p, int in_dtype, hipStream_t st);
// The same for 16-bit launches of few row blocks (see sddmm_rows16.hip); `kt`: K is stored along the keys.
int launch_sddmm_rows16(const SddmmParams& p, int in_dtype, bool kt, hipStream_t st);
// The same for float32 inputs (see operators_f32.hip).
int launch_sddmm_f32(const SddmmParams& p, bool kt, hipStream_t st);

}  // namespace splat

// ACSR builder and mask generators.
//
// splat_acsr_build, splat_acsr_build_record: one wavefront per mask row streams the row once (16-byte loads), reducing the byte sum (nnz), the first two columns whose byte equals 1 (the affine map's anchors a < b) and the
// first/last nonzero column.  The first wavefront of a workgroup then evaluates the 2x2 solve of acsr_helpers.py:122 for up to 64 of its rows,
// a lane each, in closed form in double precision and rounds to float32, which is what the reference's
// float64 -> torch.FloatTensor conversion stores.  The per-row-block span pairs (acsr_helpers.py:135-140) come from the
// same kernel, or, with the summary on the device, from a second, tiny one.  HBM-bound: rows*ld bytes in, 28*rows out.
#include "splat_common.hpp"

namespace splat {

constexpr int kInf = 0x7fffffff;

// 0x80 in every byte of y that is zero (exact, no borrow artefacts).
__device__ __forceinline__ uint32_t zero_bytes(uint32_t y) {
    return ~(((y & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | y | 0x7F7F7F7Fu);
}

struct RowScan {
    uint32_t sum;  // sum of byte values
    int m1, m2;    // two smallest columns whose byte == 1
    int first, last;  // first / last nonzero column

    __device__ __forceinline__ void init() {
        sum = 0;
        m1 = m2 = first = kInf;
        last = -1;
    }
    __device__ __forceinline__ void add_one(int col) {
        if (col < m1) {
            m2 = m1;
            m1 = col;
        } else if (col < m2 && col != m1) {
            m2 = col;
        }
    }
    // 16 bytes of columns behind all that this lane has seen: bit c of a 16-bit mask for column col0 + c
    __device__ __forceinline__ void piece(const u32x4& x, int col0) {
        const uint32_t w[4] = {x.x, x.y, x.z, x.w};
        uint32_t nz[4], one[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            sum = __builtin_amdgcn_sad_u8(w[k], 0u, sum);
            nz[k] = ~zero_bytes(w[k]) & 0x80808080u;
            one[k] = zero_bytes(w[k] ^ 0x01010101u);
        }
        const uint32_t live = columns(nz), ones = columns(one);
        if (live) {
            first = min(first, col0 + __builtin_ctz(live));
            last = col0 + 31 - __builtin_clz(live);
        }
        if (ones && m2 == kInf) {
            const int a = col0 + __builtin_ctz(ones);
            const uint32_t rest = ones & (ones - 1);
            const int b = rest ? col0 + __builtin_ctz(rest) : kInf;
            m2 = m1 == kInf ? b : a;
            m1 = min(m1, a);
        }
    }
    // the 0x80 of 16 bytes as 16 bits: a dot product with the powers of two (sums of at most 128 * 255)
    static __device__ __forceinline__ uint32_t columns(const uint32_t (&f)[4]) {
        const uint32_t lo = __builtin_amdgcn_udot4(f[1], 0x80402010u, __builtin_amdgcn_udot4(f[0], 0x08040201u, 0u, false), false);
        const uint32_t hi = __builtin_amdgcn_udot4(f[3], 0x80402010u, __builtin_amdgcn_udot4(f[2], 0x08040201u, 0u, false), false);
        return (lo >> 7) | (hi << 1);
    }
    __device__ __forceinline__ void byte(uint32_t x, int col) {
        if (x == 0) return;
        sum += x;
        first = min(first, col);
        last = max(last, col);
        if (x == 1) add_one(col);
    }
    __device__ __forceinline__ void wave_reduce() {
        sum = (uint32_t)over_lanes<64>((int)sum, [](int a, int b) { return a + b; });
        const int a = wave_min_i(m1);  // (in one lane, whose second one is the only other candidate it has)
        m2 = wave_min_i(m1 == a ? m2 : m1);
        m1 = a;
        first = wave_min_i(first);
        last = wave_max_i(last);
    }
};

// The summary's starting values, written by the first workgroup of the rows kernel (no kernel of its own): the rows
// kernels themselves never touch the summary otherwise, the span kernel that follows them reduces into it.
__device__ __forceinline__ void init_summary(int32_t* summary) {
    if (blockIdx.x == 0 && threadIdx.x < 8) summary[threadIdx.x] = (threadIdx.x == 2 || threadIdx.x == 5) ? 0x7fffffff : 0;
}
constexpr float kUnpackFailed = 0.0f;  // stored as a row's sTod_lin (a real step is >= 1) until the span kernel has counted it

// Where a build's arrays go.  `twin` / `twin_i`, when not 0, are the distances in elements from every float32 / int32 array to its
// duplicate: a caller that keeps a build and hands out another copy gets both from one kernel.
struct RowOut {
    float *dTos_lin, *dTos_trans, *sTod_lin, *sTod_trans, *nnz;
    int32_t *row_first, *row_last;
    float *span_start, *span_end;
    int64_t twin, twin_i;
    __device__ __forceinline__ void put(float* p, int i, float x) const {
        p[i] = x;
        if (twin) p[i + twin] = x;
    }
    __device__ __forceinline__ void put(int32_t* p, int i, int32_t x) const {
        p[i] = x;
        if (twin_i) p[i + twin_i] = x;
    }
};

// What one row contributes once its scan is reduced: the closed-form 2x2 solve.  (The summary extrema are
// reduced per row block: per-row atomics on one address cost more than streaming the whole mask.)  Returns whether the
// row is one the reference asserts on (acsr_helpers.py:119); its stored step is `failed_lin`.
__device__ __forceinline__ bool finish_row(const RowScan& s, int row, int cols, const RowOut& o, float failed_lin, float* lin_out,
                                           float* trans_out) {
    const int nnz = (int)s.sum;
    double x0 = 1.0, x1 = 0.0;
    int step = 1;
    bool failed = false;
    if (nnz > 1) {
        if (s.m1 == kInf || s.m2 == kInf) {
            failed = true;
        } else {
            step = s.m2 - s.m1;
            x0 = 1.0 / (double)step;
            // the solve yields +0.0 (not -0.0) for a == 0
            x1 = (s.m1 == 0) ? 0.0 : -(double)s.m1 / (double)step;
        }
    }
    *lin_out = failed ? failed_lin : (float)step;
    *trans_out = (float)fabs(x1);
    o.put(o.dTos_lin, row, (float)x0);
    o.put(o.dTos_trans, row, (float)x1);
    o.put(o.sTod_lin, row, *lin_out);
    o.put(o.sTod_trans, row, *trans_out);
    o.put(o.nnz, row, (float)nnz);
    if (o.row_first) o.put(o.row_first, row, (s.first == kInf) ? cols : s.first);
    if (o.row_last) o.put(o.row_last, row, s.last);
    return failed;
}

// The rows of one span block folded together: span_start = min(cols, min_r trans_r), span_end = max(-1, max_r nnz_r*lin_r +
// trans_r), evaluated in double from the exact integers (a, lin, nnz) and rounded once to float32, and the block's share of
// the summary: T = max nnz, smallest / largest column step over rows with nnz > 1, how many of these have a first column that
// is not congruent to the row index modulo their step (for callers of the C interface: the grouping here asks the residues), the
// smallest / largest residue of the first column less the row index, and how many rows the reference would have asserted on.
struct BlockFold {
    float lo, hi;  // (a rounding is monotone: the least of the rounded is the least, rounded)
    int t_max, step_min, step_max, off_phase, res_min, res_max, failed;
    __device__ __forceinline__ void init(int cols) {
        lo = (float)cols, hi = -1.0f;
        t_max = 0, step_min = 0x7fffffff, step_max = 0, off_phase = 0, res_min = 0x7fffffff, res_max = 0, failed = 0;
    }
    __device__ __forceinline__ void row(int r, float linf, float trans, int cnt) {
        const int lin = (int)linf;
        const int a = (int)rintf(linf * trans);
        const double t = (double)a / (double)lin;
        lo = fminf(lo, (float)t);
        hi = fmaxf(hi, (float)((double)((int64_t)cnt * lin) + t));
        t_max = max(t_max, cnt);
        if (cnt > 1) {
            step_min = min(step_min, lin);
            step_max = max(step_max, lin);
            const int rem = (a - r) % lin;
            const int res = rem < 0 ? rem + lin : rem;
            off_phase += res != 0;
            res_min = min(res_min, res);
            res_max = max(res_max, res);
        }
    }
    __device__ __forceinline__ void wave_reduce() {
        auto add = [](int a, int b) { return a + b; };
        lo = over_lanes<64>(lo, [](float a, float b) { return fminf(a, b); }), hi = wave_max(hi);
        t_max = wave_max_i(t_max), step_min = wave_min_i(step_min), step_max = wave_max_i(step_max);
        res_min = wave_min_i(res_min), res_max = wave_max_i(res_max);
        off_phase = over_lanes<64>(off_phase, add), failed = over_lanes<64>(failed, add);
    }
};

// A workgroup takes `per_block` consecutive rows, a wavefront one row at a time: 16-byte pieces from the row's first aligned
// address on (rows of any pitch), NB per lane in flight, and single bytes at the two ends.  Sixteen wavefronts and at most
// 64 registers, so that a CU holds two workgroups: a mask of 8192 rows is one wave of workgroups over the chip.  What a
// wavefront found goes to LDS; the first one solves up to 64 rows at once, a lane each, and stores them side by side.
//
// FOLD: the workgroup's rows are one span block; its spans and its share of the summary (7 integers, 8 apart, into memory
// that the host reads) come from the same kernel.  With a second kernel for the spans, which walks 16 rows a thread with
// few threads, and the summary read back through a copy, an 8192 x 8192 mask took 23 us on the GPU in two kernels and 95 us
// for the whole call.  One kernel in which every wavefront's first lane solved its row and the workgroup's first thread
// folded the wavefronts' one by one: 17.4 us.  This one, whose pieces are read without a branch per dword: 12.7 us with
// four pieces in flight and 15.1 with eight, whose code and spills (with the fold) cost more than they hide; the 67 MB of that mask come
// from the last-level cache, with caches flushed it takes 16.3 (23.7 before, 21.3 with eight).
// Rows of 16384 bytes, 268 MB, bound by HBM: with the fold four pieces 49.7 / 52.5 flushed, eight 50.3 / 55.0; without the fold and its
// registers (splat_acsr_build, both kernels) eight do not spill, and win where the cache does not hold the mask: 55.1 / 57.4
// against 59.5 / 62.6, at rows of 12288 bytes 35.5 / 37.8 against 35.2 / 37.9, of 8192 23.3 / 26.5 against 22.7 / 26.3.
constexpr int kRowWaves = 16;
constexpr int kLongRow = 12288;  // bytes a row from which on eight pieces are in flight, without FOLD
template <bool FOLD, int NB = 4>
__global__ __launch_bounds__(64 * kRowWaves, 8) void acsr_rows_kernel(const uint8_t* __restrict__ mask, int rows, int cols, int64_t ld,
                                                                      int per_block, RowOut o, int32_t* __restrict__ summary,
                                                                      int32_t* __restrict__ shares) {
    __shared__ RowScan s_row[2][64];
    if constexpr (!FOLD) init_summary(summary);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_waves = blockDim.x >> 6;
    const int r_end = min(rows, ((int)blockIdx.x + 1) * per_block);
    BlockFold f;
    f.init(cols);
    int turn = 0;
    for (int base = blockIdx.x * per_block; base < r_end; base += 64, turn ^= 1) {
        const int n = min(64, r_end - base);
        for (int k = wave; k < n; k += n_waves) {
            const uint8_t* p = mask + (int64_t)(base + k) * ld;
            const int head = min(cols, (int)(-reinterpret_cast<uintptr_t>(p) & 15));
            const int nvec = (cols - head) >> 4;
            const u32x4* pv = reinterpret_cast<const u32x4*>(p + head);
            RowScan s;
            s.init();
            const int tail0 = head + (nvec << 4);  // fewer than 16 bytes before `head` and fewer than 16 from `tail0` on
            uint32_t edge = 0;
            const int edge_col = lane < 16 ? lane : tail0 + lane - 16;
            if (lane < 16 ? lane < head : (lane < 32 && edge_col < cols)) edge = p[edge_col];
            for (int i0 = lane; i0 < nvec; i0 += 64 * NB) {
                u32x4 xs[NB];
#pragma unroll
                for (int u = 0; u < NB; ++u) xs[u] = i0 + 64 * u < nvec ? __builtin_nontemporal_load(pv + i0 + 64 * u) : u32x4{0, 0, 0, 0};
#pragma unroll
                for (int u = 0; u < NB; ++u)
                    if ((xs[u].x | xs[u].y | xs[u].z | xs[u].w) != 0) s.piece(xs[u], head + ((i0 + 64 * u) << 4));
            }
            s.byte(edge, edge_col);
            s.wave_reduce();
            if (lane == 0) s_row[turn][k] = s;
        }
        __syncthreads();  // (one is enough: wavefront 0 has read the half before when it comes to the next one)
        if (wave == 0 && lane < n) {
            float lin, trans;
            const RowScan s = s_row[turn][lane];
            const bool failed = finish_row(s, base + lane, cols, o, FOLD ? 1.0f : kUnpackFailed, &lin, &trans);
            if constexpr (FOLD) {
                f.failed += failed;
                f.row(base + lane, lin, trans, (int)s.sum);
            }
        }
    }
    if constexpr (FOLD) {
        if (wave == 0) {
            f.wave_reduce();
            if (lane == 0) {
                o.put(o.span_start, blockIdx.x, f.lo);
                o.put(o.span_end, blockIdx.x, f.hi);
                int4* const mine = reinterpret_cast<int4*>(shares) + 2 * blockIdx.x;
                mine[0] = make_int4(f.t_max, f.failed, f.step_min, f.step_max);
                mine[1] = make_int4(f.off_phase, f.res_min, f.res_max, 0);
            }
        }
    }
}

// One thread per row block: spans and summary (BlockFold) of rows that are in memory.
__global__ __launch_bounds__(256) void acsr_spans_kernel(float* __restrict__ sTod_lin,
                                                         const float* __restrict__ sTod_trans,
                                                         const float* __restrict__ nnz, int rows, int cols,
                                                         int block_height, float* __restrict__ span_start,
                                                         float* __restrict__ span_end, int32_t* __restrict__ summary) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    const int n_blocks = (rows + block_height - 1) / block_height;
    BlockFold f;
    f.init(cols);
    if (g < n_blocks) {
        const int r1 = min(rows, (g + 1) * block_height);
        for (int r = g * block_height; r < r1; ++r) {
            float linf = sTod_lin[r];
            if (linf == kUnpackFailed) {  // a row the reference would have asserted on: counted, then stored as (1, 0) like
                ++f.failed;               // the rows with at most one live column
                linf = 1.0f;
                sTod_lin[r] = linf;
            }
            f.row(r, linf, sTod_trans[r], (int)nnz[r]);
        }
        span_start[g] = f.lo;
        span_end[g] = f.hi;
    }
    const int t_max = wave_max_i(f.t_max);
    const int step_min = wave_min_i(f.step_min);
    const int step_max = wave_max_i(f.step_max);
    const int res_min = wave_min_i(f.res_min);
    const int res_max = wave_max_i(f.res_max);
    const int off_phase = (int)wave_sum((float)f.off_phase);  // at most 64 * block_height per wavefront: exact in float
    const int failed = (int)wave_sum((float)f.failed);
    if ((threadIdx.x & 63) == 0) {
        if (failed) atomicAdd(&summary[1], failed);
        atomicMax(&summary[0], t_max);
        atomicMin(&summary[2], step_min);
        atomicMax(&summary[3], step_max);
        if (off_phase) atomicAdd(&summary[4], off_phase);
        atomicMin(&summary[5], res_min);
        atomicMax(&summary[6], res_max);
    }
}

__device__ __forceinline__ bool mask_pred(int pattern, int64_t i, int64_t j, int64_t p0, int64_t p1) {
    if (pattern & SPLAT_MASK_TRANSPOSED) {  // entry (i, j) of the transposed pattern is entry (j, i) of the pattern
        const int64_t t = i;
        i = j;
        j = t;
        pattern &= ~SPLAT_MASK_TRANSPOSED;
    }
    switch (pattern) {
        case SPLAT_MASK_BLOCKED: {
            if (i < p0) return j < p0;
            int64_t start = (i / p0 - 1) * p0;
            return start <= j && j < start + 2 * p0;
        }
        case SPLAT_MASK_WINDOWED:
            return i - p0 <= j && j <= i + p0;
        case SPLAT_MASK_CAUSAL_WINDOWED:
            return i - p0 <= j && j <= i;
        case SPLAT_MASK_DILATED: {
            int64_t rel = j - (i - (p0 * p1) / 2);
            return rel >= 0 && rel < p0 * p1 && rel % p1 == 0;
        }
        case SPLAT_MASK_STRIDED_LOCAL:
            return j <= i && j > i - p0;
        case SPLAT_MASK_STRIDED_FAR:
            return j <= i - p0 && j % p1 == p1 - 1;
    }
    return false;
}

// What a scan of row i of the s x s pattern would find, in closed form: every pattern's row is an arithmetic
// progression of columns (first, step, count), clipped to [0, s).
__device__ __forceinline__ RowScan pattern_row(int pattern, int64_t i, int64_t s, int64_t p0, int64_t p1) {
    int64_t first = 0, step = 1, count = 0;
    switch (pattern) {
        case SPLAT_MASK_BLOCKED: {
            const int64_t start = (i < p0) ? 0 : (i / p0 - 1) * p0;
            const int64_t end = (i < p0) ? p0 : start + 2 * p0;  // exclusive
            first = start;
            count = min(end, s) - start;
            break;
        }
        case SPLAT_MASK_WINDOWED:
            first = max((int64_t)0, i - p0);
            count = min(s - 1, i + p0) - first + 1;
            break;
        case SPLAT_MASK_CAUSAL_WINDOWED:
            first = max((int64_t)0, i - p0);
            count = min(s - 1, i) - first + 1;
            break;
        case SPLAT_MASK_STRIDED_LOCAL:
            first = max((int64_t)0, i - p0 + 1);
            count = min(s - 1, i) - first + 1;
            break;
        case SPLAT_MASK_DILATED: {
            const int64_t base = i - (p0 * p1) / 2;  // column of t = 0; columns base + t * p1, t in [0, p0)
            const int64_t t_lo = base < 0 ? (-base + p1 - 1) / p1 : 0;
            const int64_t room = s - 1 - base;
            const int64_t t_hi = room < 0 ? -1 : min(p0 - 1, room / p1);
            step = p1;
            first = base + t_lo * p1;
            count = t_hi - t_lo + 1;
            break;
        }
        case SPLAT_MASK_STRIDED_FAR: {
            const int64_t room = min(i - p0, s - 1) - (p1 - 1);  // columns p1 - 1 + t * p1 <= i - p0
            step = p1;
            first = p1 - 1;
            count = room < 0 ? 0 : room / p1 + 1;
            break;
        }
        // ---- rows of the transposed patterns = columns of the patterns: which rows keep column i ----
        case SPLAT_MASK_TRANSPOSED | SPLAT_MASK_BLOCKED: {
            // row block b >= 1 keeps column blocks b - 1 and b, row block 0 keeps column block 0: column block c is kept
            // by row blocks c and c + 1
            const int64_t c = i / p0;
            first = c * p0;
            count = min((c + 2) * p0, s) - first;
            break;
        }
        case SPLAT_MASK_TRANSPOSED | SPLAT_MASK_WINDOWED:
            first = max((int64_t)0, i - p0);
            count = min(s - 1, i + p0) - first + 1;
            break;
        case SPLAT_MASK_TRANSPOSED | SPLAT_MASK_CAUSAL_WINDOWED:
            first = i;
            count = min(s - 1, i + p0) - first + 1;
            break;
        case SPLAT_MASK_TRANSPOSED | SPLAT_MASK_STRIDED_LOCAL:
            first = i;
            count = min(s - 1, i + p0 - 1) - first + 1;
            break;
        case SPLAT_MASK_TRANSPOSED | SPLAT_MASK_DILATED: {
            // row r keeps column r - h + t * p1, t in [0, p0), h = p0 * p1 / 2: column i is kept by rows i + h - t * p1,
            // in ascending order base + u * p1, u in [0, p0)
            const int64_t base = i + (p0 * p1) / 2 - (p0 - 1) * p1;
            const int64_t u_lo = base < 0 ? (-base + p1 - 1) / p1 : 0;
            const int64_t room = s - 1 - base;
            const int64_t u_hi = room < 0 ? -1 : min(p0 - 1, room / p1);
            step = p1;
            first = base + u_lo * p1;
            count = u_hi - u_lo + 1;
            break;
        }
        case SPLAT_MASK_TRANSPOSED | SPLAT_MASK_STRIDED_FAR:
            // only columns congruent to p1 - 1 are kept, by every row from i + p0 on
            first = i + p0;
            count = (i % p1 == p1 - 1) ? s - first : 0;
            break;
    }
    RowScan r;
    r.init();
    if (count > 0) {
        r.sum = (uint32_t)count;
        r.m1 = r.first = (int)first;
        if (count > 1) r.m2 = (int)(first + step);
        r.last = (int)(first + (count - 1) * step);
    }
    return r;
}

__global__ __launch_bounds__(256) void acsr_rows_pattern_kernel(int pattern, int s, int64_t p0, int64_t p1, RowOut o,
                                                                int32_t* __restrict__ summary) {
    init_summary(summary);
    const int row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= s) return;
    float lin, trans;
    finish_row(pattern_row(pattern, row, s, p0, p1), row, s, o, kUnpackFailed, &lin, &trans);
}

__global__ __launch_bounds__(256) void mask_generate_kernel(uint8_t* __restrict__ mask, int rows, int cols,
                                                            int64_t ld, int pattern, int64_t p0, int64_t p1,
                                                            int vec_ok) {
    const int chunks = (cols + 15) >> 4;
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= (int64_t)rows * chunks) return;
    const int i = (int)(id / chunks);
    const int c0 = (int)(id % chunks) << 4;
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int b = 0; b < 16; ++b) {
        int j = c0 + b;
        if (j < cols && mask_pred(pattern, i, j, p0, p1)) w[b >> 2] |= 1u << ((b & 3) * 8);
    }
    uint8_t* dst = mask + (int64_t)i * ld + c0;
    if (vec_ok && c0 + 16 <= cols) {
        *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
        for (int b = 0; b < 16 && c0 + b < cols; ++b) dst[b] = (uint8_t)((w[b >> 2] >> ((b & 3) * 8)) & 0xff);
    }
}

}  // namespace splat

using namespace splat;

extern "C" int splat_acsr_build(const uint8_t* mask, int64_t rows, int64_t cols, int64_t ld, int32_t block_height,
                                float* dTos_lin, float* dTos_trans, float* sTod_lin, float* sTod_trans, float* nnz,
                                float* span_start, float* span_end, int32_t* row_first, int32_t* row_last,
                                int32_t* summary, void* stream) {
    begin_launch();
    if (!mask || !dTos_lin || !dTos_trans || !sTod_lin || !sTod_trans || !nnz || !span_start || !span_end || !summary)
        return fail(SPLAT_E_NULL, "splat_acsr_build: null pointer argument");
    if (rows <= 0 || cols <= 0 || ld < cols || block_height <= 0)
        return fail(SPLAT_E_SHAPE, "splat_acsr_build: need rows > 0, cols > 0, ld >= cols, block_height > 0 (got %lld, %lld, %lld, %d)",
                    (long long)rows, (long long)cols, (long long)ld, block_height);
    // a row sum must fit int32 and columns must be exactly representable in float32 metadata
    if (rows > (1 << 23) || cols > (1 << 23))
        return fail(SPLAT_E_SHAPE, "splat_acsr_build: rows and cols are limited to 2^23 (got %lld, %lld)", (long long)rows, (long long)cols);
    hipStream_t st = (hipStream_t)stream;
    const RowOut out{dTos_lin, dTos_trans, sTod_lin, sTod_trans, nnz, row_first, row_last, nullptr, nullptr, 0, 0};
    const auto kern = cols > kLongRow ? acsr_rows_kernel<false, 8> : acsr_rows_kernel<false>;
    kern<<<(unsigned)((rows + kRowWaves - 1) / kRowWaves), 64 * kRowWaves, 0, st>>>(mask, (int)rows, (int)cols, ld, kRowWaves, out, summary, nullptr);
    const int n_blocks = (int)((rows + block_height - 1) / block_height);
    acsr_spans_kernel<<<(n_blocks + 255) / 256, 256, 0, st>>>(sTod_lin, sTod_trans, nnz, (int)rows, (int)cols, block_height,
                                                               span_start, span_end, summary);
    return check_launch("splat_acsr_build");
}

extern "C" int splat_acsr_build_record(const uint8_t* mask, int64_t rows, int64_t cols, int64_t ld, int32_t block_height, float* record,
                                       int32_t* extents, int32_t duplicate, int32_t* shares, void* stream) {
    begin_launch();
    if (!mask || !record || !extents || !shares) return fail(SPLAT_E_NULL, "splat_acsr_build_record: null pointer argument");
    if (rows <= 0 || cols <= 0 || ld < cols || block_height <= 0 || rows > (1 << 23) || cols > (1 << 23))
        return fail(SPLAT_E_SHAPE, "splat_acsr_build_record: need 0 < rows, cols <= 2^23, ld >= cols, block_height > 0 (got %lld, %lld, %lld, %d)",
                    (long long)rows, (long long)cols, (long long)ld, block_height);
    const int64_t n_blocks = (rows + block_height - 1) / block_height;
    const int64_t row_step = (rows + 63) & ~(int64_t)63, span_step = (n_blocks + 63) & ~(int64_t)63;
    if ((reinterpret_cast<uintptr_t>(record) & 3) != 0 || (reinterpret_cast<uintptr_t>(extents) & 3) != 0 ||
        (reinterpret_cast<uintptr_t>(shares) & 15) != 0)
        return fail(SPLAT_E_ALIGN, "splat_acsr_build_record: misaligned record, extents or shares");
    float* const f = record;
    const RowOut out{f, f + row_step, f + 2 * row_step, f + 3 * row_step, f + 4 * row_step, extents, extents + row_step,
                     f + 5 * row_step, f + 5 * row_step + span_step, duplicate ? 5 * row_step + 2 * span_step : 0,
                     duplicate ? 2 * row_step : 0};
    const int waves = (int)min((int64_t)kRowWaves, min((int64_t)block_height, rows));
    acsr_rows_kernel<true><<<(unsigned)n_blocks, 64 * waves, 0, (hipStream_t)stream>>>(mask, (int)rows, (int)cols, ld, block_height, out,
                                                                                       nullptr, shares);
    return check_launch("splat_acsr_build_record");
}

static int check_pattern(const char* who, int64_t s, int32_t pattern, int64_t p0, int64_t p1) {
    if (s <= 0 || s > (1 << 23)) return fail(SPLAT_E_SHAPE, "%s: need 0 < s <= 2^23 (got %lld)", who, (long long)s);
    const int base = pattern & ~SPLAT_MASK_TRANSPOSED;
    if (pattern < 0 || base < SPLAT_MASK_BLOCKED || base > SPLAT_MASK_STRIDED_FAR)
        return fail(SPLAT_E_UNSUPPORTED, "%s: unknown pattern %d", who, pattern);
    const bool needs_p1 = base == SPLAT_MASK_DILATED || base == SPLAT_MASK_STRIDED_FAR;
    if (p0 < 0 || (base == SPLAT_MASK_BLOCKED && p0 <= 0) || (needs_p1 && p1 <= 0))
        return fail(SPLAT_E_SHAPE, "%s: bad pattern parameters p0=%lld p1=%lld", who, (long long)p0, (long long)p1);
    return 0;
}

extern "C" int splat_acsr_build_pattern(int32_t pattern, int64_t s, int64_t p0, int64_t p1, int32_t block_height,
                                        float* dTos_lin, float* dTos_trans, float* sTod_lin, float* sTod_trans, float* nnz,
                                        float* span_start, float* span_end, int32_t* row_first, int32_t* row_last,
                                        int32_t* summary, void* stream) {
    begin_launch();
    const char* who = "splat_acsr_build_pattern";
    if (!dTos_lin || !dTos_trans || !sTod_lin || !sTod_trans || !nnz || !span_start || !span_end || !summary)
        return fail(SPLAT_E_NULL, "%s: null pointer argument", who);
    if (block_height <= 0) return fail(SPLAT_E_SHAPE, "%s: block_height must be > 0 (got %d)", who, block_height);
    if (int rc = check_pattern(who, s, pattern, p0, p1)) return rc;
    if (p0 > (1 << 23) || p1 > (1 << 23)) return fail(SPLAT_E_SHAPE, "%s: pattern parameters are limited to 2^23", who);
    hipStream_t st = (hipStream_t)stream;
    const RowOut out{dTos_lin, dTos_trans, sTod_lin, sTod_trans, nnz, row_first, row_last, nullptr, nullptr, 0, 0};
    acsr_rows_pattern_kernel<<<(unsigned)((s + 255) / 256), 256, 0, st>>>(pattern, (int)s, p0, p1, out, summary);
    const int n_blocks = (int)((s + block_height - 1) / block_height);
    acsr_spans_kernel<<<(n_blocks + 255) / 256, 256, 0, st>>>(sTod_lin, sTod_trans, nnz, (int)s, (int)s, block_height, span_start,
                                                               span_end, summary);
    return check_launch(who);
}

extern "C" int splat_mask_generate(uint8_t* mask, int64_t rows, int64_t cols, int64_t ld, int32_t pattern, int64_t p0,
                                   int64_t p1, void* stream) {
    begin_launch();
    if (!mask) return fail(SPLAT_E_NULL, "splat_mask_generate: null mask");
    if (rows <= 0 || cols <= 0 || ld < cols || rows > (1 << 23) || cols > (1 << 23))
        return fail(SPLAT_E_SHAPE, "splat_mask_generate: bad shape rows=%lld cols=%lld ld=%lld", (long long)rows, (long long)cols, (long long)ld);
    {
        const int base = pattern & ~SPLAT_MASK_TRANSPOSED;
        if (pattern < 0 || base < SPLAT_MASK_BLOCKED || base > SPLAT_MASK_STRIDED_FAR)
            return fail(SPLAT_E_UNSUPPORTED, "splat_mask_generate: unknown pattern %d", pattern);
        const bool needs_p1 = base == SPLAT_MASK_DILATED || base == SPLAT_MASK_STRIDED_FAR;
        if (p0 < 0 || (base == SPLAT_MASK_BLOCKED && p0 <= 0) || (needs_p1 && p1 <= 0))
            return fail(SPLAT_E_SHAPE, "splat_mask_generate: bad pattern parameters p0=%lld p1=%lld", (long long)p0, (long long)p1);
    }
    const int vec_ok = ((reinterpret_cast<uintptr_t>(mask) & 15) == 0 && (ld & 15) == 0) ? 1 : 0;
    const int64_t n = rows * ((cols + 15) >> 4);
    mask_generate_kernel<<<(unsigned)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>(mask, (int)rows, (int)cols, ld, pattern, p0, p1, vec_ok);
    return check_launch("splat_mask_generate");
}

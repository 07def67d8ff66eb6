// Row softmax over the live slots of compressed [BH, L, T] score rows.
//
// One wavefront owns whole rows.  A row's live slots are read once with 16/32-byte loads (8 elements
// per lane per step), kept in registers, reduced with wavefront shuffles (max, then sum of
// exp2((x - max) * log2 e)) and written back once; dead slots (s >= nnz) are neither read as data nor
// written.  HBM-bound: 2 * live slots * element size bytes per row.  Rows whose length is not a multiple of 8 are read and written in
// pieces that start where the row does, the last one ending with it: next to the aligned pieces of the buffer that cover a row, whose ends
// had to be stored slot by slot, 262144 rows of 191 slots take 37.8 -> 32.9 us, of 255 75.7 -> 42.2, of 277 84 -> 75, float32, 191 slots
// 99 -> 79.  Rows longer than 2048 slots take a three-pass kernel that re-reads the row from cache.
#include <type_traits>

#include "softmax_rows.hpp"

namespace splat {

template <typename Tin, typename Tout, int NCH, int LPR, int RIF, bool ALIGNED, bool AROUND>
__global__ __launch_bounds__(256) void softmax_rows_vec(const Tin* __restrict__ x, Tout* __restrict__ y, SoftmaxSegs segs,
                                                        int64_t n_rows, int L, int T, Divisor by_l) {
    load_args(x, y, n_rows, L, T, by_l.m, by_l.shift, segs.n, segs.nnz[0], segs.off[0]);
    constexpr int RPW = 64 / LPR;  // rows per wavefront and group
    const int64_t row0 = (((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * RIF) * RPW + ((threadIdx.x & 63) / LPR);
    if (RPW == 1 && row0 >= n_rows) return;
    softmax_rows<Tin, Tout, NCH, LPR, RIF, ALIGNED, AROUND>(x, y, segs, T, [&](int i, int64_t& row, int& in_head) {
        const int64_t at = row0 + (int64_t)i * RPW;
        row = at < n_rows ? at : n_rows - 1;
        in_head = n_rows < ((int64_t)1 << 31) ? (int)row - quotient((int)row, by_l) * L : (int)(row % L);
        return at < n_rows;
    });
}

template <typename Tin, typename Tout>
__global__ __launch_bounds__(256) void softmax_rows_any(const Tin* __restrict__ x, Tout* __restrict__ y, SoftmaxSegs segs,
                                                        int64_t n_rows, int L, int T) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n_rows) return;
    LiveRanges lr;
    lr.load(segs, (int)(row % L), T);
    const Tin* xr = x + row * (int64_t)T;
    Tout* yr = y + row * (int64_t)T;
    float mx = kNegBig;
    for (int s = lane; s < T; s += 64)
        if (lr.live(s)) mx = fmaxf(mx, (float)xr[s]);
    mx = wave_max(mx);
    const float mb = mx * kLog2e;
    float sum = 0.f;
    for (int s = lane; s < T; s += 64)
        if (lr.live(s)) sum += fast_exp2(fmaf((float)xr[s], kLog2e, -mb));
    sum = wave_sum(sum);
    const float inv = sum > 0.f ? 1.0f / sum : 0.f;
    // in-place safe: every lane rewrites only the slots it reads in this loop
    for (int s = lane; s < T; s += 64)
        if (lr.live(s)) yr[s] = (Tout)(fast_exp2(fmaf((float)xr[s], kLog2e, -mb)) * inv);
}

template <typename Tin, typename Tout>
static int launch_softmax(const void* x, void* y, const SoftmaxSegs& segs, int64_t n_rows, int L, int T, hipStream_t st) {
    begin_launch();
    unsigned grid = (unsigned)((n_rows + 3) / 4);
    const bool aligned = ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 31) == 0;
    const Tin* xi = (const Tin*)x;
    Tout* yo = (Tout*)y;
    const Divisor by_l = divisor(L);
    if (T <= 2048) {
        auto groups = [&](int rows_per_wave) { return (unsigned)((n_rows + 4 * rows_per_wave - 1) / (4 * rows_per_wave)); };
        auto go = [&](auto aligned_c, auto around_c) {
            constexpr bool ALIGNED = decltype(aligned_c)::value, AROUND = decltype(around_c)::value;
            // 16-bit rows of 129 to 512 slots: 16 lanes a row, one to four chunks each, so that four rows share a wavefront's instructions and lanes
            // idle for less than a chunk in 128 slots.  Against 32 or 64 lanes a row and four row groups in flight (one up to 20000 rows),
            // us, bfloat16, 32000 / 72000 / 240000 rows: 136 slots 8.1 / 13.1 / 30.2 -> 5.9 / 10.5 / 27.7, 256 8.7 / 14.2 -> 6.4 / 13.4, 301 14.1 / 22.6 /
            // 66.3 -> 8.9 / 16.4 / 49.5, 384 in two segments 16.1 / 28.5 / 85.3 -> 10.3 / 21.3 / 61.3, 448 14.1 / 23.2 / 70.5 -> 11.9 / 22.7 / 67.3.  Around
            // the caches 32 lanes are as fast up to 256 slots (256: 40.9 both) or faster (200: 35.7 against 40.5), and so are 64 where they
            // have a chunk each (512 slots, 524288 rows: 165.6 against 168.7).
            // Short rows: four lanes up to 32 slots, eight up to 64 (float32: 48) or, 16-bit types and two chunks each, 128; against 16, bfloat16, 480000 /
            // 1600000 rows, us: 21 slots 34.5 / 108 -> 11.1 / 29.2, 40 33.7 / 123 -> 17.8 / 52.9, 64 35.1 / 128 -> 20.3 / 65.9, 100 36.0 / 130 -> 29.6 / 112 (32000
            // rows, 21, 40 and 100 slots 10.8 -> 4.6, 10.5 -> 6.6, 11.8 -> 10.0); float32, 21 slots 32.3 / 101 -> 13.8 / 39.7, 40 30.7 / 111 -> 23.5 / 99.5, 64 slots
            // of 32000 rows 11.5 -> 12.3.  Matrices that the caches do not hold: 104 slots around them 43.4 / 138 -> 46.6 / 151 with two chunks,
            // 37.9 / 119 with two row groups of 16 lanes; 127 slots in two segments 229 -> 244.
            if (T <= 32) {
                softmax_rows_vec<Tin, Tout, 1, 4, 1, ALIGNED, AROUND><<<groups(16), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                return;
            }
            if (T <= (sizeof(Tin) == 4 ? 48 : 64)) {
                constexpr int RIF = sizeof(Tin) == 4 ? 1 : 2;
                softmax_rows_vec<Tin, Tout, 1, 8, RIF, ALIGNED, AROUND><<<groups(8 * RIF), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                return;
            }
            if constexpr (sizeof(Tin) == 2 && !AROUND) {
                if (T <= (n_rows * T * (int64_t)sizeof(Tin) <= kCachedBytes ? 128 : 112)) {
                    softmax_rows_vec<Tin, Tout, 2, 8, 1, ALIGNED, AROUND><<<groups(8), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                    return;
                }
            }
            if (T <= 128) {
                constexpr int RIF = sizeof(Tin) == 2 && AROUND ? 2 : 1;
                softmax_rows_vec<Tin, Tout, 1, 16, RIF, ALIGNED, AROUND><<<groups(4 * RIF), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                return;
            }
            if constexpr (sizeof(Tin) == 2) {
                if (T <= 256) {
                    if constexpr (!ALIGNED)
                        // eight rows of odd lengths share a wavefront's instructions: 262144 rows, 129 slots 37.3 -> 26.7 us over 32 lanes a row, 191
                        // 38.8 -> 32.9 (float32 is better off with those: 191 slots 99 against 79)
                        softmax_rows_vec<Tin, Tout, 4, 8, 1, ALIGNED, AROUND><<<groups(8), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                    else if constexpr (!AROUND)
                        softmax_rows_vec<Tin, Tout, 2, 16, 1, ALIGNED, AROUND><<<groups(4), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                    else
                        softmax_rows_vec<Tin, Tout, 1, 32, 4, ALIGNED, AROUND><<<groups(2 * 4), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                    return;
                }
                if constexpr (AROUND) {
                    if (T > 448 && T <= 512) {
                        softmax_rows_vec<Tin, Tout, 1, 64, 4, ALIGNED, AROUND><<<groups(4), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                        return;
                    }
                }
                if (T <= 512) {
                    if (T <= 384)
                        softmax_rows_vec<Tin, Tout, 3, 16, 1, ALIGNED, AROUND><<<groups(4), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                    else
                        softmax_rows_vec<Tin, Tout, 4, 16, 1, ALIGNED, AROUND><<<groups(4), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                    return;
                }
            } else if (T <= 512) {
                // float32: one row group a wavefront, two of up to 256 slots, and four in flight in large launches (16384 rows of 512 slots 16.6 -> 14.0
                // with one, 131072 56.1 and 103.7 against 51.1 and 99.3; 16 lanes a row 2 to 12 % slower up to 72000 rows)
                const bool few = n_rows <= 1 << 17;
                if (T <= 256 && few)
                    softmax_rows_vec<Tin, Tout, 1, 32, 1, ALIGNED, AROUND><<<groups(2), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                else if (T <= 256)
                    softmax_rows_vec<Tin, Tout, 1, 32, 4, ALIGNED, AROUND><<<groups(2 * 4), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                else if (few)
                    softmax_rows_vec<Tin, Tout, 1, 64, 1, ALIGNED, AROUND><<<groups(1), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                else
                    softmax_rows_vec<Tin, Tout, 1, 64, 4, ALIGNED, AROUND><<<groups(4), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
                return;
            }
            if (T <= 1024)
                softmax_rows_vec<Tin, Tout, 2, 64, 1, ALIGNED, AROUND><<<groups(1), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
            else
                softmax_rows_vec<Tin, Tout, 4, 64, 1, ALIGNED, AROUND><<<groups(1), 256, 0, st>>>(xi, yo, segs, n_rows, L, T, by_l);
        };
        if (!aligned || T % 8 != 0)
            go(std::false_type{}, std::false_type{});
        // (through the caches where the rows are there and where the next operator finds them there: the three operators, bfloat16 and float32,
        // d = 64 and 128, 300 to 1000 slots, up to 80 MB 0.86 to 0.97 of the time around them; 134 to 270 MB 1.00 to 1.10)
        else if (n_rows * T * (int64_t)sizeof(Tin) <= kCachedBytes)
            go(std::true_type{}, std::false_type{});
        else
            go(std::true_type{}, std::true_type{});
    } else {
        softmax_rows_any<Tin, Tout><<<grid, 256, 0, st>>>(xi, yo, segs, n_rows, L, T);
    }
    return check_launch("splat_softmax");
}

template <typename Tin>
static int dispatch_out(const void* x, void* y, const SoftmaxSegs& segs, int64_t n_rows, int L, int T, int out_dtype, hipStream_t st) {
    switch (out_dtype) {
        case SPLAT_F32: return launch_softmax<Tin, float>(x, y, segs, n_rows, L, T, st);
        case SPLAT_F16: return launch_softmax<Tin, f16>(x, y, segs, n_rows, L, T, st);
        case SPLAT_BF16: return launch_softmax<Tin, bf16>(x, y, segs, n_rows, L, T, st);
    }
    return fail(SPLAT_E_DTYPE, "splat_softmax: unknown out_dtype %d", out_dtype);
}

}  // namespace splat

using namespace splat;

extern "C" int splat_softmax(const void* x, void* y, const splat_acsr_seg* segs, int32_t n_seg, int64_t BH, int32_t L,
                             int32_t T, int32_t in_dtype, int32_t out_dtype, void* stream) {
    if (!x || !y || !segs) return fail(SPLAT_E_NULL, "splat_softmax: null pointer argument");
    if (n_seg < 1 || n_seg > SPLAT_MAX_SEGMENTS) return fail(SPLAT_E_SHAPE, "splat_softmax: n_seg must be 1..%d (got %d)", SPLAT_MAX_SEGMENTS, n_seg);
    if (BH <= 0 || L <= 0 || T <= 0) return fail(SPLAT_E_SHAPE, "splat_softmax: need BH, L, T > 0 (got %lld, %d, %d)", (long long)BH, L, T);
    if (BH * (int64_t)L > ((int64_t)1 << 33)) return fail(SPLAT_E_SHAPE, "splat_softmax: too many rows");
    SoftmaxSegs s;
    s.n = n_seg;
    for (int k = 0; k < SPLAT_MAX_SEGMENTS; ++k) {
        s.nnz[k] = nullptr;
        s.off[k] = 0;
    }
    for (int k = 0; k < n_seg; ++k) {
        if (!segs[k].nnz) return fail(SPLAT_E_NULL, "splat_softmax: segment %d has a null nnz array", k);
        if (segs[k].slot_offset < 0 || segs[k].slot_offset >= T)
            return fail(SPLAT_E_SHAPE, "splat_softmax: segment %d slot_offset %d outside [0, T=%d)", k, segs[k].slot_offset, T);
        s.nnz[k] = segs[k].nnz;
        s.off[k] = segs[k].slot_offset;
    }
    for (int k = n_seg; k < SPLAT_MAX_SEGMENTS; ++k) s.nnz[k] = segs[0].nnz;
    const int64_t n_rows = BH * L;
    hipStream_t st = (hipStream_t)stream;
    switch (in_dtype) {
        case SPLAT_F32: return dispatch_out<float>(x, y, s, n_rows, L, T, out_dtype, st);
        case SPLAT_F16: return dispatch_out<f16>(x, y, s, n_rows, L, T, out_dtype, st);
        case SPLAT_BF16: return dispatch_out<bf16>(x, y, s, n_rows, L, T, out_dtype, st);
    }
    return fail(SPLAT_E_DTYPE, "splat_softmax: unknown in_dtype %d", in_dtype);
}

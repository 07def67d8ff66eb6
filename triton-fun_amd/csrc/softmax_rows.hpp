// Row softmax over the live slots of compressed score rows, of one wavefront (softmax.hip, and the ends of the SDDMM kernels' workgroups, which
// take their own rows).
#pragma once
#include "splat_common.hpp"

namespace splat {

struct SoftmaxSegs {
    const float* nnz[SPLAT_MAX_SEGMENTS];
    int off[SPLAT_MAX_SEGMENTS];
    int n;  // nnz[k] for k >= n repeats the first one, so that a row's counts are requested without a branch between them
};

struct LiveRanges {
    int lo[SPLAT_MAX_SEGMENTS], hi[SPLAT_MAX_SEGMENTS];
    int n;
    float cnt[SPLAT_MAX_SEGMENTS];
    __device__ __forceinline__ void request(const SoftmaxSegs& s, int row) {
        cnt[0] = s.nnz[0][row];
        if (s.n > 1) {  // uniform
#pragma unroll
            for (int k = 1; k < SPLAT_MAX_SEGMENTS; ++k) cnt[k] = s.nnz[k][row];
        }
    }
    __device__ __forceinline__ void load(const SoftmaxSegs& s, int row, int T) {
        request(s, row);
        set(s, T);
    }
    __device__ __forceinline__ void set(const SoftmaxSegs& s, int T) {
        n = s.n;
#pragma unroll
        for (int k = 0; k < SPLAT_MAX_SEGMENTS; ++k) {
            lo[k] = hi[k] = 0;
            if (k < s.n) {
                lo[k] = s.off[k];
                hi[k] = min(T, s.off[k] + (int)cnt[k]);
            }
        }
    }
    __device__ __forceinline__ bool live(int slot) const {
        bool v = false;
#pragma unroll
        for (int k = 0; k < SPLAT_MAX_SEGMENTS; ++k) v |= (k < n) && slot >= lo[k] && slot < hi[k];
        return v;
    }
    // 8-bit liveness of slots [s0, s0+8)
    __device__ __forceinline__ uint32_t live8(int s0) const {
        uint32_t m = 0;
#pragma unroll
        for (int k = 0; k < SPLAT_MAX_SEGMENTS; ++k) {
            if (k < n) {
                int a = max(lo[k], s0) - s0, b = min(hi[k], s0 + 8) - s0;
                if (b > a) m |= ((1u << b) - 1u) & ~((1u << a) - 1u);
            }
        }
        return m;
    }
};

template <typename T>
struct Vec8 {
    typedef T type __attribute__((ext_vector_type(8)));
};

// Bytes of a compressed matrix that the next kernel still finds in the last-level cache (256 MB, with its operands and results).
constexpr int64_t kCachedBytes = (int64_t)80 << 20;

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegBig = -1.0e30f;

// s plus the values of a chunk from slot `again` on (CUT; else all of them), one after the other.  FRESH: s is nothing yet.
template <bool CUT, bool FRESH>
__device__ __forceinline__ float add_chunk(float s, const float (&v)[8], int again) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float x = !CUT || e >= again ? v[e] : 0.f;
        s = FRESH && e == 0 ? x : s + x;
    }
    return s;
}

// LPR lanes share one row (64 / LPR rows per wavefront): rows shorter than 512 slots still fill every lane.  A wavefront
// takes RIF such row groups at once and requests all of their chunks before it looks at any (bytes in flight per
// wavefront are what a streaming kernel lives on).
// ALIGNED: T is a multiple of 8 and every chunk of 8 slots starts on a 16-byte boundary.  Otherwise a row's chunks start where it does, and the
// last one ends where the row ends: it repeats slots of the chunk before it, which count once and may be stored twice, by lanes of one
// wavefront and with one value.  No row's lanes touch another's slots.
// A row of up to 512 slots is added in one order, whatever the split: each chunk from its first slot on, then the sums of the chunks 32 apart,
// 16 apart and so on, of which a lane has some and its neighbours the others.  So its bits depend neither on how many rows a call has, on
// where they start, nor on which kernel takes them.  (Longer rows, which have one split each, add a lane's chunks one after the other.)
// AROUND: loads and stores go around the cache.  row_at(i, row, in_head): the row that this lane's part of group i takes, among all rows and
// among its head's, and whether it is to be stored; a surplus lane shadows some other row.
template <typename Tin, typename Tout, int NCH, int LPR, int RIF, bool ALIGNED, bool AROUND, typename RowAt>
__device__ __forceinline__ void softmax_rows(const Tin* __restrict__ x, Tout* __restrict__ y, const SoftmaxSegs& segs, int T, RowAt row_at) {
    typedef typename Vec8<Tin>::type vin;
    typedef typename Vec8<Tout>::type vout;
    const int lane = threadIdx.x & (LPR - 1);
    const int nchunk = (T + 7) >> 3;  // chunks that cover a row

    // The loads do not wait for the rows' live counts: a chunk inside the row is fetched whole and the dead slots in it are
    // discarded afterwards.  All of them, and the counts, are requested before anything is waited for: with a test of the segment's index
    // before each count, a wavefront waited for memory up to three times (float16, 32 heads of 4096 rows: 256 slots 29.6 -> 27.3 us,
    // 128 slots 16.4 -> 15.2; 64 heads of 8192 rows, 512 slots: 175 -> 172).
    int at[NCH], again[NCH];  // first slot of the lane's chunk; how many of its slots the chunk before it has
    bool mine[NCH];
    const int cut = !ALIGNED && T % 8 != 0 ? (nchunk - 1) / LPR : -1;  // which chunk of a lane can be a row's last one
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int ch = lane + LPR * c;
        mine[c] = ch < nchunk;
        at[c] = ALIGNED ? ch << 3 : max(min(ch << 3, T - 8), 0);
        again[c] = ALIGNED ? 0 : (ch << 3) - at[c];
    }
    vin raw[RIF][NCH];
    bool row_ok[RIF];
    int64_t row[RIF];
    int in_head[RIF];
#pragma unroll
    for (int i = 0; i < RIF; ++i) {
        row_ok[i] = row_at(i, row[i], in_head[i]);
        const Tin* xr = x + row[i] * (int64_t)T;
        if constexpr (ALIGNED) {
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                if (mine[c]) {
                    if constexpr (AROUND)
                        raw[i][c] = __builtin_nontemporal_load(reinterpret_cast<const vin*>(xr + at[c]));
                    else
                        raw[i][c] = *reinterpret_cast<const vin*>(xr + at[c]);
                }
            }
        } else if (T >= 8) {
            // through the cache: neighbouring rows share the lines at their ends.  Every lane loads, with no branch between the requests
#pragma unroll
            for (int c = 0; c < NCH; ++c) __builtin_memcpy(&raw[i][c], xr + at[c], sizeof(vin));
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) raw[i][0][e] = xr[min(e, T - 1)];
#pragma unroll
            for (int c = 1; c < NCH; ++c) raw[i][c] = raw[i][0];
        }
    }
    LiveRanges lr[RIF];
#pragma unroll
    for (int i = 0; i < RIF; ++i) lr[i].request(segs, in_head[i]);
#pragma unroll
    for (int i = 0; i < RIF; ++i) {
        lr[i].set(segs, T);
        Tout* yr = y + row[i] * (int64_t)T;
        float v[NCH][8];
        uint32_t live[NCH];
        float mx = kNegBig;
        bool whole = true;  // every chunk of this lane is live in all 8 slots
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            live[c] = mine[c] ? lr[i].live8(at[c]) : 0u;
            whole = whole && live[c] == 0xffu;
        }
        // the common case, decided for the whole wavefront: no dead slot anywhere in its rows, so no per-slot selects
        const bool all_whole = !__any(!whole);
        constexpr int NP = LPR == 64 ? 1 : NCH;
        float part[NP];
#pragma unroll
        for (int c = 0; c < NP; ++c) part[c] = 0.f;
        auto add = [&](int c) {  // (with a chunk's sum of its own, nothing is added to zero)
            float& s = part[c % NP];
            if (!ALIGNED && c == cut) {
#if defined(__HIP_DEVICE_COMPILE__)
                // (compared here: answers found beforehand take two scalar registers a slot until then)
                if constexpr (LPR == 16) asm("" : "+v"(again[c]));
#endif
                s = NP > 1 || c == 0 ? add_chunk<true, true>(s, v[c], again[c]) : add_chunk<true, false>(s, v[c], again[c]);
            } else {
                s = NP > 1 || c == 0 ? add_chunk<false, true>(s, v[c], again[c]) : add_chunk<false, false>(s, v[c], again[c]);
            }
        };
        if (all_whole) {
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                const vin t = raw[i][c];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    v[c][e] = (float)t[e];
                    mx = fmaxf(mx, v[c][e]);
                }
            }
            mx = wave_max<LPR>(mx);
            const float mb = mx * kLog2e;
#pragma unroll
            for (int c = 0; c < NCH; ++c)
#pragma unroll
                for (int e = 0; e < 8; ++e) v[c][e] = fast_exp2(fmaf(v[c][e], kLog2e, -mb));
#pragma unroll
            for (int c = 0; c < NCH; ++c) add(c);
        } else {
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                if (live[c]) {
                    const vin t = raw[i][c];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        v[c][e] = ((live[c] >> e) & 1u) ? (float)t[e] : kNegBig;
                        mx = fmaxf(mx, v[c][e]);
                    }
                }
            }
            mx = wave_max<LPR>(mx);
            const float mb = mx * kLog2e;
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                if (live[c]) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        // dead slots hold -1e30 and underflow to exactly 0 against any real maximum; a row without live
                        // slots stores nothing, so what its lanes compute does not matter
                        v[c][e] = fast_exp2(fmaf(v[c][e], kLog2e, -mb));
                    }
                    add(c);
                }
            }
        }
        float sum = part[0];
        if constexpr (NP > 2) sum += part[2];
        if constexpr (NP > 3)
            sum += part[1] + part[3];
        else if constexpr (NP > 1)
            sum += part[1];
        sum = wave_sum<LPR>(sum);
        const float inv = sum > 0.f ? 1.0f / sum : 0.f;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            if (live[c] && row_ok[i]) {
                if (live[c] == 0xffu) {
                    vout o;
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = rounded<Tout>(v[c][e] * inv);
                    if constexpr (!ALIGNED)
                        __builtin_memcpy(yr + at[c], &o, sizeof(vout));
                    else if constexpr (AROUND)
                        __builtin_nontemporal_store(o, reinterpret_cast<vout*>(yr + at[c]));
                    else
                        *reinterpret_cast<vout*>(yr + at[c]) = o;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if ((live[c] >> e) & 1u) yr[at[c] + e] = rounded<Tout>(v[c][e] * inv);
                }
            }
        }
    }
}

}  // namespace splat

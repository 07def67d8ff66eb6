// Shared device/host helpers for the gfx950 SPLAT kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <initializer_list>
#include <type_traits>

#include "../../include/splat_hip.h"

namespace splat {

using bf16 = __bf16;
using f16 = _Float16;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef f16 f16x8 __attribute__((ext_vector_type(8)));
typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef f16 f16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// ---- host side error plumbing (defined in api_common.cpp) ---------------------------------
void set_error(const char* fmt, ...);
int fail(int code, const char* fmt, ...);
void begin_launch();  // first statement of every function that launches and then calls check_launch
int check_launch(const char* what);

// Raise a kernel's dynamic LDS limit once per device (the attribute belongs to the device's copy of the kernel, so a
// process that uses several GPUs needs it on each): `done` is a bit mask over device ordinals, one per kernel.
int reserve_dynamic_lds(uint64_t* done, const void* kernel, size_t bytes, const char* who);

// The bytes from the first element of a strided operand to its last one.
struct Extent {
    uintptr_t first, end;
    bool meets(const Extent& o) const { return first < o.end && o.first < end; }
};
struct Dim {
    int64_t size, stride;
};
inline Extent extent_of(const void* base, int element_bytes, std::initializer_list<Dim> dims) {
    Extent e{reinterpret_cast<uintptr_t>(base), reinterpret_cast<uintptr_t>(base) + element_bytes};
    for (const Dim& d : dims) {
        const int64_t reach = (d.size - 1) * d.stride * element_bytes;
        (reach < 0 ? e.first : e.end) += reach;
    }
    return e;
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <int N, int I = 0, typename F>
__host__ __device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

template <typename T>
struct ElemTraits;
template <>
struct ElemTraits<float> {
    static constexpr int kDtype = SPLAT_F32;
};
template <>
struct ElemTraits<f16> {
    static constexpr int kDtype = SPLAT_F16;
};
template <>
struct ElemTraits<bf16> {
    static constexpr int kDtype = SPLAT_BF16;
};

// An MFMA operand fragment: what one lane feeds into one 32x32 x (16 contraction values) step.
// Lane (i = lane%32, g = lane/32) holds contraction slots 8g..8g+7 of row/column i.
template <typename T>
struct Frag {
    typedef T vec __attribute__((ext_vector_type(8)));
    vec v;
};

// acc[32x32] += A[32x16] * B[16x32]; A fragment rows = output rows, B fragment rows = output cols.
// Output layout: lane (n = lane%32, g = lane/32), register j holds row 8*(j/4) + 4*g + j%4, col n.
__device__ __forceinline__ void mma32(f32x16& acc, const Frag<bf16>& a, const Frag<bf16>& b) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, acc, 0, 0, 0);
}
__device__ __forceinline__ void mma32(f32x16& acc, const Frag<f16>& a, const Frag<f16>& b) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.v, b.v, acc, 0, 0, 0);
}
__device__ __forceinline__ void mma32(f32x16& acc, const Frag<float>& a, const Frag<float>& b) {
#pragma unroll
    for (int j = 0; j < 8; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[j], b.v[j], acc, 0, 0, 0);
}

// acc[16x16] += A[16x32] * B[32x16].  Lane (i = lane%16, g = lane/16) holds contraction slots 8g..8g+7 of row i (A) or
// column i (B); of the output, lane (n = lane%16, g = lane/16) holds rows 4g..4g+3 of column n.
typedef float f32x4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void mma16(f32x4v& acc, const Frag<bf16>& a, const Frag<bf16>& b) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc, 0, 0, 0);
}
__device__ __forceinline__ void mma16(f32x4v& acc, const Frag<f16>& a, const Frag<f16>& b) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.v, b.v, acc, 0, 0, 0);
}

// Row (within a 32-row tile) held by accumulator register j of lane group g.
__device__ __forceinline__ constexpr int acc_row(int j, int g) { return 8 * (j >> 2) + 4 * g + (j & 3); }

// x, which is the result of a product, as T: rounded to float32 first.  Left to itself the compiler multiplies and rounds to float16 in one instruction
// in some places and not in others (v_fma_mixlo_f16), and the same value has different bits in two kernels.  For the kernels whose results have to meet: the
// 16-bit sampled products, the softmax of rows of up to 2048 slots, the three operators in one.  (The second rounding adds 2^-24 of a value.  Errors of scores and
// probabilities against float64, float16, 40 to 400 slots, d = 64 and 128, 8 and 32 heads of 2048 rows: the same seven digits with and without, 2.08e-4 and 2.0e-4 to
// 2.07e-4; times of the two operators by themselves 0.97 to 1.02, but for the softmax of 64 slots in 8 heads, 3.55 -> 3.70 us.)
template <typename T>
__device__ __forceinline__ T rounded(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (std::is_same_v<T, f16>) asm("" : "+v"(x));
#endif
    return (T)x;
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Store a float as element `idx` of a buffer whose element type is chosen at run time.
__device__ __forceinline__ void store_as(void* base, int64_t idx, float x, int dtype) {
    if (dtype == SPLAT_BF16)
        ((bf16*)base)[idx] = (bf16)x;
    else if (dtype == SPLAT_F16)
        ((f16*)base)[idx] = (f16)x;
    else
        ((float*)base)[idx] = x;
}

// f(v of this lane, v of lane ^ O) for a commutative f, O a power of two, by the vector unit's own exchanges.  Through
// __shfl_xor, which is a permute through LDS, every step of a reduction waits some 130 cycles for the one before it.
// Same pairs, same bits.  Where a kernel has other work to hide the wait behind, it gives no more than two runs differ by (fused forward,
// 64 heads of 4096, d = 64, window 256, 44.9 -> 44.6 us).
// N: the lanes 2 * O apart hold the same already, which an exchange of 4 lanes in groups of 16 or of 2 * O may rely on.
template <int O, int N, typename V, typename F>
__device__ __forceinline__ V with_lane_xor(V v, F f) {
    static_assert(sizeof(V) == 4, "");
    const int x = __builtin_bit_cast(int, v);
    int y;
    if constexpr (O == 32 || O == 16) {
        const auto a = O == 32 ? __builtin_amdgcn_permlane32_swap(x, x, false, false) : __builtin_amdgcn_permlane16_swap(x, x, false, false);
        const int a0 = a[0], a1 = a[1];
        return f(__builtin_bit_cast(V, a0), __builtin_bit_cast(V, a1));
    } else if constexpr (O == 8) {
        y = __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, true);  // a rotation by 8 of 16 lanes
    } else if constexpr (O == 4 && N >= 16) {
        y = __builtin_amdgcn_update_dpp(0, x, 0x124, 0xf, 0xf, true);  // a rotation by 4: lanes 8 apart are alike
    } else if constexpr (O == 4) {
        y = __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, true);  // 8 lanes mirrored (lane ^ 7), then 4 (lane ^ 3)
        y = __builtin_amdgcn_update_dpp(0, y, 0x1b, 0xf, 0xf, true);
    } else if constexpr (O == 2) {
        y = __builtin_amdgcn_update_dpp(0, x, 0x4e, 0xf, 0xf, true);
    } else {
        y = __builtin_amdgcn_update_dpp(0, x, 0xb1, 0xf, 0xf, true);
    }
    return f(v, __builtin_bit_cast(V, y));
}

// f over each group of N consecutive lanes, N a power of two; every lane gets its group's result.  Lanes N/2 apart are
// paired first, then N/4, and so on.  All 64 lanes have to be active.
template <int N, typename V, typename F>
__device__ __forceinline__ V over_lanes(V v, F f) {
    if constexpr (N >= 64) v = with_lane_xor<32, N>(v, f);
    if constexpr (N >= 32) v = with_lane_xor<16, N>(v, f);
    if constexpr (N >= 16) v = with_lane_xor<8, N>(v, f);
    if constexpr (N >= 8) v = with_lane_xor<4, N>(v, f);
    if constexpr (N >= 4) v = with_lane_xor<2, N>(v, f);
    if constexpr (N >= 2) v = with_lane_xor<1, N>(v, f);
    return v;
}
template <int N = 64>
__device__ __forceinline__ float wave_max(float v) {
    return over_lanes<N>(v, [](float a, float b) { return fmaxf(a, b); });
}
template <int N = 64>
__device__ __forceinline__ float wave_sum(float v) {
    return over_lanes<N>(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ int wave_min_i(int v) {
    return over_lanes<64>(v, [](int a, int b) { return min(a, b); });
}
__device__ __forceinline__ int wave_max_i(int v) {
    return over_lanes<64>(v, [](int a, int b) { return max(a, b); });
}

// Integer view of one row's affine map, recovered from the float32 metadata.
//   a   = first live dense column, lin = column step, cnt = live slots.
// sTod_trans stores a/lin rounded to float32, so a = rint(lin * trans) is exact for a < 2^23.
struct RowMap {
    int a, lin, cnt;
};
__device__ __forceinline__ RowMap load_row_map(const float* sTod_lin, const float* sTod_trans, const float* nnz,
                                               const int32_t* first_col, int r) {
    RowMap m;
    m.cnt = (int)nnz[r];
    float lin = sTod_lin[r];
    m.lin = max((int)lin, 1);
    m.a = (int)rintf(lin * sTod_trans[r]);
    if (first_col != nullptr && m.cnt == 1) m.a = first_col[r];
    return m;
}

// Division by a number that the host knows: n / d is the high part of one product, for every 0 <= n < 2^31 (Granlund and Montgomery,
// "Division by Invariant Integers using Multiplication", 1994).  A kernel's own division by one of its arguments takes some forty
// instructions, two of them at the beginning of every workgroup; with load_args below, 16-bit forward of 16 heads of 576 rows, d = 128, window 64
// 6.85 -> 6.40 us, 12 heads of 1037 12.05 -> 11.57, 64 of 4096 at d = 64 44.2 -> 42.9; one float32 head of 512 rows 8.74 -> 8.34; the three
// operators, 128 heads of 958 rows of 39 slots, 43.6 -> 41.3 (whose softmax divides once a row in every lane).
struct Divisor {
    uint32_t m;
    int32_t shift;
};
inline Divisor divisor(int64_t d) {
    int l = 0;
    while (((int64_t)1 << l) < d) ++l;
    return Divisor{(uint32_t)((((uint64_t)1 << (31 + l)) + d - 1) / d), 31 + l};
}
__device__ __forceinline__ int quotient(int n, Divisor d) { return (int)(((uint64_t)(uint32_t)n * d.m) >> d.shift); }

// Kernel arguments that are wanted now, in one round of loads.  Left to itself the compiler loads them where they are used, and a
// workgroup that has a CU to itself waits some 400 cycles for each of four or five rounds before its first operand is requested.
template <typename A>
__device__ __forceinline__ void load_arg(A a) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" ::"s"(a));
#endif
}
template <typename... A>
__device__ __forceinline__ void load_args(A... a) {
    (load_arg(a), ...);
}

// Workgroup barrier that hands LDS contents over and nothing else: it waits for this wavefront's LDS traffic, not for
// its global loads and stores.  __syncthreads() waits for both counters, which serialises a kernel whose loads of the
// next tile or stores of the previous one are meant to stay in flight across the barrier.  (The empty statements keep
// the compiler from moving memory accesses across the barrier.)
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Map a launch-order workgroup id onto a logical id so that logically consecutive ids run on the
// same XCD (hardware deals consecutive workgroup ids round-robin over the 8 XCDs, each with its own
// L2).  The grid is `total` rounded up to a multiple of 8; ids >= total are idle.
__device__ __forceinline__ int xcd_remap(int wg, int total) {
    const int chunk = (total + 7) >> 3;
    return (wg & 7) * chunk + (wg >> 3);
}

}  // namespace splat

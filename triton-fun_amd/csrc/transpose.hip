// K^T [B, H, d, L] with the keys contiguous (the reference's layout, r_sddmm.py:230-231) -> K [B, H, L, d] with rows
// contiguous, which is what the kernels read without waste when rows step over columns (a dilated window's every second
// key, a strided far field's every 128th): there they fetch only the keys a tile needs, while K^T can only be read in
// dense runs of keys.  Pure streaming kernels: every byte read once and written once, in whole 16-byte pieces on both
// sides (source rows at any alignment); the turn goes through an LDS tile.
#include "splat_common.hpp"
#include "tile_copy.hpp"

namespace splat {

struct TransposeParams {
    const void* src;
    void* dst;
    int64_t s_sb, s_sh, s_sd;  // element strides of the source's batch, head and d index; keys have stride 1
    int B, H, L, d;
    int total;                      // workgroups, tiles of d first, then tiles of keys: neighbours on one XCD share the lines that
    Divisor by_dt, by_kt, by_h;     // rows at odd addresses straddle
};

constexpr int kTurnD = 64, kTurnKeys = 128;  // values of d and keys a workgroup

// 16-bit types.  One workgroup: 128 keys x 64 values of d of one (batch, head), four rows of eight keys a thread, which it turns to four
// values of each key on their way into LDS; pieces of a key's row there are permuted by its place among the pieces of eight, so that neither the
// 8-byte writes (of keys eight apart) nor the 16-byte reads (of whole rows) meet in a bank.  Eight lanes store a key's whole 128 bytes.
// Bound: HBM and, up to some hundred workgroups, one round of latencies.  Against a tile of 64 x 64 written in 4-byte pieces and read back two bytes
// at a time, bfloat16, us (TB/s): 16 heads of 9134 keys, d = 128 19.6 -> 11.6 (3.8 -> 6.5); 64 of 4099, d = 64 17.4 -> 10.8, of 4096 13.6 ->
// 10.8; 32 of 8191, d = 80 21.5 -> 14.3; 224 of 2849, d = 128 72.8 -> 59.7; 12 of 1037, d = 128 4.0 -> 3.4; 4 of 999, d = 64 3.1 both.  Without the
// order by XCDs the first took 14.9.  Transposing reads of a tile that lies as it came (16 keys of 16 bytes an instruction) leave eight lanes a
// line to eight stores: 20.8.
__global__ __launch_bounds__(256) void transpose_keys16_kernel(const TransposeParams p) {
    constexpr int TK = kTurnKeys, PPR = TK / 8, ROWB = 2 * kTurnD;
    __shared__ __attribute__((aligned(1024))) char tile[TK * ROWB];
    const int tid = threadIdx.x;
    load_args(p.total, p.by_dt.m, p.by_dt.shift, p.by_kt.m, p.by_kt.shift, p.by_h.m, p.by_h.shift, p.src, p.dst, p.s_sb, p.s_sh, p.s_sd, p.H, p.L, p.d);
    const int logical = xcd_remap(blockIdx.x, p.total);
    if (logical >= p.total) return;
    const int L = p.L, d = p.d;
    const int n_dt = (d + kTurnD - 1) / kTurnD, n_kt = (L + TK - 1) / TK;
    const int block = quotient(logical, p.by_dt), bh = quotient(block, p.by_kt), b = quotient(bh, p.by_h), h = bh - b * p.H;
    const int d0 = (logical - block * n_dt) * kTurnD, k0 = (block - bh * n_kt) * TK;
    const uint16_t* const src = (const uint16_t*)p.src + b * p.s_sb + h * p.s_sh;

    // (pieces are requested whole and without a branch: rows and keys that do not exist are others here and are not stored, and the piece
    // that the end of a row cuts is the row's last whole one, moved down below)
    const int pc = tid % PPR, quad = tid / PPR, kk0 = k0 + 8 * pc;
    u32x4 in[4];
    auto row_of = [&](int i) { return src + (int64_t)min(d0 + 4 * quad + i, d - 1) * p.s_sd; };
    if (L >= 8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) __builtin_memcpy(&in[i], row_of(i) + min(kk0, L - 8), 16);
        if (const int over = kk0 + 8 - L; over > 0 && over < 8) {
#pragma unroll
            for (int i = 0; i < 4; ++i) in[i] = __builtin_bit_cast(u32x4, __builtin_bit_cast(unsigned __int128, in[i]) >> (16 * over));
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint16_t v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = row_of(i)[min(kk0 + e, L - 1)];
            __builtin_memcpy(&in[i], v, 16);
        }
    }
    const uint32_t to = lds_address(tile) + 8 * pc * ROWB + (((quad >> 1) ^ (pc & 7)) << 4) + ((quad & 1) << 3);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const uint32_t halves = e & 1 ? 0x07060302u : 0x05040100u;  // the upper or the lower ones of two registers
        const u32x2 x = {__builtin_amdgcn_perm(in[1][e >> 1], in[0][e >> 1], halves), __builtin_amdgcn_perm(in[3][e >> 1], in[2][e >> 1], halves)};
        *reinterpret_cast<__attribute__((address_space(3))) u32x2*>((uintptr_t)(to + e * ROWB)) = x;
    }
    __syncthreads();

    uint16_t* const dst = (uint16_t*)p.dst + (int64_t)bh * L * d;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int key = tid / 8 + TK / 4 * i, c = tid % 8;
        const u32x4 x = lds_load128(lds_address(tile) + key * ROWB + ((c ^ (key >> 3 & 7)) << 4));
        const int kk = k0 + key, dd = d0 + 8 * c;
        if (kk >= L || dd >= d) continue;
        uint16_t* const out = dst + (int64_t)kk * d + dd;
        if (d % 8 == 0) {
            *reinterpret_cast<u32x4*>(out) = x;
        } else {
            uint16_t v[8];
            __builtin_memcpy(v, &x, 16);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (dd + e < d) out[e] = v[e];
        }
    }
}

// float32.  One workgroup: 64 keys x 64 values of d of one (batch, head).  LDS tile [d index][key], written in 4-byte pieces, read back key by key.
__global__ __launch_bounds__(256) void transpose_keys32_kernel(const TransposeParams p) {
    typedef float T;
    constexpr int ES = sizeof(T), EPC = 16 / ES;  // elements per 16-byte piece
    constexpr int TK = 64, TD = 64;
    constexpr int PITCH = TK * ES + 4;            // odd number of banks between rows: the column reads spread out
    __shared__ __attribute__((aligned(16))) char tile[TD * PITCH];
    const int tid = threadIdx.x;
    const int n_kt = (p.L + TK - 1) / TK, n_dt = (p.d + TD - 1) / TD;
    int blk = blockIdx.x;
    const int kt = blk % n_kt;
    blk /= n_kt;
    const int dt = blk % n_dt;
    const int bh = blk / n_dt;
    const int b = bh / p.H, h = bh % p.H;
    const int k0 = kt * TK, d0 = dt * TD;
    const T* src = (const T*)p.src + (int64_t)b * p.s_sb + (int64_t)h * p.s_sh;
    T* dst = (T*)p.dst + (int64_t)bh * p.L * p.d;

    // in: rows = d index, 64 keys each
    constexpr int PPR = TK / EPC;  // pieces per row
    constexpr int NI = TD * PPR / 256;
    u32x4 in[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int idx = tid + 256 * i, row = idx / PPR, pc = idx % PPR;
        const int dd = d0 + row, kk = k0 + pc * EPC;
        if (dd < p.d && kk + EPC <= p.L) {
            __builtin_memcpy(&in[i], src + (int64_t)dd * p.s_sd + kk, 16);
        } else {
            T v[EPC];
#pragma unroll
            for (int e = 0; e < EPC; ++e) v[e] = (dd < p.d && kk + e < p.L) ? src[(int64_t)dd * p.s_sd + kk + e] : (T)0.f;
            __builtin_memcpy(&in[i], v, 16);
        }
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int idx = tid + 256 * i, row = idx / PPR, pc = idx % PPR;
#pragma unroll
        for (int w = 0; w < 4; ++w) *reinterpret_cast<uint32_t*>(tile + row * PITCH + pc * 16 + 4 * w) = in[i][w];
    }
    __syncthreads();
    // out: rows = keys, 64 values of d each (one 16-byte piece per thread and pass)
    constexpr int PPK = TD / EPC;  // pieces per key
    const bool dvec = (p.d % EPC) == 0;  // every destination piece starts on a 16-byte boundary
#pragma unroll
    for (int i = 0; i < TK * PPK / 256; ++i) {
        const int idx = tid + 256 * i, key = idx / PPK, pc = idx % PPK;
        const int kk = k0 + key, dd = d0 + pc * EPC;
        if (kk >= p.L || dd >= p.d) continue;
        T v[EPC];
#pragma unroll
        for (int e = 0; e < EPC; ++e) v[e] = *reinterpret_cast<const T*>(tile + (pc * EPC + e) * PITCH + key * ES);
        T* out = dst + (int64_t)kk * p.d + dd;
        if (dvec && dd + EPC <= p.d) {
            __builtin_memcpy(__builtin_assume_aligned(out, 16), v, 16);
        } else {
#pragma unroll
            for (int e = 0; e < EPC; ++e)
                if (dd + e < p.d) out[e] = v[e];
        }
    }
}

}  // namespace splat

using namespace splat;

extern "C" int splat_transpose_keys(const void* kT, int64_t kT_sb, int64_t kT_sh, int64_t kT_sd, void* k_rows, int32_t B,
                                    int32_t H, int32_t L, int32_t d, int32_t dtype, void* stream) {
    begin_launch();
    if (!kT || !k_rows) return fail(SPLAT_E_NULL, "splat_transpose_keys: null pointer argument");
    if (B <= 0 || H <= 0 || L <= 0 || d <= 0) return fail(SPLAT_E_SHAPE, "splat_transpose_keys: need B, H, L, d > 0 (got %d, %d, %d, %d)", B, H, L, d);
    if (kT_sd < L) return fail(SPLAT_E_SHAPE, "splat_transpose_keys: the stride of the d index (%lld) is shorter than a row of %d keys", (long long)kT_sd, L);
    const int es = dtype == SPLAT_F32 ? 4 : 2;
    if (dtype != SPLAT_F32 && dtype != SPLAT_F16 && dtype != SPLAT_BF16) return fail(SPLAT_E_DTYPE, "splat_transpose_keys: unknown dtype %d", dtype);
    if ((reinterpret_cast<uintptr_t>(k_rows) & 15) != 0) return fail(SPLAT_E_ALIGN, "splat_transpose_keys: k_rows must be 16-byte aligned");
    if ((reinterpret_cast<uintptr_t>(kT) & (es - 1)) != 0) return fail(SPLAT_E_ALIGN, "splat_transpose_keys: kT is not aligned to its element size");
    const int64_t blocks = (int64_t)B * H * ((L + 63) / 64) * ((d + kTurnD - 1) / kTurnD);
    if (blocks > 0x7ffffff0) return fail(SPLAT_E_SHAPE, "splat_transpose_keys: problem too large for one launch");
    TransposeParams p;
    p.src = kT, p.dst = k_rows;
    p.s_sb = kT_sb, p.s_sh = kT_sh, p.s_sd = kT_sd;
    p.B = B, p.H = H, p.L = L, p.d = d;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == SPLAT_F32) {
        transpose_keys32_kernel<<<(int)blocks, 256, 0, st>>>(p);
    } else {  // the two 16-bit types move alike
        const int n_kt = (L + kTurnKeys - 1) / kTurnKeys, n_dt = (d + kTurnD - 1) / kTurnD;
        p.total = B * H * n_kt * n_dt;
        p.by_dt = divisor(n_dt), p.by_kt = divisor(n_kt), p.by_h = divisor(H);
        transpose_keys16_kernel<<<(p.total + 7) / 8 * 8, 256, 0, st>>>(p);
    }
    return check_launch("splat_transpose_keys");
}

// gemm_rows.hip — quantized weights times a batch of FP32 token rows on
// gfx950 MFMA, for any row count, any token count and row lengths the tiled
// prompt GEMMs do not take.
//
//   y[t][m] = sum_k W[m][k] x[t][k]       W: OIL8 (src/kernel_oil8.cpp:14-27), OIL4 with codebooks per cb_block
//   columns or one per tensor (src/kernel_oil4.cpp:31-54), or ternary (src/kernel_i2s.cpp:42-65, o[m][t])
//
// Arithmetic (as the batched GEMVs and the prompt GEMMs): each token row is
// scaled by a power of two and split into FP16 hi + lo (rows_split_k, once per
// call); OIL4 and ternary weights are exact in FP16 (two products per weight
// and token), OIL8 codebook entries are split the same way (three products;
// lo x lo lies below FP32's rounding).  lo parts are held times 2^11, so that a
// value keeps its 22 bits down to 2^-28 of its row's (its codebook's) maximum.
// Products are exact in FP32, sums FP32
// on v_mfma_f32_16x16x32_f16, the hi x hi products and the rest in accumulators
// of their own.  OIL8 and OIL4 add the hi x hi products of a step of 128 columns
// up from zero and then to the slice's sum: one accumulator per slice rounds at
// its full size some K / 10 times, and at 4080 .. 13696 columns in one slice was
// 4.1e-7 .. 7.4e-7 of the norm off (64-bit sums), where the FP32 FMAs of the
// kernels that walk the tokens are 1.1e-7 .. 2.7e-7 and this 1.4e-7 .. 2.1e-7
// (OIL8 2 % slower, OIL4 the same time; the ternary sums were below the FP32
// kernel's without it).  The OIL8 kernel that walks the tokens in rows of up to
// 4096 columns sums 16 products per lane and is 0.96e-7 .. 1.09e-7 off.  Where it
// is the other route (fp32) FINE adds lo x lo, starts every product of 32
// columns from zero and keeps the roundings of the additions: 0.89e-7 .. 0.97e-7
// (without FINE 1.18e-7 .. 1.5e-7) on token tiles of at most 48, for 3 .. 30 % of
// the time (40 tokens x 12000 x 4080 38 -> 46 us, walking them 349 us).
// A token row that holds Inf or NaN takes FP32 FMAs over the reference's
// products instead, as do all rows of a non-finite OIL8 codebook.  Where the
// other route is FP32 products (fp32), so do single outputs: of a token row (or
// an OIL8 codebook) that spans more than 28 binades those so small that only
// values with fewer bits can have made them (its largest met weights of 0), and
// an OIL4 output that comes out NaN, where an infinite entry may have met a
// value that both parts miss.  bf16 rows are one FP16 part, as in the tiled
// prompt kernels.
//
// Tiling.  A workgroup of 4 waves takes 128 weight rows (32 per wave: two A
// tiles share every B read, which otherwise bounds the kernel: a tile-step
// reads 32 KB of B per wave from LDS) x 16 G tokens (G <= 4) over a K slice in
// steps of 128 columns.  Weights go from memory straight into A registers (two
// steps ahead), B fragments of a step through LDS (one step ahead in
// registers); two workgroups per CU cover each other's barriers.  gridDim.z > 1:
// K slices, whose sums rows_reduce_k adds in order.
//
// Bound: per workgroup ~5 us before the first step and after the last (load latency, table, output) and then, on a
// full chip, LDS for OIL8 (counters at 48 tokens: a workgroup's step keeps it busy for 2180 cycles, 256 gathers of 5.5
// and 770 for B, 0.9 of the 1.36 us that a CU takes per step) and half of the MFMA rate for the others (64 tokens: 1024
// matrix cycles per SIMD, 0.43 of 0.83 us).  Measured against the routes before it (one
// call, eager): OIL8 4000 x 4096, 40 tokens 32.9 -> 19.3 us; 2000 x 8976, 256 tokens 9.9 ms -> 52 us; OIL4 5000 x
// 9088 (codebooks per 64), 64 tokens 5.4 ms -> 36 us; ternary 4096 x 4096, 300 tokens 5.8 ms -> 36 us.  bf16 rows (one
// part and product): 100 tokens x 1200 x 4096 103 -> 18 us, 160 x 5120 x 4096 50 -> 33 us.
#include <algorithm>

#include "common.h"
#include "launch.h"
#include "oil4_common.h"

namespace mth {
namespace {

constexpr int kRmStep = 128;              // columns per step
constexpr int kRmRows = 128, kRmT = 256;  // weight rows and threads per workgroup
constexpr int kRmSlices = 16;             // most K slices (rows_reduce_k)
constexpr int kRmFineCols = 4096;         // OIL8 rows of up to so many columns: FINE where the other route is FP32

// kOil4B: OIL4 weights, bf16 token rows (one FP16 part), bf16 outputs
enum RowsFmt { kOil8, kOil4, kTern, kOil4B };
template <int FMT>
constexpr int kParts = FMT == kOil4B ? 1 : 2;  // FP16 parts of a token row

// ---- token rows -> FP16 hi / lo B fragments ------------------------------------
// Row t: shift s with max|x| 2^s in [2^14, 2^15) into rsh[t] (kRowFp32 for a row holding Inf / NaN; s + kRowWide, with
// guard, for one whose nonzero values span more than 28 binades), then 2^s x = hi + 2^-11 lo, group t / 16, part (hi,
// lo), 32-column chunk c: 1 KB of [8-column piece m][token t % 16][8].  TERN: the pieces hold the columns in the order
// of the ternary codes' planes (element e of piece m: column 16 (m / 2) + 2 (m % 2) + e / 4 + 4 (e % 4) of the chunk).
// Columns past K are zeros; rows past the batch are not written (their products only reach their own, discarded,
// outputs).  One workgroup per row, the row read once (16384 columns in registers; the rest of a longer row twice).
constexpr int kRsN = 4;
constexpr int kRowFp32 = kRowNonFinite, kRowWide = 1 << 16;
template <bool TERN, bool VEC>
__global__ __launch_bounds__(kRmT) void rows_split_k(const float* __restrict__ x, uint16_t* __restrict__ a16,
                                                     int* __restrict__ rsh, int K, int chunks, bool guard) {
    __shared__ uint32_t red[kRmT / 64], redn[kRmT / 64];
    const int tid = threadIdx.x, row = blockIdx.x;
    const float* xr = x + (int64_t)row * K;
    const int n16 = 2 * chunks;  // 16-column groups
    auto load = [&](int g, float (&v)[16]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 16 * g + 4 * i;
            if constexpr (VEC) {
                const float4 f = g < n16 && k < K ? ldf4(xr + k) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                v[4 * i] = f.x, v[4 * i + 1] = f.y, v[4 * i + 2] = f.z, v[4 * i + 3] = f.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * i + e] = g < n16 && k + e < K ? xr[k + e] : 0.0f;
            }
        }
    };
    float v[kRsN][16], u[16];
#pragma unroll
    for (int j = 0; j < kRsN; ++j) load(tid + j * kRmT, v[j]);
    uint32_t mb = 0, mn = 0;  // max |x| bits; 2^32 - the least nonzero |x| bits (0: all zeros)
    auto range = [&](const float (&f)[16]) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t ab = __float_as_uint(f[i]) & 0x7fffffffu;
            mb = max(mb, ab);
            mn = max(mn, 0u - ab);
        }
    };
#pragma unroll
    for (int j = 0; j < kRsN; ++j) range(v[j]);
    for (int g = tid + kRsN * kRmT; g < n16; g += kRmT) {
        load(g, u);
        range(u);
    }
    mb = group_reduce<64>(mb, UMaxOp{});
    mn = group_reduce<64>(mn, UMaxOp{});
    if ((tid & 63) == 0) red[tid >> 6] = mb, redn[tid >> 6] = mn;
    __syncthreads();
    mb = max(max(red[0], red[1]), max(red[2], red[3]));
    mn = 0u - max(max(redn[0], redn[1]), max(redn[2], redn[3]));
    const int sh = fp16_scale_shift(__uint_as_float(mb));
    if (tid == 0)
        rsh[row] = mb >= 0x7f800000u ? kRowFp32 : guard && (int)(mb >> 23) - (int)(mn >> 23) > 28 ? sh + kRowWide : sh;
    uint16_t* hi = a16 + (int64_t)(row >> 4) * 2 * chunks * 512 + 8 * (row & 15);
    uint16_t* lo = hi + (int64_t)chunks * 512;
    auto store = [&](int g, const float (&f)[16]) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            half8 h, l;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float xs = ldexpf(f[TERN ? 2 * p + (e >> 2) + 4 * (e & 3) : 8 * p + e], sh);
                h[e] = (_Float16)xs;
                l[e] = (_Float16)((xs - (float)h[e]) * 2048.0f);
            }
            const int64_t off = (int64_t)(g >> 1) * 512 + 128 * (2 * (g & 1) + p);
            *(half8*)(hi + off) = h;
            *(half8*)(lo + off) = l;
        }
    };
#pragma unroll
    for (int j = 0; j < kRsN; ++j)
        if (tid + j * kRmT < n16) store(tid + j * kRmT, v[j]);
    for (int g = tid + kRsN * kRmT; g < n16; g += kRmT) {
        load(g, u);
        store(g, u);
    }
}

// bf16 rows, K % 32 == 0, 16-byte aligned: one part per group (2^s x, rounded to FP16 only 2^-24 below the row's
// maximum and less); rows with an Inf or a NaN: s = 0, the value in the part.
__global__ __launch_bounds__(kRmT) void rows_half_k(const uint16_t* __restrict__ x, uint16_t* __restrict__ a16,
                                                    int* __restrict__ rsh, int K, int chunks) {
    __shared__ uint32_t red[kRmT / 64];
    const int tid = threadIdx.x, row = blockIdx.x;
    const uint16_t* xr = x + (int64_t)row * K;
    const int n8 = 4 * chunks;  // 8-column pieces, zeros past K
    auto load = [&](int c) { return 8 * c < K ? ld16(xr + 8 * c) : make_uint4(0, 0, 0, 0); };
    uint4 v[2 * kRsN];
#pragma unroll
    for (int j = 0; j < 2 * kRsN; ++j) v[j] = load(tid + j * kRmT);
    uint32_t mb = 0;
    auto most = [&](uint4 w) {
#pragma unroll
        for (int e = 0; e < 4; ++e) mb = max(mb, max(u4get(w, e) & 0x7fffu, (u4get(w, e) >> 16) & 0x7fffu));
    };
#pragma unroll
    for (int j = 0; j < 2 * kRsN; ++j) most(v[j]);
    for (int c = tid + 2 * kRsN * kRmT; c < n8; c += kRmT) most(load(c));
    mb = group_reduce<64>(mb, UMaxOp{});
    if ((tid & 63) == 0) red[tid >> 6] = mb;
    __syncthreads();
    const int sh = fp16_scale_shift(__uint_as_float(max(max(red[0], red[1]), max(red[2], red[3])) << 16));
    if (tid == 0) rsh[row] = sh;
    uint16_t* dst = a16 + (int64_t)(row >> 4) * chunks * 512 + 8 * (row & 15);
    auto store = [&](int c, uint4 w) {
        *(half8*)(dst + (int64_t)(c >> 2) * 512 + 128 * (c & 3)) = bf16x8_to_f16(w, sh);
    };
#pragma unroll
    for (int j = 0; j < 2 * kRsN; ++j)
        if (tid + j * kRmT < n8) store(tid + j * kRmT, v[j]);
    for (int c = tid + 2 * kRsN * kRmT; c < n8; c += kRmT) store(c, load(c));
}

// ---- the product ----------------------------------------------------------------
struct RowsArgs {
    const uint8_t* w;      // OIL8 indices [M][K], OIL4 nibbles [M][K / 2], ternary codes [M][K / 4]
    const void* cb;        // OIL8: 256 floats; OIL4: FP16 codebooks
    const uint16_t* a16;   // rows_split_k's fragments
    const int* rsh;
    const float* x;        // [batch][K] (FP32 rows)
    float* out;            // [batch][M] (ternary: [M][batch]; kOil4B: bf16)
    float* partial;        // [slice] of the same
    int M, K, batch, steps, cb_block;
    bool fp32;             // FP32 products for the outputs that a wide range may have left inexact and OIL4's NaN
};
// OIL8: up to three matrices over the same token rows (a decoder's Q, K and V), their row tiles one after another in
// the grid; t1: the first row tile past matrix i.  Matrix i's partial sums start at partial + p0[i].
struct RowsSegs {
    const uint8_t* w[3];
    const void* cb[3];
    float* out[3];
    int M[3], t1[3];
    int64_t p0[3];
    int n;
};

// a weight tile's registers of one step: 16 rows x 128 columns
template <int FMT>
struct RowsTile;
template <>
struct RowsTile<kOil8> {
    uint4 x, y;  // rows 0-7 / 8-15, 8 lanes of 16 bytes per row (128-byte runs); h3_pieces hands them out
};
template <>
struct RowsTile<kOil4> {
    uint4 n, c0, c1;  // the lane's row: nibbles of columns 32 q .., its block's 16 entries
};
template <>
struct RowsTile<kOil4B> : RowsTile<kOil4> {};
template <>
struct RowsTile<kTern> {
    uint2 c;  // the lane's row: codes of columns 32 q ..
};

__device__ __forceinline__ uint32_t rows_hl(float c) {
    const _Float16 h = (_Float16)c;
    const _Float16 l = (_Float16)((c - (float)h) * 2048.0f);
    return (uint32_t)__builtin_bit_cast(uint16_t, h) | ((uint32_t)__builtin_bit_cast(uint16_t, l) << 16);
}

// 8 ternary weights (planes f, f + 1 of a code dword) as FP16: code 0 -> -1, 1 -> 0, 2 and 3 -> 1.  A byte lookup
// gives the high bytes 0xBC, 0, 0x3C, 0x3C; the low bytes are 0.
__device__ __forceinline__ half8 rows_tern8(uint32_t d, int f) {
    typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
    const uint32_t h0 = __builtin_amdgcn_perm(0u, 0x3c3c00bcu, (d >> (2 * f)) & 0x03030303u);
    const uint32_t h1 = __builtin_amdgcn_perm(0u, 0x3c3c00bcu, (d >> (2 * f + 2)) & 0x03030303u);
    const u32x4v r = {__builtin_amdgcn_perm(0u, h0, 0x010c000cu), __builtin_amdgcn_perm(0u, h0, 0x030c020cu),
                      __builtin_amdgcn_perm(0u, h1, 0x010c000cu), __builtin_amdgcn_perm(0u, h1, 0x030c020cu)};
    return __builtin_bit_cast(half8, r);
}

// FP32 products over every inc-th column of [k0, k1) of one output, the reference's arithmetic in column order.
template <int FMT>
__device__ float rows_fma(const RowsArgs& p, int row, int tok, int k0, int k1, int inc = 1) {
    const float* x = p.x + (int64_t)tok * p.K;
    float s = 0.0f;
    if constexpr (FMT == kOil8) {
        const uint8_t* w = p.w + (int64_t)row * p.K;
        const float* cb = (const float*)p.cb;
        for (int k = k0; k < k1; k += inc) s = fmaf(cb[w[k]], x[k], s);
    } else if constexpr (FMT == kOil4 || FMT == kOil4B) {
        const uint8_t* w = p.w + (int64_t)row * (p.K >> 1);
        const uint16_t* cb = (const uint16_t*)p.cb;
        for (int k = k0; k < k1; k += inc) {
            const int e = (w[k >> 1] >> (4 * (k & 1))) & 15;
            const int64_t b = p.cb_block ? (int64_t)row * (p.K / p.cb_block) + k / p.cb_block : 0;
            s = fmaf(h2f(cb[b * 16 + e]), x[k], s);
        }
    } else {
        const uint8_t* w = p.w + (int64_t)row * (p.K >> 2);
        for (int k = k0; k < k1; k += inc) {
            const int c = (w[k >> 2] >> (2 * (k & 3))) & 3;
            s += c == 1 ? 0.0f : (c == 0 ? -x[k] : x[k]);
        }
    }
    return s;
}

template <int FMT, int G, bool FINE = false>
__global__ __launch_bounds__(kRmT, 2) void rows_mfma_k(RowsArgs p, RowsSegs sg) {
    constexpr int P = kParts<FMT>;
    constexpr bool O4 = FMT == kOil4 || FMT == kOil4B;
    constexpr bool STEP = FMT == kOil8 || FMT == kOil4;  // hi x hi sums of a step, added up outside
    constexpr int NB = P * G;  // 16-byte pieces of a step's B per thread (4 KB per token group and part)
    __shared__ __align__(16) uint8_t bs[P * G * 4096];
    __shared__ uint32_t tab[FMT == kOil8 ? 256 : 1];
    __shared__ float wred[kRmT / 64];
    __shared__ uint32_t wleast[kRmT / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = lane & 15, q = lane >> 4;
    int bx = blockIdx.x;
    if constexpr (FMT == kOil8) {
        if (sg.n > 1) {
            const int i = (bx >= sg.t1[0] ? 1 : 0) + (bx >= sg.t1[1] ? 1 : 0);
            bx -= i == 0 ? 0 : i == 1 ? sg.t1[0] : sg.t1[1];
            p.w = i == 0 ? sg.w[0] : i == 1 ? sg.w[1] : sg.w[2];
            p.cb = i == 0 ? sg.cb[0] : i == 1 ? sg.cb[1] : sg.cb[2];
            p.out = i == 0 ? sg.out[0] : i == 1 ? sg.out[1] : sg.out[2];
            p.M = i == 0 ? sg.M[0] : i == 1 ? sg.M[1] : sg.M[2];
            p.partial += i == 0 ? sg.p0[0] : i == 1 ? sg.p0[1] : sg.p0[2];
        }
    }
    const int row0 = bx * kRmRows + wave * 32, tok0 = blockIdx.y * 16 * G;
    const int S = gridDim.z;
    const int s0 = (int)((int64_t)blockIdx.z * p.steps / S), s1 = (int)((int64_t)(blockIdx.z + 1) * p.steps / S);
    const int M = p.M, K = p.K;

    // ---- loads of a step: every address in bounds (rows past M - 1: row M - 1; columns past the row: its last
    // 16 bytes, whose products meet zeros; steps past the slice: its last)
    RowsTile<FMT> wt[2][2];  // [step parity][tile]
    const int64_t tend = FMT == kTern ? (int64_t)M * (K >> 2) : 0;
    auto load_w = [&](int step, RowsTile<FMT> (&dst)[2]) {
        const int st = min(step, s1 - 1);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if constexpr (FMT == kOil8) {
                const int col = min(kRmStep * st + 16 * (2 * q + (j >> 3)), K - 16);
                dst[t].x = ld_stream(p.w + (int64_t)min(row0 + 16 * t + (j & 7), M - 1) * K + col);
                dst[t].y = ld_stream(p.w + (int64_t)min(row0 + 16 * t + 8 + (j & 7), M - 1) * K + col);
            } else if constexpr (O4) {
                const int64_t row = min(row0 + 16 * t + j, M - 1);
                const int col = min(kRmStep * st + 32 * q, K - 32);
                dst[t].n = ld_stream(p.w + row * (K >> 1) + (col >> 1));
                const uint16_t* cb = (const uint16_t*)p.cb;
                if (p.cb_block) cb += (row * (K / p.cb_block) + col / p.cb_block) * 16;
                dst[t].c0 = ld16(cb);
                dst[t].c1 = ld16(cb + 8);
            } else {
                const int64_t pos = (int64_t)min(row0 + 16 * t + j, M - 1) * (K >> 2) + (kRmStep / 4) * st + 8 * q;
                dst[t].c = ld_codes8(p.w, pos, tend);
            }
        }
    };
    uint4 bv[NB];
    // B: thread's pieces tid + 256 i of [group][part][4 KB of the step's 4 chunks]
    const int64_t part_bytes = (int64_t)p.steps * 4096;
    const uint8_t* a16 = (const uint8_t*)p.a16 + (int64_t)(tok0 >> 4) * P * part_bytes + 16 * tid;
    auto load_b = [&](int step) {
        const uint8_t* base = a16 + (int64_t)min(step, s1 - 1) * 4096;
#pragma unroll
        for (int i = 0; i < NB; ++i) bv[i] = ld16(base + i * part_bytes);
    };
    // the small operands first (the CU returns loads in issue order), then B and the weights
    int rs[G];  // this lane's tokens' shifts (rows past the batch: the last row's)
#pragma unroll
    for (int g = 0; g < G; ++g) rs[g] = p.rsh[min(tok0 + 16 * g + j, p.batch - 1)];
    float cbv = 0.0f;
    if constexpr (FMT == kOil8) cbv = ((const float*)p.cb)[tid];
    __builtin_amdgcn_sched_barrier(0);
    load_b(s0);
    load_w(s0, wt[0]);
    load_w(s0 + 1, wt[1]);
    __builtin_amdgcn_sched_barrier(0);

    // ---- the codebook's table, the scales, the non-finite check
    bool fin = true;
    if constexpr (FMT == kOil8) {
        fin = __builtin_isfinite(cbv);
        const float m = wave_max(fabsf(cbv));
        const uint32_t least = group_reduce<64>(0u - (__float_as_uint(cbv) & 0x7fffffffu), UMaxOp{});  // (rows_split_k)
        if (lane == 0) wred[wave] = m, wleast[wave] = least;
    }
    const int64_t zs = (int64_t)p.batch * M;
    float* out = S == 1 ? p.out : p.partial + blockIdx.z * zs;
    auto at = [&](int row, int tok) { return FMT == kTern ? (int64_t)row * p.batch + tok : (int64_t)tok * M + row; };
    // the tile's outputs of one token with FP32 products: two threads per weight row, half of the slice each
    auto fp32_token = [&](int tok) {
        const int row = bx * kRmRows + (tid >> 1), k0 = kRmStep * s0, k1 = min(K, kRmStep * s1), mid = (k0 + k1) / 2;
        float v = row < M ? rows_fma<FMT>(p, row, tok, tid & 1 ? mid : k0, tid & 1 ? k1 : mid) : 0.0f;
        v += lane_xor1(v);
        if (row < M && (tid & 1) == 0) out[at(row, tok)] = v;
    };
    if constexpr (FMT == kOil8) {
        if (__syncthreads_or(!fin)) {
            for (int tok = tok0; tok < min(tok0 + 16 * G, p.batch); ++tok) fp32_token(tok);
            return;
        }
    }
    int sw = 0;
    if constexpr (FMT == kOil8) {
        sw = fp16_scale_shift(fmaxf(fmaxf(wred[0], wred[1]), fmaxf(wred[2], wred[3])));
        tab[tid] = rows_hl(ldexpf(cbv, sw));
    }
    CbPlanes shared_planes;
    if constexpr (O4)
        if (!p.cb_block) shared_planes = cb_planes(wt[0][0].c0, wt[0][0].c1);

    floatx4 ah[2][G], ax[2][G];  // hi x hi; the other products
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int g = 0; g < G; ++g) ah[t][g] = ax[t][g] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    const bool edge = FMT == kTern && bx == (int)gridDim.x - 1;  // a tile with the matrix's last row
    const uint8_t* brow = bs + q * 1024 + j * 16;  // lane (token j, chunk q) of piece m: + 256 m
    auto step_body = [&](int step, RowsTile<FMT> (&w)[2]) {
#pragma unroll
        for (int i = 0; i < NB; ++i) *(uint4*)(bs + i * 4096 + 16 * tid) = bv[i];
        __syncthreads();
        load_b(step + 1);
        RowsTile<FMT> cur[2] = {w[0], w[1]};
        load_w(step + 2, w);
        __builtin_amdgcn_sched_barrier(0);
        uint4 wa[2], wb[2];  // OIL8: the lane's 32 index bytes
        CbPlanes pl[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if constexpr (FMT == kOil8) {
                wa[t] = make_uint4(dpp_mix<0xc>(cur[t].x.x, cur[t].y.x), dpp_mix<0xc>(cur[t].x.y, cur[t].y.y),
                                   dpp_mix<0xc>(cur[t].x.z, cur[t].y.z), dpp_mix<0xc>(cur[t].x.w, cur[t].y.w));
                wb[t] = make_uint4(dpp_mix<0x3>(cur[t].y.x, cur[t].x.x), dpp_mix<0x3>(cur[t].y.y, cur[t].x.y),
                                   dpp_mix<0x3>(cur[t].y.z, cur[t].x.z), dpp_mix<0x3>(cur[t].y.w, cur[t].x.w));
            } else if constexpr (O4) {
                pl[t] = p.cb_block ? cb_planes(cur[t].c0, cur[t].c1) : shared_planes;
                if (kRmStep * step + 32 * q >= K) {  // columns past the row: weight 0 (an Inf entry would meet 0)
#pragma unroll
                    for (int e = 0; e < 4; ++e) pl[t].l[e] = pl[t].h[e] = 0;
                }
            } else if (edge) {
                const int64_t pos = (int64_t)min(row0 + 16 * t + j, M - 1) * (K >> 2) + (kRmStep / 4) * step + 8 * q;
                cur[t].c = codes8_at(cur[t].c, pos, tend);
            }
        }
        // piece m (columns 8 m .. of every 32) of tile t as A operands: hi, and OIL8's lo
        auto weights = [&](int t, int m, half8& Ah, half8& Al) {
            if constexpr (FMT == kOil8) {
                const uint32_t w0 = m == 0 ? wa[t].x : m == 1 ? wa[t].z : m == 2 ? wb[t].x : wb[t].z;
                const uint32_t w1 = m == 0 ? wa[t].y : m == 1 ? wa[t].w : m == 2 ? wb[t].y : wb[t].w;
                uint32_t gv[8];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    gv[e] = tab[(w0 >> (8 * e)) & 0xffu];
                    gv[4 + e] = tab[(w1 >> (8 * e)) & 0xffu];
                }
                u32x4 hv, lv;
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    hv[d] = __builtin_amdgcn_perm(gv[2 * d + 1], gv[2 * d], 0x05040100u);
                    lv[d] = __builtin_amdgcn_perm(gv[2 * d + 1], gv[2 * d], 0x07060302u);
                }
                Ah = __builtin_bit_cast(half8, hv);
                Al = __builtin_bit_cast(half8, lv);
            } else if constexpr (O4) {
                Ah = lookup8_natural(u4get(cur[t].n, m), pl[t]);
            } else {
                Ah = rows_tern8(m < 2 ? cur[t].c.x : cur[t].c.y, 2 * (m & 1));
            }
        };
        // the token operands of piece m and group g
        auto tokens = [&](int m, int g, half8& bh, half8& bl) {
            bh = *(const half8*)(brow + g * P * 4096 + 256 * m);
            if constexpr (P == 2) bl = *(const half8*)(brow + g * 8192 + 4096 + 256 * m);
        };
        // tile t's products with group g; h: the hi x hi sums (a step's alone, or from the slice's start)
        auto product = [&](int m, int t, int g, half8 Ah, half8 Al, half8 bh, half8 bl, floatx4& h) {
            if constexpr (FINE) {
                const floatx4 zero{0.0f, 0.0f, 0.0f, 0.0f};
                const floatx4 r = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ah, bh, zero, 0, 0, 0);
                h = m == 0 ? r : h + r;
            } else {
                if (STEP && m == 0) h = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                h = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ah, bh, h, 0, 0, 0);
            }
            if constexpr (P == 2) ax[t][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ah, bl, ax[t][g], 0, 0, 0);
            if constexpr (FMT == kOil8) ax[t][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Al, bh, ax[t][g], 0, 0, 0);
            if constexpr (FINE) {  // (2^22 lo x lo: one of them at 2^-11 of its scale, exact where it counts)
                const half8 a = Al * (_Float16)0x1p-11f;
                ax[t][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bl, ax[t][g], 0, 0, 0);
            }
        };
        if constexpr (FMT == kOil4) {  // the step's A operands first: a group's step sums are then 8 registers
            half8 Ah[4][2], Al;
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int t = 0; t < 2; ++t) weights(t, m, Ah[m][t], Al);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                floatx4 st[2];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    half8 bh, bl;
                    tokens(m, g, bh, bl);
#pragma unroll
                    for (int t = 0; t < 2; ++t) product(m, t, g, Ah[m][t], Al, bh, bl, st[t]);
                }
                ah[0][g] += st[0];
                ah[1][g] += st[1];
            }
        } else {
            floatx4 st[2][G];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                half8 bh[G], bl[G];
#pragma unroll
                for (int g = 0; g < G; ++g) tokens(m, g, bh[g], bl[g]);
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    half8 Ah, Al;
                    weights(t, m, Ah, Al);
#pragma unroll
                    for (int g = 0; g < G; ++g) product(m, t, g, Ah, Al, bh[g], bl[g], STEP ? st[t][g] : ah[t][g]);
                }
            }
            if constexpr (STEP) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        if constexpr (FINE) {  // the addition's rounding joins the small products
                            const floatx4 s = ah[t][g] + st[t][g];
                            ax[t][g] += (st[t][g] - (s - ah[t][g])) * 2048.0f;
                            ah[t][g] = s;
                        } else {
                            ah[t][g] += st[t][g];
                        }
                    }
            }
        }
        __syncthreads();
    };
    for (int step = s0; step < s1; step += 2) {
        step_body(step, wt[0]);
        if (step + 1 < s1) step_body(step + 1, wt[1]);
    }

    uint32_t wide = 0;  // this lane's tokens of a wide range
    if constexpr (FMT != kOil4B) {
        if (p.fp32) {
            bool wide_cb = false;
            if constexpr (FMT == kOil8) {
                const uint32_t least = 0u - max(max(wleast[0], wleast[1]), max(wleast[2], wleast[3]));
                wide_cb = least != 0 && 141 - sw - (int)(least >> 23) > 28;  // (141 - sw: the largest entry's exponent)
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const bool w = rs[g] > kRowWide / 2 && rs[g] != kRowFp32;  // (a shift is -128 .. 165)
                if (w) rs[g] -= kRowWide;
                if (w || wide_cb) wide |= 1u << g;
            }
        }
    }
    // the scaled sum of row 16 t + 4 q + i and token 16 g + j
    auto scaled = [&](int t, int g, int i) {
        const float hi = ah[t][g][i], lo = ax[t][g][i] * 0x1p-11f;
        return P == 1 ? hi : FMT == kOil8 ? hi + lo : oil4_hi_lo(hi, lo);
    };
    // ---- D: lane (j, q) holds rows 4q + i of token j
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int tok = tok0 + 16 * g + j;
        if (tok >= p.batch || (FMT != kOil4B && rs[g] == kRowFp32)) continue;
        const int sh = rs[g] + sw;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int row = row0 + 16 * t + 4 * q;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = ldexpf(scaled(t, g, i), -sh);
            if constexpr (FMT == kOil4B) {
                if (S == 1) {
                    uint16_t* d16 = (uint16_t*)p.out + (int64_t)tok * M + row;
                    uint16_t h[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) h[i] = f32_to_bf16_rne(v[i]);
                    if (row + 3 < M && ((uintptr_t)d16 & 7u) == 0) {
                        *(uint2*)d16 = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (row + i < M) d16[i] = h[i];
                    }
                    continue;
                }
            }
            float* dst = out + at(row, tok);
            if (FMT != kTern && row + 3 < M && ((uintptr_t)dst & 15u) == 0) {
                *(float4*)dst = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (row + i < M) out[at(row + i, tok)] = v[i];
            }
        }
    }
    if constexpr (FMT != kOil4B) {  // (every wave holds the tile's shifts)
#pragma unroll
        for (int g = 0; g < G; ++g)
            for (uint64_t m = __builtin_amdgcn_ballot_w64(q == 0 && tok0 + 16 * g + j < p.batch && rs[g] == kRowFp32); m;
                 m &= m - 1)
                fp32_token(tok0 + 16 * g + __builtin_ctzll(m));
        bool nan = false;  // OIL4: also an infinite entry times a value whose parts are 0, where the product is infinite
        if constexpr (FMT == kOil4) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                float z = 0.0f;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) z = fmaf(0.0f, ax[t][g][i], fmaf(0.0f, ah[t][g][i], z));
                nan = nan || (p.fp32 && z != 0.0f && tok0 + 16 * g + j < p.batch);  // (past it: whatever was there)
            }
        }
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(wide != 0 || nan) == 0, 1)) return;
        // A value below 2^-28 of its row's maximum (scaled: 2^-14) is held to 2^-36 only.  FP32 products are as far off
        // as n of those are together from outputs of sqrt(n) 2^-13 of the largest weight: an output below that is done
        // again, by the wave.  (All outputs of such a token in FP32, in every workgroup: 40 tokens x 4000 x 4080, 1, 10 and
        // 40 of them of a wide range, 86, 660 and 2530 us; this 23 us for any of them, and walking all tokens 125.)
        const int k0 = kRmStep * s0, k1 = min(K, kRmStep * s1);
        const float n = sqrtf((float)(k1 - k0)) * 0x1p-13f;
        float top = FMT == kOil8 ? 0x1p15f : 1.0f;  // OIL4: the largest entry of row lane % 32's blocks in the slice
        if constexpr (O4) {
            const int blk = p.cb_block ? p.cb_block : K, b1 = (k1 - 1) / blk;
            const uint16_t* cb = (const uint16_t*)p.cb;
            if (p.cb_block) cb += (int64_t)min(row0 + (lane & 31), M - 1) * (K / blk) * 16;
            top = 0.0f;
#pragma unroll 4
            for (int b = k0 / blk + (lane >> 5); b <= b1; b += 2) {
                const uint4 c[2] = {ld16(cb + 16 * b), ld16(cb + 16 * b + 8)};
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t d = u4get(c[e >> 2], e & 3);
                    top = fmaxf(top, fmaxf(fabsf(h2f(d & 0xffffu)), fabsf(h2f(d >> 16))));
                }
            }
            top = fmaxf(top, __shfl_xor(top, 32, 64));
        }
        uint32_t again = 0;  // this lane's outputs (8 g + 4 t + i)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float least = n * (O4 ? __shfl(top, 16 * t + 4 * q + i, 64) : top);
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const float d = scaled(t, g, i);
                    const bool redo = (((wide >> g) & 1u) != 0 && !(fabsf(d) >= least)) || (FMT == kOil4 && d != d);
                    if (redo && row0 + 16 * t + 4 * q + i < M && tok0 + 16 * g + j < p.batch && rs[g] != kRowFp32)
                        again |= 1u << (8 * g + 4 * t + i);
                }
            }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores above: the same addresses follow
        for (uint64_t m = __builtin_amdgcn_ballot_w64(again != 0); m; m &= m - 1) {
            const int l = __builtin_ctzll(m);
            for (uint32_t e = __builtin_amdgcn_readlane(again, l); e; e &= e - 1) {
                const int b = __builtin_ctz(e), tok = tok0 + 16 * (b >> 3) + (l & 15);
                const int row = row0 + 16 * ((b >> 2) & 1) + 4 * (l >> 4) + (b & 3);
                const float v = group_sum<64>(rows_fma<FMT>(p, row, tok, k0 + lane, k1, 64));
                if (lane == 0) out[at(row, tok)] = v;
            }
        }
    }
}

// what t = a + b left out of a + b (exact; 0 where t is not finite, so that t stays the result)
__device__ __forceinline__ float rows_rest(float a, float b, float t) {
    const float z = t - a, r = (a - (t - z)) + (b - z);
    return __builtin_isfinite(t) ? r : 0.0f;
}

// FINE: with the roundings of the additions added up beside.
// out[i] = sum over slices z = 0, 1, ... of partial[z][i] (a fixed order); all loads before the first add.  Four
// values per thread where both arrays are 16-byte aligned (n % 4 == 0).  HALF: out is bf16.  gridDim.y > 1: sg's matrix
// blockIdx.y.
template <bool VEC, bool HALF = false, bool FINE = false>
__global__ __launch_bounds__(kRmT) void rows_reduce_k(const float* __restrict__ partial, float* __restrict__ out,
                                                      int64_t n, int S, RowsSegs sg, int batch) {
    const int64_t i = ((int64_t)blockIdx.x * kRmT + threadIdx.x) * (VEC ? 4 : 1);
    if (gridDim.y > 1) {
        const int y = blockIdx.y;
        n = (int64_t)batch * (y == 0 ? sg.M[0] : y == 1 ? sg.M[1] : sg.M[2]);
        out = y == 0 ? sg.out[0] : y == 1 ? sg.out[1] : sg.out[2];
        partial += y == 0 ? sg.p0[0] : y == 1 ? sg.p0[1] : sg.p0[2];
    }
    if (i >= n) return;
    if constexpr (VEC) {
        float4 v[kRmSlices];
#pragma unroll
        for (int z = 0; z < kRmSlices; ++z) v[z] = z < S ? ldf4(partial + z * n + i) : make_float4(0, 0, 0, 0);
        float4 s = v[0], e = make_float4(0, 0, 0, 0);
#pragma unroll
        for (int z = 1; z < kRmSlices; ++z)
            if (z < S) {
                const float4 t = make_float4(s.x + v[z].x, s.y + v[z].y, s.z + v[z].z, s.w + v[z].w);
                if constexpr (FINE)
                    e = make_float4(e.x + rows_rest(s.x, v[z].x, t.x), e.y + rows_rest(s.y, v[z].y, t.y),
                                    e.z + rows_rest(s.z, v[z].z, t.z), e.w + rows_rest(s.w, v[z].w, t.w));
                s = t;
            }
        if constexpr (FINE) s = make_float4(s.x + e.x, s.y + e.y, s.z + e.z, s.w + e.w);
        if constexpr (HALF)
            *(uint2*)((uint16_t*)out + i) = make_uint2(f32_to_bf16_rne(s.x) | ((uint32_t)f32_to_bf16_rne(s.y) << 16),
                                                       f32_to_bf16_rne(s.z) | ((uint32_t)f32_to_bf16_rne(s.w) << 16));
        else
            *(float4*)(out + i) = s;
    } else {
        float v[kRmSlices];
#pragma unroll
        for (int z = 0; z < kRmSlices; ++z) v[z] = z < S ? partial[z * n + i] : 0.0f;
        float s = v[0], e = 0.0f;
#pragma unroll
        for (int z = 1; z < kRmSlices; ++z)
            if (z < S) {
                const float t = s + v[z];
                if constexpr (FINE) e += rows_rest(s, v[z], t);
                s = t;
            }
        if constexpr (FINE) s += e;
        if constexpr (HALF) ((uint16_t*)out)[i] = f32_to_bf16_rne(s);
        else out[i] = s;
    }
}

struct RowsPlan {
    int G, tiles, S, steps;
    int64_t rtiles;
};
// (M rows in nseg matrices: at most nseg - 1 row tiles more than M fills; alone: a call's only product; fine: token
// tiles of at most 48, whose sums the FINE kernels hold in registers)
inline RowsPlan rows_plan(int64_t M, int64_t K, int64_t batch, int nseg = 1, bool alone = false, bool fine = false) {
    RowsPlan p{};
    p.steps = (int)((K + kRmStep - 1) / kRmStep);
    const int64_t most = fine ? 48 : 64, nt = (batch + most - 1) / most;
    p.G = (int)((batch + 16 * nt - 1) / (16 * nt));  // token tiles of 16, 32, 48 or 64, as even as they go
    p.tiles = (int)((batch + 16 * p.G - 1) / (16 * p.G));
    p.rtiles = (M + kRmRows - 1) / kRmRows + nseg - 1;
    const int64_t wgs = p.rtiles * p.tiles;
    // K slices: about one workgroup per CU (a workgroup's fixed cost, ~5 us of load latency, table and output, is then
    // paid once per CU: 4096 x 4096 at 40 tokens 24.2 / 19.5 / 23.0 us for 4 / 8 / 16 slices); two per CU for long
    // slices (16384 x 11008: 87 -> 80 us) or where one leaves a CU in three idle (4096 x 4096 at 300 tokens, 160
    // workgroups: 51 / 43 / 37 us for 1 / 2 / 3 slices); one slice for more workgroups than CUs.
    const int64_t per = wgs > 256 ? 1 : wgs > 128 ? (p.steps >= 16 ? 512 / wgs : 1)
                      : wgs >= 64 && p.steps >= 48 ? 512 / wgs : 256 / wgs;
    p.S = (int)std::max<int64_t>(1, std::min<int64_t>({per, p.steps / 2, kRmSlices}));
    // alone, up to 512 columns and 48 tokens per tile: one slice, since the reduction's launch (3 us of host time) costs
    // more than two steps more in a chain (M = 256 .. 16384, 17 .. 32 tokens 15.1 .. 15.8 us with two slices, 12.3 ..
    // 13.1 with one, 64 tokens 15.1 and 15.9); within a prompt's queue the split is the faster (60 tokens of hidden 512:
    // 5 %).
    if (alone && p.steps <= 4 && p.G <= 3) p.S = 1;
    return p;
}
inline size_t al256r(size_t n) { return (n + 255) & ~(size_t)255; }
inline size_t rows_a16_bytes(const RowsPlan& p, int parts = 2) {
    return (size_t)p.tiles * p.G * parts * p.steps * 4096;
}

template <int FMT, bool FINE = false>
hipError_t rows_run(RowsArgs a, const RowsPlan& p, void* ws, hipStream_t s, const RowsSegs& sg = RowsSegs{}) {
    int64_t n = (int64_t)a.M * a.batch;
    uint16_t* a16 = (uint16_t*)ws;
    int* rsh = (int*)((char*)ws + rows_a16_bytes(p, kParts<FMT>));
    float* partial = (float*)((char*)rsh + al256r((size_t)a.batch * 4));
    a.a16 = a16;
    a.rsh = rsh;
    a.partial = partial;
    a.steps = p.steps;
    const bool vec = ((uintptr_t)a.x & 15u) == 0 && a.K % 4 == 0;
    if constexpr (FMT == kOil4B)
        rows_half_k<<<(unsigned)a.batch, kRmT, 0, s>>>((const uint16_t*)a.x, a16, rsh, a.K, 4 * p.steps);
    else if (vec)
        rows_split_k<FMT == kTern, true><<<(unsigned)a.batch, kRmT, 0, s>>>(a.x, a16, rsh, a.K, 4 * p.steps, a.fp32);
    else
        rows_split_k<FMT == kTern, false><<<(unsigned)a.batch, kRmT, 0, s>>>(a.x, a16, rsh, a.K, 4 * p.steps, a.fp32);
    const dim3 grid((unsigned)(sg.n > 1 ? sg.t1[sg.n - 1] : p.rtiles), (unsigned)p.tiles, (unsigned)p.S);
    switch (p.G) {
        case 1: rows_mfma_k<FMT, 1, FINE><<<grid, kRmT, 0, s>>>(a, sg); break;
        case 2: rows_mfma_k<FMT, 2, FINE><<<grid, kRmT, 0, s>>>(a, sg); break;
        case 3: rows_mfma_k<FMT, 3, FINE><<<grid, kRmT, 0, s>>>(a, sg); break;
        default:
            if constexpr (FINE) return hipErrorInvalidValue;  // (rows_plan: fine)
            else rows_mfma_k<FMT, 4><<<grid, kRmT, 0, s>>>(a, sg);
    }
    if (p.S > 1) {
        bool vec4 = n % 4 == 0 && ((uintptr_t)a.out & 15u) == 0;
        if (sg.n > 1) {
            n = 0;
            vec4 = true;
            for (int i = 0; i < sg.n; ++i) {
                n = std::max(n, (int64_t)sg.M[i] * a.batch);
                vec4 = vec4 && (int64_t)sg.M[i] * a.batch % 4 == 0 && ((uintptr_t)sg.out[i] & 15u) == 0;
            }
        }
        const unsigned ny = sg.n > 1 ? sg.n : 1;
        constexpr bool HALF = FMT == kOil4B;
        if (vec4)
            rows_reduce_k<true, HALF, FINE><<<dim3((unsigned)((n / 4 + kRmT - 1) / kRmT), ny), kRmT, 0, s>>>(
                partial, a.out, n, p.S, sg, a.batch);
        else
            rows_reduce_k<false, HALF, FINE><<<dim3((unsigned)((n + kRmT - 1) / kRmT), ny), kRmT, 0, s>>>(
                partial, a.out, n, p.S, sg, a.batch);
    }
    return hipGetLastError();
}

inline bool rows_sizes(int64_t M, int64_t K, int64_t batch) {
    return M >= 1 && M < (1ll << 31) - kRmRows && K >= 32 && K <= (1 << 20) && batch >= 1 && batch <= 65536 &&
           M * batch < (1ll << 37);
}

}  // namespace

size_t rows_mfma_workspace_bytes(int64_t M, int64_t K, int64_t batch, int nseg) {
    size_t need = 0;
    for (const bool fine : {false, true}) {
        const RowsPlan p = rows_plan(M, K, batch, nseg, false, fine);
        need = std::max(need, rows_a16_bytes(p) + al256r((size_t)batch * 4) + (p.S > 1 ? (size_t)(p.S * M * batch * 4) : 0));
    }
    return need;
}

size_t rows_bf16_workspace_bytes(int64_t M, int64_t K, int64_t batch) {
    const RowsPlan p = rows_plan(M, K, batch);
    return rows_a16_bytes(p, 1) + al256r((size_t)batch * 4) + (p.S > 1 ? (size_t)(p.S * M * batch * 4) : 0);
}

// ---- which route: estimated microseconds (eager calls, MI355X) ------------------
namespace {
// this file's three launches: 14.8 us for any little work (each launch costs the host ~3 us), 1.7 us (OIL8) or
// 1.85 us (OIL4) per step of 128 columns of a full 128 x 64 tile on a CU, and for few tokens the weight stream
double rows_us(int64_t M, int64_t K, int64_t batch, double step_us) {
    const RowsPlan p = rows_plan(M, K, batch);
    const double steps = (double)p.rtiles * p.tiles * p.steps / 256.0;
    return 14.8 + std::max(steps * step_us * (p.G + 1) / 5.0 - 4.0, 0.0);
}
// the same for whole rounds of a full chip, against a tiled GEMM: the busiest CU's steps, and the slices' partial sums
// written and read (within 15 % at 128 .. 512 tokens x 4096 .. 32000 x 2048 .. 4096)
double rows_busy_us(int64_t M, int64_t K, int64_t batch, double step_us) {
    const RowsPlan p = rows_plan(M, K, batch);
    const double most = (double)((p.rtiles * p.tiles * p.S + 255) / 256);
    return 10.8 + most * p.steps / p.S * step_us * (p.G + 1) / 5.0 + (p.S > 1 ? 2e-6 * p.S * M * batch : 0.0);
}
// the kernels that walk tokens one after another (a launch of their own: 8.7 us eagerly).  Measured at M = 512 ..
// 16384, 1 .. 16 tokens: OIL8 rows of up to 4096 0.98 .. 11.9 us per token, OIL4 rows of up to 2048 / 4096 1.85 / 3.9
// us per token up to 4400 rows, longer rows (one wave per output) 2.8 / 3.2 us per 1024 columns up to 1600 / 2900 rows
double walk_us(int64_t M, int64_t K, int64_t batch, bool oil8, bool fast) {
    if (!fast) return batch * (K / 1024.0) * (oil8 ? 2.8 * std::max(1.0, M / 1600.0) : 3.2 * std::max(1.0, M / 2900.0));
    if (oil8) return batch * (0.7 + M / 4096.0 * (0.8 + K / 1860.0));
    return batch * (K <= 2048 ? 1.85 : 3.9) * std::max(1.0, M / 4400.0);
}
}  // namespace

// OIL8: K % 16 == 0, 16-byte aligned indices.  gemm: the prompt GEMM takes the call (128 tokens and more); bt: the
// batched GEMV does (16 tokens per launch pair).
bool oil8_rows_better(const Oil8Seg* seg, int nseg, int64_t K, int64_t batch, bool aligned, bool gemm, bool bt) {
    if (nseg < 1 || nseg > 3) return false;
    int64_t M = 0;
    for (int i = 0; i < nseg; ++i) {
        if (seg[i].rows < 1 || ((uintptr_t)seg[i].idx & 15u) != 0) return false;
        M += seg[i].rows;
    }
    if (!rows_sizes(M, K, batch) || K % 16 != 0) return false;
    if (gemm) {
        // a round of 256 tiles of 128 x 64 (54 us at K = 4096), or of 256 x 64 where those fill the chip (98 us; 384
        // tiles, 476 tokens x 12288, 150 us, and 204 us here)
        const int64_t t = M / 64, wide = (batch + 255) / 256 * t, narrow = (batch + 127) / 128 * t;
        const double g = wide >= 256 ? 5.0 + 23.3 * (K / 1024.0) * (wide / 256.0)
                                     : 5.0 + (12.2 + narrow / 110.0) * (K / 1024.0);
        return 1.05 * rows_busy_us(M, K, batch, 1.7) < g;
    }
    const double us = rows_us(M, K, batch, bt || K > kRmFineCols ? 1.7 : 2.1);
    // 16 tokens per launch, or launch pair where K is split (K > 512), against two launches or three: 17 tokens of K =
    // 1024 .. 4096 20 .. 86 us against 15 .. 48, of K = 512 14.7 .. 16.0 against 12.3 .. 12.9
    if (bt) return batch > 16;
    return us < walk_us(M, K, batch, true, aligned && K <= 4096);
}

// OIL4: K % 32 == 0, codebook blocks of a multiple of 32 columns, 16-byte aligned weights.
bool oil4_rows_better(const uint8_t* nib, const uint16_t* cbs, int64_t cb_block, int64_t M, int64_t K, int64_t batch,
                      bool aligned, bool gemm, bool bt) {
    if (!rows_sizes(M, K, batch) || K % 32 != 0 || cb_block % 32 != 0 || cb_block >= (1 << 30) ||
        (((uintptr_t)nib | (uintptr_t)cbs) & 15u) != 0)
        return false;
    if (gemm) return 1.05 * rows_busy_us(M, K, batch, 1.6) < oil4_gemm_x32_us(batch, M, K);
    const double us = rows_us(M, K, batch, 1.85);
    // as for OIL8: 17 tokens of K = 1024 .. 4096 18 .. 94 us against 15 .. 52.  K = 512 in two launches: 11.5 .. 12.3 us up
    // to 16384 rows against 12.4 .. 12.7, 15.4 us at 32000 against 12.9 (about 2 x (4.4 us + 1e-4 us per row))
    if (bt) return batch > 16 && !(K == 512 && batch <= 32 && M < 18000);
    return us < walk_us(M, K, batch, false, aligned && K <= 4096);
}

// Ternary weights, FP32 tokens: against one wave per output (8 us for little work, 3.5 us per 1024 columns for up to
// 8000 outputs).
bool tern_rows_better(int64_t M, int64_t K, int64_t batch) {
    return rows_sizes(M, K, batch) && K % 4 == 0 && M * (K / 4) >= 8 &&
           K * std::max(1.0, (double)M * batch / 8000.0) > 4000.0;
}

// bf16 prompt rows (M: weight rows), K % 32 == 0 and codebook blocks of a multiple of 32 columns: against the tiled
// kernels' estimate (oil4_prefill_us).  Here 13.5 us for any little work, 3 us for the slice reduction, 1.05 us per step
// of a 128 x 64 tile on the busiest CU (measured at 100 .. 2000 tokens x 1200 .. 28672 x 1664 .. 8192: within 15 %, hence the
// margin).  Few tokens or rows: the tiled kernels' 256-token tiles leave CUs idle and split no K (158 x 5120 x 3840:
// 47 us there, 33 here; 300 x 14336 x 3840: 68 and 105).
bool oil4_rows_bf16_better(int64_t M, int64_t K, int64_t batch, double tiled_us) {
    if (!rows_sizes(M, K, batch) || K % 32 != 0) return false;
    const RowsPlan p = rows_plan(M, K, batch);
    const double most = (double)((p.rtiles * p.tiles * p.S + 255) / 256);  // workgroups on the busiest CU
    const double us = 13.5 + (p.S > 1 ? 3.0 : 0.0) + 1.05 * most * p.steps / p.S;
    return 1.12 * us < tiled_us;
}

hipError_t launch_oil8_rows(const Oil8Seg* seg, int nseg, const float* x, int64_t K, int64_t batch, bool fp32, void* ws,
                            hipStream_t s, bool alone) {
    RowsSegs sg{};
    int64_t M = 0, tiles = 0;
    for (int i = 0; i < nseg; ++i) M += seg[i].rows;
    const bool fine = fp32 && K <= kRmFineCols;
    const RowsPlan p = rows_plan(M, K, batch, nseg, alone, fine);
    sg.n = nseg;
    M = 0;
    for (int i = 0; i < 3; ++i) {
        const Oil8Seg& g = seg[i < nseg ? i : nseg - 1];
        sg.w[i] = g.idx, sg.cb[i] = g.cb, sg.out[i] = g.y;
        sg.M[i] = (int)g.rows;
        sg.p0[i] = p.S * M * batch;
        if (i < nseg) {
            M += g.rows;
            tiles += (g.rows + kRmRows - 1) / kRmRows;
        }
        sg.t1[i] = (int)tiles;
    }
    RowsArgs a{seg[0].idx, seg[0].cb, nullptr, nullptr, x, seg[0].y, nullptr, (int)seg[0].rows, (int)K, (int)batch, 0, 0,
               fp32};
    return fine ? rows_run<kOil8, true>(a, p, ws, s, sg) : rows_run<kOil8>(a, p, ws, s, sg);
}
hipError_t launch_oil4_rows(const uint8_t* nib, const uint16_t* cbs, int64_t cb_block, const float* x, float* y,
                            int64_t M, int64_t K, int64_t batch, bool fp32, void* ws, hipStream_t s, bool alone) {
    RowsArgs a{nib, cbs, nullptr, nullptr, x, y, nullptr, (int)M, (int)K, (int)batch, 0, (int)cb_block, fp32};
    return rows_run<kOil4>(a, rows_plan(M, K, batch, 1, alone), ws, s);
}
hipError_t launch_oil4_rows_bf16(const uint8_t* nib, const uint16_t* cbs, int64_t cb_block, const uint16_t* x,
                                 uint16_t* y, int64_t M, int64_t K, int64_t batch, void* ws, hipStream_t s) {
    RowsArgs a{nib, cbs, nullptr, nullptr, (const float*)x, (float*)y, nullptr, (int)M, (int)K, (int)batch, 0,
               (int)cb_block, false};
    return rows_run<kOil4B>(a, rows_plan(M, K, batch), ws, s);
}
hipError_t launch_tern_rows(const uint8_t* w, const float* x, float* out, int64_t M, int64_t K, int64_t batch,
                            void* ws, hipStream_t s) {
    RowsArgs a{w, nullptr, nullptr, nullptr, x, out, nullptr, (int)M, (int)K, (int)batch, 0, 0, true};
    return rows_run<kTern>(a, rows_plan(M, K, batch), ws, s);
}

}  // namespace mth

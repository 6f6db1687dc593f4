// attn_prefill.hip — causal attention of a prompt chunk on gfx950 MFMA.
//
// Workgroup (head h, sequence b, tile of 64 query rows): rows b np + i of q /
// out at positions p0 + i, each attending to cache rows 0 .. p0 + i of kv head
// h % kv_heads (src/transformer.cpp:188-348 for every prompt row), scale
// 1/sqrt(D).  The context streams through LDS in tiles of 64 positions with a
// running maximum and rescaled sums, so each K / V row is read once per 64
// query rows.
//
// Arithmetic.  FP32 accurate on bf16 matrix cores: a value x is split into
// three bf16 parts, x = x1 + x2 + x3 (8 significant bits each, FP32's exponent
// range, so no scaling; x3 is exact), and a product takes the part pairs down to
// 2^-16 of it: 1x1, 1x2, 2x1, 2x2, 1x3, 3x1 (what is left lies below FP32's
// rounding); rows of a bf16 cache are one part, and a product takes three.  Each
// part product is exact in FP32; v_mfma_f32_16x16x32_bf16 sums in FP32, with
// fewer roundings per score (24) and per output and tile (12) than one FMA per
// element.  Softmax in FP32.  A tile with an Inf or a NaN in q, K or V (which
// cannot be split) sends the workgroup to FP32 FMAs over the same rows.
//
// Tiling.  8 waves, two per SIMD: wave (r, c) takes 16 query rows and half c of
// every tile's positions, with a maximum, sum and output of its own; the halves
// meet through LDS at the end (no exchange inside the loop).  A wave holds its
// Q parts in registers (A), reads K parts [position][d] from LDS (B), writes
// its 16 x 32 probabilities to its own LDS rows, reads them back as A parts, and
// reads V parts, stored transposed [d][position] (B).  16-byte chunks
// XOR-swizzled by row.  The next tile's K and V rows are loaded into registers
// while this one is computed.
// Tiles of 64 rows, latest first: 32 heads x 16 tiles of a 1024-row chunk give
// the CUs even shares of the triangle.
//
// Bound: MFMA issue (half of the wave cycles) and, between the two barriers of a
// tile, the splitting of K and V.  Times of one layer at 32 heads x 128, FP32
// cache (FP32 FMAs with both operands from LDS -> here): 1024 rows 406 -> 95 us,
// 476 rows after 1024 431 -> 120; 16 x 64 rows of a bf16 cache 50 -> 20; one
// sequence of 2000 rows and 8 heads 481 -> 148.  Four waves of whole tiles took
// 146 us on average where eight of halves take 107.  Relative error against 64
// bits: 6.8e-7 -> 4.8e-7, 1.1e-6 -> 7.2e-7.
#include <type_traits>

#include "common.h"
#include "launch.h"

namespace mth {
namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));

constexpr int kApQ = 64, kApK = 64, kApT = 512;  // query rows, positions per tile, threads
constexpr int kApP = kApK / 2 + 4;               // floats per probability row

template <int D, int KP>
struct ApLds {
    static constexpr int k = 0;                           // [KP][64 positions][D] bf16
    static constexpr int v = KP * kApK * D * 2;           // [KP][D][64 positions] bf16
    static constexpr int p = 2 * v;                       // [8 waves][16 rows][kApP] f32
    static constexpr int bytes = p + 8 * 16 * kApP * 4;
    static_assert(4 * 16 * D * 4 <= p, "the second halves' outputs fit over the K and V parts");
};

// x[0..7] = sum of P bf16 parts; bad (0 so far) becomes NaN where a part is not finite (a product with 0 per value)
template <int P>
__device__ __forceinline__ void ap_split(const float (&x)[8], bf8 (&part)[P], float& bad) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        f2 r = {x[e], x[e + 1]};
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const bf2 b = __builtin_convertvector(r, bf2);
            part[i][e] = b[0];
            part[i][e + 1] = b[1];
            const f2 w = __builtin_convertvector(b, f2);
            if (i == 0) bad = fmaf(w[0], 0.0f, fmaf(w[1], 0.0f, bad));
            r = r - w;
        }
    }
}

// FP32 path of one workgroup: wave w takes rows w, w + 8, ...; lane = position of a block of 64 for the scores, D / 64
// columns for the weighted sum.
template <int D, typename KV>
__device__ __noinline__ void ap_fp32(const float* q, const KV* kc, const KV* vc, float* out, int64_t row0, int64_t crow,
                                     int64_t qstride, int nq, int pos0, float scale) {
    auto wide = [](KV v) {
        if constexpr (sizeof(KV) == 2) return __uint_as_float((uint32_t)v << 16);
        else return v;
    };
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr int NC = D / 64;
    for (int r = wave; r < nq; r += kApT / 64) {
        const float* qr = q + (row0 + r) * qstride;
        const int ctx = pos0 + r + 1;
        float m = -INFINITY, l = 0.0f, o[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) o[c] = 0.0f;
        for (int t0 = 0; t0 < ctx; t0 += 64) {
            const int t = t0 + lane, tc = min(t, ctx - 1);
            float s = 0.0f;
            for (int d = 0; d < D; ++d) s = fmaf(qr[d], wide(kc[(crow + tc) * D + d]), s);
            s = t < ctx ? s * scale : -INFINITY;
            const float mn = fmaxf(m, wave_max(s)), alpha = expf(m - mn), p = t < ctx ? expf(s - mn) : 0.0f;
            l = fmaf(l, alpha, group_sum<64>(p));
            m = mn;
#pragma unroll
            for (int c = 0; c < NC; ++c) o[c] *= alpha;
            const int n = min(64, ctx - t0);
            for (int j = 0; j < n; ++j) {
                const float pj = __shfl(p, j, 64);
#pragma unroll
                for (int c = 0; c < NC; ++c) o[c] = fmaf(pj, wide(vc[(crow + t0 + j) * D + 64 * c + lane]), o[c]);
            }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) out[(row0 + r) * qstride + 64 * c + lane] = o[c] * (1.0f / l);
    }
}

template <int D, typename KV>
__global__ __launch_bounds__(kApT) void attn_prefill_k(const float* __restrict__ q, const KV* __restrict__ kc,
                                                       const KV* __restrict__ vc, float* __restrict__ out, int np,
                                                       int p0, int heads, int kv_heads, int max_seq, float scale) {
    constexpr int KP = sizeof(KV) == 2 ? 1 : 3, KS = D / 32, NT = D / 16;
    constexpr int NU = kApK * D / 8 / kApT;  // 8-element units of a K (or V) tile per thread
    using L = ApLds<D, KP>;
    __shared__ __align__(16) uint8_t lds[L::bytes];
    const int h = blockIdx.x, b = blockIdx.y, i0 = (gridDim.z - 1 - blockIdx.z) * kApQ;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = lane & 15, g = lane >> 4;
    const int wr = wave & 3, wc = wave >> 2;
    const int nq = min(kApQ, np - i0), kh = h % kv_heads;
    const int64_t crow = ((int64_t)b * kv_heads + kh) * max_seq;  // cache row of position 0
    const int64_t qstride = (int64_t)heads * D, row0 = (int64_t)b * np + i0;
    const int ctx = p0 + i0 + nq;                                 // positions the tile's last row attends to
    const float* qh = q + h * D;

    // ---- K / V tile t0 into registers: K unit = (position u / (D / 8), columns 8 (u % (D / 8)) ..), V unit = (column
    // u % D, positions 8 (u / D) ..); positions past ctx are zeros
    typedef typename std::conditional<sizeof(KV) == 2, uint16_t, float>::type KE;
    KE kr[NU][8], vr[NU][8];
    // (FULL: every position of the tile is in the context: no clamps, one address per unit)
    auto load_as = [&](int t0, auto full) {
        constexpr bool FULL = decltype(full)::value;
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int u = tid + i * kApT;
            const int kp = t0 + u / (D / 8), kd = 8 * (u % (D / 8));
            const bool in = FULL || kp < ctx;
            const KV* ks = kc + (crow + (FULL ? kp : min(kp, ctx - 1))) * D + kd;
            if constexpr (KP == 1) {
                const uint4 w = ld16(ks);
#pragma unroll
                for (int e = 0; e < 8; ++e) kr[i][e] = in ? (uint16_t)(u4get(w, e >> 1) >> (16 * (e & 1))) : 0;
            } else {
                const float4 a = ldf4(ks), c = ldf4(ks + 4);
                const float f[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) kr[i][e] = in ? f[e] : 0.0f;
            }
            const int vd = u % D, vp = t0 + 8 * (u / D);
            const KV* vs = vc + (crow + vp) * D + vd;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const KE v = FULL ? vs[e * D] : vc[(crow + min(vp + e, ctx - 1)) * D + vd];
                vr[i][e] = FULL || vp + e < ctx ? v : (KE)0;
            }
        }
    };
    auto load = [&](int t0) {
        if (t0 + kApK <= ctx) load_as(t0, std::true_type{});
        else load_as(t0, std::false_type{});
    };
    float bad = 0.0f;  // NaN once a value of q, K or V was not finite
    auto parts = [&](const KE (&x)[8], bf8 (&part)[KP]) {
        if constexpr (KP == 1) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                part[0][e] = __builtin_bit_cast(__bf16, x[e]);
                bad = fmaf(__uint_as_float((uint32_t)x[e] << 16), 0.0f, bad);
            }
        } else {
            ap_split<KP>(x, part, bad);
        }
    };
    load(0);

    // ---- this wave's Q rows as A parts (rows past the tile: its last row)
    bf8 qa[KS][3];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const float* p = qh + (row0 + min(16 * wr + j, nq - 1)) * qstride + 32 * s + 8 * g;
        const float4 a = ldf4(p), c = ldf4(p + 4);
        const float f[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
        ap_split<3>(f, qa[s], bad);
    }
    float m[4], l[4];
    f4 o[NT];
#pragma unroll
    for (int i = 0; i < 4; ++i) m[i] = -INFINITY, l[i] = 0.0f;
#pragma unroll
    for (int n = 0; n < NT; ++n) o[n] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    // part pairs (A part, B part), smallest products first
    constexpr int NP = KP == 1 ? 3 : 6;
    constexpr int PA[2][6] = {{2, 1, 0, 0, 0, 0}, {2, 0, 1, 1, 0, 0}}, PB[2][6] = {{0, 0, 0, 0, 0, 0}, {0, 2, 1, 0, 1, 0}};
    constexpr int PI = KP == 1 ? 0 : 1;
    float* pw = (float*)(lds + L::p) + wave * 16 * kApP;
    const int qlast = p0 + i0 + 16 * wr + 15;  // the last position a row of this wave attends to

    for (int t0 = 0; t0 < ctx; t0 += kApK) {
        // ---- the tile's parts into LDS
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int u = tid + i * kApT;
            bf8 part[KP];
            parts(kr[i], part);
            const int kp = u / (D / 8), kch = u % (D / 8);
#pragma unroll
            for (int e = 0; e < KP; ++e)
                *(bf8*)(lds + L::k + (e * kApK + kp) * D * 2 + 16 * (kch ^ (kp & (D / 8 - 1)))) = part[e];
            parts(vr[i], part);
            const int vd = u % D, vch = u / D;
#pragma unroll
            for (int e = 0; e < KP; ++e) *(bf8*)(lds + L::v + (e * D + vd) * kApK * 2 + 16 * (vch ^ (vd & 7))) = part[e];
        }
        if (__syncthreads_or(bad != 0.0f)) {
            ap_fp32<D, KV>(qh, kc, vc, out + h * D, row0, crow, qstride, nq, p0 + i0, scale);
            return;
        }
        if (t0 + kApK < ctx) load(t0 + kApK);
        __builtin_amdgcn_sched_barrier(0);
        if (t0 + 32 * wc <= qlast) {  // (uniform per wave; later positions are masked for all of its rows)
            // ---- scores: D layout, lane (position 32 wc + 16 n + j, rows 4 g + i)
            f4 s[2];
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                s[n] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    bf8 kb[KP];
#pragma unroll
                    for (int e = 0; e < KP; ++e)
                        kb[e] = *(const bf8*)(lds + L::k + (e * kApK + 32 * wc + 16 * n + j) * D * 2 +
                                              16 * ((4 * ks + g) ^ ((16 * n + j) & (D / 8 - 1))));
#pragma unroll
                    for (int e = 0; e < NP; ++e)
                        s[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[ks][PA[PI][e]], kb[PB[PI][e]], s[n], 0, 0, 0);
                }
            }
            // ---- mask, running maximum, probabilities (FP32)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int qp = p0 + i0 + 16 * wr + 4 * g + i;
                float tm = -INFINITY;
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    s[n][i] = t0 + 32 * wc + 16 * n + j <= qp ? s[n][i] * scale : -INFINITY;
                    tm = fmaxf(tm, s[n][i]);
                }
                tm = group_reduce<16>(tm, MaxOp{});
                const float mn = fmaxf(m[i], tm);
                const float mref = mn == -INFINITY ? 0.0f : mn;  // (a row that sees none of this half yet)
                const float alpha = expf(m[i] - mref);
                float rs = 0.0f;
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const float p = expf(s[n][i] - mref);
                    pw[(4 * g + i) * kApP + 16 * n + j] = p;
                    rs += p;
                }
                l[i] = fmaf(l[i], alpha, group_reduce<16>(rs, AddOp{}));
                m[i] = mn;
#pragma unroll
                for (int n = 0; n < NT; ++n) o[n][i] *= alpha;
            }
            asm volatile("" ::: "memory");  // the wave's own LDS rows: program order
            // ---- P V
            {
                const float4 a = *(const float4*)(pw + j * kApP + 8 * g);
                const float4 c = *(const float4*)(pw + j * kApP + 8 * g + 4);
                const float f[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
                bf8 pa[3];
                float unused = 0.0f;  // (probabilities are finite)
                ap_split<3>(f, pa, unused);
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    bf8 vb[KP];
#pragma unroll
                    for (int e = 0; e < KP; ++e)
                        vb[e] = *(const bf8*)(lds + L::v + (e * D + 16 * n + j) * kApK * 2 + 16 * ((4 * wc + g) ^ (j & 7)));
#pragma unroll
                    for (int e = 0; e < NP; ++e)
                        o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[PA[PI][e]], vb[PB[PI][e]], o[n], 0, 0, 0);
                }
            }
        }
        __syncthreads();  // the tile is consumed
    }
    // ---- the two halves: second halves' outputs over the K and V parts, their (m, l) over the probabilities
    float* ob = (float*)lds + wr * 16 * D;
    float* mlb = (float*)(lds + L::p) + wr * 32;
    if (wc == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int n = 0; n < NT; ++n) ob[(4 * g + i) * D + 16 * n + j] = o[n][i];
            if (j == 0) mlb[2 * (4 * g + i)] = m[i], mlb[2 * (4 * g + i) + 1] = l[i];
        }
    }
    __syncthreads();
    if (wc == 1) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 16 * wr + 4 * g + i;
        if (r >= nq) continue;
        const float m2 = mlb[2 * (4 * g + i)], l2 = mlb[2 * (4 * g + i) + 1];
        const float mx = fmaxf(m[i], m2);  // finite: every row sees position 0
        const float w1 = expf(m[i] - mx), w2 = expf(m2 - mx);
        const float inv = 1.0f / fmaf(l[i], w1, l2 * w2);
        float* dst = out + (row0 + r) * qstride + h * D + j;
#pragma unroll
        for (int n = 0; n < NT; ++n) dst[16 * n] = fmaf(o[n][i], w1, ob[(4 * g + i) * D + 16 * n + j] * w2) * inv;
    }
}

}  // namespace

hipError_t launch_attn_prefill(const float* q, const void* kc, const void* vc, bool kv_bf16, float* out, int64_t rows,
                               int np, int p0, int heads, int kv_heads, int head_dim, int max_seq, hipStream_t s) {
    const dim3 grid((unsigned)heads, (unsigned)(rows / np), (unsigned)((np + kApQ - 1) / kApQ));
    const float scale = 1.0f / sqrtf((float)head_dim);
    const uint16_t *kb = (const uint16_t*)kc, *vb = (const uint16_t*)vc;
    const float *kf = (const float*)kc, *vf = (const float*)vc;
    if (head_dim == 64) {
        if (kv_bf16) attn_prefill_k<64, uint16_t><<<grid, kApT, 0, s>>>(q, kb, vb, out, np, p0, heads, kv_heads, max_seq, scale);
        else attn_prefill_k<64, float><<<grid, kApT, 0, s>>>(q, kf, vf, out, np, p0, heads, kv_heads, max_seq, scale);
    } else {
        if (kv_bf16) attn_prefill_k<128, uint16_t><<<grid, kApT, 0, s>>>(q, kb, vb, out, np, p0, heads, kv_heads, max_seq, scale);
        else attn_prefill_k<128, float><<<grid, kApT, 0, s>>>(q, kf, vf, out, np, p0, heads, kv_heads, max_seq, scale);
    }
    return hipGetLastError();
}

}  // namespace mth

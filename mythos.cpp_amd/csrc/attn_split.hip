// attn_split.hip — decode attention over a long KV cache, the context split
// over workgroups (gfx950).
//
// The semantics of attention_k without RoPE (dense.hip; the reference's
// inference branch with one query, src/transformer.cpp:188-348): head h of
// token b attends to cache rows 0 .. ctx-1 of kv head h % kv_heads, scale
// 1/sqrt(D), softmax, weighted sum of V.  One workgroup per (head, token)
// leaves most of the 256 CUs idle at decode sizes and every head of a
// grouped-query group reads the same K and V; here a workgroup takes one
// slice of T positions of one (token, kv head) for HG query heads at once,
// so each cache row is read once per HG heads and the slices fill the chip.
// Slice s leaves, per head, its maximum m, the sum l of exp(score - m) and
// the unnormalised output o[D] (FP32); attn_combine_k adds the slices in
// order with the weights exp(m - max m).
//
// Bound: the cache's bytes.  A wave issues its NL K rows' loads and its NL V
// rows' loads (16 bytes per lane, whole rows per D / 4 lanes) before it waits
// for any: 128 KB per workgroup at NL = 16, two workgroups per CU.  A score
// is 4 FMAs per lane and a sum over the row's D / 4 lanes (DPP).  2 tokens x
// 32 heads (8 kv heads) x 6000 positions of 128: 91.3 -> 28.4 us (98 MB); 16 x 40
// heads (5 kv heads) x 3000: 279 -> 87 us; 4 x 32 x 6000 without shared rows: 145 -> 138 us (786 MB, 5.7 TB/s).
#include "common.h"
#include "launch.h"

#pragma clang fp contract(off)

namespace mth {
namespace {

constexpr int kAsW = 4;  // waves per workgroup

// float4 of D / 4 lanes per row: rows per load instruction, positions per workgroup
template <int D, int NL>
constexpr int as_rows() { return (64 / (D / 4)) * kAsW * NL; }

template <int D, int HG, int NL>
__global__ __launch_bounds__(64 * kAsW, 2) void attn_split_k(const float* __restrict__ q, const float* kc,
                                                             const float* vc, float* __restrict__ po,
                                                             float* __restrict__ pml, int ctx, int heads, int kv_heads,
                                                             int max_seq, float scale) {
    constexpr int LPR = D / 4, PPI = 64 / LPR, T = as_rows<D, NL>(), NT = 64 * kAsW;
    __shared__ __align__(16) float sc[T * HG];         // scores, then probabilities: [position][head]
    __shared__ __align__(16) float part[kAsW][HG][D];
    __shared__ float red[kAsW][HG], lsum[kAsW][HG];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane % LPR, pr = lane / LPR;         // this lane's 4 columns, its row of a load
    const int s = blockIdx.x, S = gridDim.x, b = blockIdx.z;
    const int kh = blockIdx.y % kv_heads, hg = blockIdx.y / kv_heads;  // heads kh + kv_heads (HG hg + j), j < HG
    const int t0 = s * T, n = min(T, ctx - t0);        // positions of this slice (n >= 1)
    const int64_t row0 = ((int64_t)b * kv_heads + kh) * max_seq + t0;

    // position of load i: PPI kAsW i + PPI wave + pr (past the slice: clamped to its last row and not used)
    float4 qv[HG];
#pragma unroll
    for (int j = 0; j < HG; ++j)
        qv[j] = ldf4(q + ((int64_t)b * heads + kh + kv_heads * (HG * hg + j)) * D + 4 * c);
    float4 kv[NL], vv[NL];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NL; ++i) kv[i] = ldf4(kc + (row0 + min(PPI * (kAsW * i + wave) + pr, n - 1)) * D + 4 * c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NL; ++i) vv[i] = ldf4(vc + (row0 + min(PPI * (kAsW * i + wave) + pr, n - 1)) * D + 4 * c);
    __builtin_amdgcn_sched_barrier(0);

    float mx[HG];
#pragma unroll
    for (int j = 0; j < HG; ++j) mx[j] = -INFINITY;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int p = PPI * (kAsW * i + wave) + pr;
#pragma unroll
        for (int j = 0; j < HG; ++j) {
            const float d01 = fmaf(qv[j].y, kv[i].y, qv[j].x * kv[i].x), d23 = fmaf(qv[j].w, kv[i].w, qv[j].z * kv[i].z);
            const float v = group_reduce<LPR>(d01 + d23, AddOp{}) * scale;
            if (p < n) {
                if (c == 0) sc[p * HG + j] = v;
                mx[j] = fmaxf(mx[j], v);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < HG; ++j) {
        mx[j] = wave_max(mx[j]);
        if (lane == 0) red[wave][j] = mx[j];
    }
    __syncthreads();
    // probabilities relative to the slice's maximum: thread -> head tid % HG (a slice of only -inf scores: 0)
    const int hj = tid % HG;
    float m = red[0][hj];
#pragma unroll
    for (int w = 1; w < kAsW; ++w) m = fmaxf(m, red[w][hj]);
    const float mref = m == -INFINITY ? 0.0f : m;
    float l = 0.0f;
    for (int i = tid; i < n * HG; i += NT) {
        const float e = expf(sc[i] - mref);
        sc[i] = e;
        l += e;
    }
#pragma unroll
    for (int o = 32; o >= HG; o >>= 1) l += __shfl_xor(l, o, 64);
    if (lane < HG) lsum[wave][lane] = l;
    __syncthreads();

    float4 acc[HG];
#pragma unroll
    for (int j = 0; j < HG; ++j) acc[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int p = PPI * (kAsW * i + wave) + pr;
        if (p < n) {
#pragma unroll
            for (int j = 0; j < HG; ++j) {
                const float w = sc[p * HG + j];
                acc[j].x = fmaf(w, vv[i].x, acc[j].x);
                acc[j].y = fmaf(w, vv[i].y, acc[j].y);
                acc[j].z = fmaf(w, vv[i].z, acc[j].z);
                acc[j].w = fmaf(w, vv[i].w, acc[j].w);
            }
        }
    }
    // the rows of one load instruction (lanes l, l ^ LPR, ...), then the waves
#pragma unroll
    for (int j = 0; j < HG; ++j) {
#pragma unroll
        for (int o = LPR; o < 64; o <<= 1) {
            acc[j].x += __shfl_xor(acc[j].x, o, 64);
            acc[j].y += __shfl_xor(acc[j].y, o, 64);
            acc[j].z += __shfl_xor(acc[j].z, o, 64);
            acc[j].w += __shfl_xor(acc[j].w, o, 64);
        }
        if (lane < LPR) *(float4*)&part[wave][j][4 * c] = acc[j];
    }
    __syncthreads();
    for (int i = tid; i < HG * D; i += NT) {
        const int j = i / D, d = i % D;
        const int64_t h = (int64_t)b * heads + kh + kv_heads * (HG * hg + j);
        po[(h * S + s) * D + d] = (part[0][j][d] + part[1][j][d]) + (part[2][j][d] + part[3][j][d]);
    }
    if (tid < HG) {
        const int64_t h = (int64_t)b * heads + kh + kv_heads * (HG * hg + tid);
        pml[(h * S + s) * 2] = m;  // (tid < HG: this thread's head is tid)
        pml[(h * S + s) * 2 + 1] = (lsum[0][tid] + lsum[1][tid]) + (lsum[2][tid] + lsum[3][tid]);
    }
}

// out[h][d] = sum_s w_s o_s[d] / sum_s w_s l_s, w_s = exp(m_s - max m).  One workgroup per (token, head): the weights
// once in LDS, then thread = (4 columns, slice group): group g adds slices g, g + NG, ... (16 bytes each, U in flight),
// the groups are added in order.  S <= kAsMaxS.  (One thread per column walking all slices took 24 us at 375 slices.)
constexpr int kAsMaxS = 512, kAsC = 512;
template <int D>
__global__ __launch_bounds__(kAsC) void attn_combine_k(const float* __restrict__ po, const float* __restrict__ pml,
                                                       float* __restrict__ out, int S) {
    constexpr int LP = D / 4, NG = kAsC / LP, U = 4;
    __shared__ __align__(16) float part[NG][D];
    __shared__ float w[kAsMaxS], redm[kAsC / 64], redl[kAsC / 64];
    const int tid = threadIdx.x, c = tid % LP, g = tid / LP;
    const int64_t h = blockIdx.x;
    const float* ml = pml + h * S * 2;
    const float* o = po + h * S * D + 4 * c;
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = ldf4(o + (int64_t)min(g + u * NG, S - 1) * D);
    const bool in = tid < S;  // S <= kAsMaxS == kAsC: one slice's m and l per thread
    const float ms = in ? ml[2 * tid] : -INFINITY, ls = in ? ml[2 * tid + 1] : 0.0f;
    float m = wave_max(ms);
    if ((tid & 63) == 0) redm[tid >> 6] = m;
    __syncthreads();
    m = redm[0];
#pragma unroll
    for (int i = 1; i < kAsC / 64; ++i) m = fmaxf(m, redm[i]);
    const float ws = expf(ms - m);  // all -inf: NaN, as the undivided softmax gives
    if (in) w[tid] = ws;
    float l = group_sum<64>(in ? ws * ls : 0.0f);
    if ((tid & 63) == 0) redl[tid >> 6] = l;
    __syncthreads();
    float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int s0 = g; s0 < S; s0 += U * NG) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = s0 + u * NG;
            if (s < S) {
                const float f = w[s];
                a.x = fmaf(f, v[u].x, a.x);
                a.y = fmaf(f, v[u].y, a.y);
                a.z = fmaf(f, v[u].z, a.z);
                a.w = fmaf(f, v[u].w, a.w);
            }
        }
        if (s0 + U * NG < S)
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = ldf4(o + (int64_t)min(s0 + (U + u) * NG, S - 1) * D);
    }
    *(float4*)&part[g][4 * c] = a;
    __syncthreads();
    if (tid < D) {
        l = redl[0];
#pragma unroll
        for (int i = 1; i < kAsC / 64; ++i) l += redl[i];
        float r = part[0][tid];
#pragma unroll
        for (int i = 1; i < NG; ++i) r += part[i][tid];
        out[h * D + tid] = r * (1.0f / l);
    }
}

// query heads per workgroup: the largest of 8, 4, 2, 1 that divides the group
inline int as_hg(int heads, int kv_heads) {
    const int r = heads / kv_heads;
    return r % 8 == 0 ? 8 : r % 4 == 0 ? 4 : r % 2 == 0 ? 2 : 1;
}
struct AsPlan {
    int hg, nl, T, S;
    int64_t groups;  // (token, kv head, head group)
};
inline AsPlan as_plan(int64_t batch, int heads, int kv_heads, int D, int ctx) {
    AsPlan p{};
    p.hg = as_hg(heads, kv_heads);
    p.groups = batch * (heads / p.hg);
    // the most rows per lane in flight (16, 8, 4) that leave a workgroup per CU, and no more than kAsMaxS slices
    // (16384 positions of 256 are 256 slices of 64)
    const int t1 = 64 / (D / 4) * kAsW;
    for (p.nl = 16; p.nl > 4; p.nl /= 2) {
        const int half = (ctx + t1 * p.nl / 2 - 1) / (t1 * p.nl / 2);
        if (p.groups * ((ctx + t1 * p.nl - 1) / (t1 * p.nl)) >= 256 || half > kAsMaxS) break;
    }
    p.T = t1 * p.nl;
    p.S = (ctx + p.T - 1) / p.T;
    return p;
}

template <int D, int HG, int NL>
void as_run(const float* q, const float* kc, const float* vc, float* po, float* pml, const AsPlan& p, int ctx,
            int64_t batch, int heads, int kv_heads, int max_seq, hipStream_t s) {
    const dim3 grid((unsigned)p.S, (unsigned)(heads / HG), (unsigned)batch);
    attn_split_k<D, HG, NL><<<grid, 64 * kAsW, 0, s>>>(q, kc, vc, po, pml, ctx, heads, kv_heads, max_seq,
                                                      1.0f / sqrtf((float)D));
}
template <int D, int HG>
void as_nl(const float* q, const float* kc, const float* vc, float* po, float* pml, const AsPlan& p, int ctx,
           int64_t batch, int heads, int kv_heads, int max_seq, hipStream_t s) {
    if (p.nl == 16) as_run<D, HG, 16>(q, kc, vc, po, pml, p, ctx, batch, heads, kv_heads, max_seq, s);
    else if (p.nl == 8) as_run<D, HG, 8>(q, kc, vc, po, pml, p, ctx, batch, heads, kv_heads, max_seq, s);
    else as_run<D, HG, 4>(q, kc, vc, po, pml, p, ctx, batch, heads, kv_heads, max_seq, s);
}
template <int D>
void as_hgs(const float* q, const float* kc, const float* vc, float* po, float* pml, const AsPlan& p, int ctx,
            int64_t batch, int heads, int kv_heads, int max_seq, float* out, hipStream_t s) {
    switch (p.hg) {
        case 8: as_nl<D, 8>(q, kc, vc, po, pml, p, ctx, batch, heads, kv_heads, max_seq, s); break;
        case 4: as_nl<D, 4>(q, kc, vc, po, pml, p, ctx, batch, heads, kv_heads, max_seq, s); break;
        case 2: as_nl<D, 2>(q, kc, vc, po, pml, p, ctx, batch, heads, kv_heads, max_seq, s); break;
        default: as_nl<D, 1>(q, kc, vc, po, pml, p, ctx, batch, heads, kv_heads, max_seq, s); break;
    }
    attn_combine_k<D><<<(unsigned)(batch * heads), kAsC, 0, s>>>(po, pml, out, p.S);
}

}  // namespace

bool attention_split_supported(const float* q, const float* kc, const float* vc, int64_t batch, int heads,
                               int kv_heads, int head_dim, int ctx, int max_seq) {
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) return false;
    if ((((uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc) & 15u) != 0 || batch * heads >= (1ll << 31)) return false;
    // Two launches cost what 300 positions of 128 cost in the one-launch kernel (12 us eagerly; it took 8.8 us at
    // ctx * D = 25600, 12.4 at 38400, 12.8 .. 17 at 51200).  512 (token, head) workgroups fill the chip by themselves:
    // without shared K / V rows the split only adds its partial sums there (70.8 -> 75.7 us at 16 x 32 x 800 x 128; at
    // 128 workgroups 145 -> 138 us at 6000 positions), with them it pays from ctx * D = 80000 (17.5 -> 19.5 us at
    // 51200, 38.7 -> 31.9 at 102400).  Rows of 64 on the one-launch kernel's 16 waves (few workgroups, a cache of more
    // than 1024 positions): 10.9 .. 11.4 us there and 11.4 .. 12.1 split at 80640, 12.0 .. 12.9 and 11.0 .. 12.2 at 89600.
    const int64_t work = (int64_t)ctx * head_dim, wgs = batch * heads;
    const int hg = as_hg(heads, kv_heads);
    const bool waves16 = head_dim == 64 && max_seq > 1024 && wgs <= 128;
    if (work < (waves16 ? 88000 : wgs > 256 ? 80000 : 42000) || (hg == 1 && wgs > 160)) return false;
    return as_plan(batch, heads, kv_heads, head_dim, ctx).S > 1;
}

size_t attention_split_workspace_bytes(int64_t batch, int heads, int kv_heads, int head_dim, int ctx) {
    const AsPlan p = as_plan(batch, heads, kv_heads, head_dim, ctx);
    return (size_t)(batch * heads * p.S * (head_dim + 2)) * 4;
}

hipError_t launch_attention_split(const float* q, const float* kc, const float* vc, float* out, int ctx, int64_t batch,
                                  int heads, int kv_heads, int head_dim, int max_seq, void* ws, hipStream_t s) {
    const AsPlan p = as_plan(batch, heads, kv_heads, head_dim, ctx);
    float* po = (float*)ws;
    float* pml = po + batch * heads * p.S * head_dim;
    if (head_dim == 64) as_hgs<64>(q, kc, vc, po, pml, p, ctx, batch, heads, kv_heads, max_seq, out, s);
    else if (head_dim == 128) as_hgs<128>(q, kc, vc, po, pml, p, ctx, batch, heads, kv_heads, max_seq, out, s);
    else as_hgs<256>(q, kc, vc, po, pml, p, ctx, batch, heads, kv_heads, max_seq, out, s);
    return hipGetLastError();
}

}  // namespace mth

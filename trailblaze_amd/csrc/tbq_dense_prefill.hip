// tbq_dense_prefill.hip -- batched prefill of a dense Qwen3-style model on
// gfx950: the T prompt tokens at positions pos0 .. pos0 + T - 1 go through
// each layer together, where the reference prefills token by token
// (layer4/tb_infer.c:1068-1075: one tb_infer_decode step per prompt token).
//
// Per layer (x: fp32 residual rows [T][H]; h16: fp16 rows with per-row
// power-of-two scales, the GEMMs' activation operand; the GEMMs are
// k_hgemm_* (tbq_gemm.hip): Q4_K weights are dequantised inside them, any other
// format to fp16 first (k_dequant_f16, one reused buffer)):
//   k_pf_norm        x += y (the previous sublayer's output, unscaled by
//                    its row scales), h16 = rmsnorm(x) * attn_norm
//   GEMM             qkv = h16 Wqkv^T             fp16 MFMA, fp32 acc
//   k_pf_qk          per (token, head): QK-norm + RoPE of q (to qb) and k;
//                    k and v rows written to the cache at pos0 + t
//   k_pf_kv16        the layer's cache rows as fp16, V transposed
//   k_pf_attn        causal GQA attention over cache positions 0 .. pos on
//                    fp16 MFMA, online softmax, key ranges split over
//                    workgroups
//   k_pf_attn_rows   merges the splits of each token's row and writes it
//                    as fp16 rows with row scales (the o GEMM's operand)
//   GEMM             y = att Wo^T
//   k_pf_norm        x += y, h16 = rmsnorm(x) * ffn_norm
//   GEMM             a = silu(h16 Wg^T) * (h16 Wu^T) (SwiGLU in the GEMM's
//                    epilogue for a fused gate|up matrix; else the two
//                    products and k_pf_swiglu_f16), then a16 = fp16 rows
//                    with row scales
//   GEMM             y = a16 Wdown^T
// then the last token's logits = Wlm rmsnorm(x + y) (the decode step's
// lm_head matvec with its norm prologue).
//
// Accuracy: fp16 weights, activations, attention scores' operands and
// probabilities (11-bit mantissa) with fp32 accumulation, fp32 norms, RoPE
// and softmax; the logits land within
// 1e-2 relative L2 of the float64 sequential decode.

#include <algorithm>

#include "tbq_dma.hpp"
#include "tbq_kernels.h"
#include "tbq_device.hpp"
#include "../../include/tbq.h"

namespace tbq {

constexpr int PN_THREADS = 256;

// Slot swizzle of 128-byte LDS rows (eight 16-byte segments).
__device__ __forceinline__ int pf_swz8(int r) { return (r & 7) ^ ((r >> 3) & 1); }

__device__ __forceinline__ float pf_block_sum(float v, float *red) {
    v = group_sum<64>(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = 0.f;
#pragma unroll
    for (int i = 0; i < PN_THREADS / 64; i++) r += red[i];
    return r;
}

__device__ __forceinline__ float pf_block_max(float v, float *red) {
    v = wave_max(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = 0.f;
#pragma unroll
    for (int i = 0; i < PN_THREADS / 64; i++) r = fmaxf(r, red[i]);
    return r;
}

// Row t: v = x[t] + y[t] * ys[t] (y may be null; x[t] = v is stored back
// when y is not; ys, the row scales of a GEMM's fp16 operand, may be null
// for 1), h = v * rsqrt(mean(v^2) + eps) * w, then h16[t] = h * 2^s in fp16
// with s putting max |h| in [2^14, 2^15) and hinv[t] = 2^-s.  grid = T.
// y may be a GEMM's ny split-K slices (slice z at y + z * ystride), added
// here in slice order.  A thread holds up to PN_V float4 of the row (H <=
// 8192), all loaded before any is used.
constexpr int PN_V = 8, PN_MAXY = 8;   // float4 per thread (H <= 8192), slices of y
template <int PV>   // float4 of the row per thread: ceil(H / 4 / PN_THREADS) <= PV
__global__ __launch_bounds__(PN_THREADS) void k_pf_norm(float *__restrict__ x, const float *__restrict__ y, int ny,
                                                        long long ystride, const float *__restrict__ ys,
                                                        const float *__restrict__ w, int H, float eps,
                                                        _Float16 *__restrict__ h16, float *__restrict__ hinv) {
    __shared__ float red[PN_THREADS / 64];
    const int t = blockIdx.x, tid = threadIdx.x, n4 = H / 4;
    float4 *xr = reinterpret_cast<float4 *>(x + (long long)t * H);
    const float4 *yr = reinterpret_cast<const float4 *>(y ? y + (long long)t * H : x + (long long)t * H);
    const float4 *wr = reinterpret_cast<const float4 *>(w);
    float4 v[PV], b[PV], g[PV];
#pragma unroll
    for (int i = 0; i < PV; i++) {
        const int j = min(tid + PN_THREADS * i, n4 - 1);   // clamped: loads stay unconditional
        v[i] = xr[j];
        b[i] = yr[j];
        g[i] = wr[j];
    }
    if (y && ny > 1) {
        // every slice's loads issued at once (slices past ny re-read the
        // last and are not added), then added in slice order
        float4 c[PN_MAXY - 1][PV];
#pragma unroll
        for (int z = 1; z < PN_MAXY; z++) {
            const float4 *yz = yr + min(z, ny - 1) * (ystride / 4);
#pragma unroll
            for (int i = 0; i < PV; i++) c[z - 1][i] = yz[min(tid + PN_THREADS * i, n4 - 1)];
        }
#pragma unroll
        for (int z = 1; z < PN_MAXY; z++) {
            if (z < ny) {
#pragma unroll
                for (int i = 0; i < PV; i++) {
                    b[i].x = b[i].x + c[z - 1][i].x; b[i].y = b[i].y + c[z - 1][i].y;
                    b[i].z = b[i].z + c[z - 1][i].z; b[i].w = b[i].w + c[z - 1][i].w;
                }
            }
        }
    }
    float ss = 0.f;
    const float yscale = ys ? ys[t] : 1.f;
#pragma unroll
    for (int i = 0; i < PV; i++) {
        if (y) {
            v[i].x += b[i].x * yscale; v[i].y += b[i].y * yscale;
            v[i].z += b[i].z * yscale; v[i].w += b[i].w * yscale;
        }
        if (tid + PN_THREADS * i < n4) ss += v[i].x * v[i].x + v[i].y * v[i].y + v[i].z * v[i].z + v[i].w * v[i].w;
    }
    if (y) {
#pragma unroll
        for (int i = 0; i < PV; i++)
            if (tid + PN_THREADS * i < n4) xr[tid + PN_THREADS * i] = v[i];
    }
    ss = pf_block_sum(ss, red);
    const float r = 1.0f / sqrtf(ss / (float)H + eps);
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < PV; i++) {
        v[i].x = v[i].x * r * g[i].x; v[i].y = v[i].y * r * g[i].y;
        v[i].z = v[i].z * r * g[i].z; v[i].w = v[i].w * r * g[i].w;
        if (tid + PN_THREADS * i < n4)
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
    }
    mx = pf_block_max(mx, red);
    int e = 0;
    frexpf(mx, &e);
    int sh = mx > 0.f ? 15 - e : 0;
    sh = sh > 126 ? 126 : (sh < -126 ? -126 : sh);
    const float s = ldexpf(1.f, sh);
    uint2 *hr = reinterpret_cast<uint2 *>(h16 + (long long)t * H);
#pragma unroll
    for (int i = 0; i < PV; i++) {
        const int j = tid + PN_THREADS * i;
        if (j < n4) {
            const _Float16 a0 = (_Float16)(v[i].x * s), a1 = (_Float16)(v[i].y * s);
            const _Float16 a2 = (_Float16)(v[i].z * s), a3 = (_Float16)(v[i].w * s);
            hr[j] = make_uint2((uint32_t)__builtin_bit_cast(uint16_t, a0) | ((uint32_t)__builtin_bit_cast(uint16_t, a1) << 16),
                               (uint32_t)__builtin_bit_cast(uint16_t, a2) | ((uint32_t)__builtin_bit_cast(uint16_t, a3) << 16));
        }
    }
    if (tid == 0) hinv[t] = ldexpf(1.f, -sh);
}

static hipError_t launch_pf_norm(int T, float *x, const float *y, int ny, long long ystride, const float *ys,
                                 const float *w, int H, float eps, _Float16 *h16, float *hinv, hipStream_t st) {
    if (ny > PN_MAXY) return hipErrorNotSupported;
    const int pv = (H / 4 + PN_THREADS - 1) / PN_THREADS;
#define TBQ_PN(V)                                                                                                  \
    case V:                                                                                                        \
        hipLaunchKernelGGL(k_pf_norm<V>, dim3(T), dim3(PN_THREADS), 0, st, x, y, ny, ystride, ys, w, H, eps, h16,  \
                           hinv);                                                                                  \
        break;
    switch (pv) {
        TBQ_PN(1) TBQ_PN(2) TBQ_PN(3) TBQ_PN(4) TBQ_PN(5) TBQ_PN(6) TBQ_PN(7) TBQ_PN(8)
    default:
        return hipErrorNotSupported;
    }
#undef TBQ_PN
    return hipGetLastError();
}

// RoPE tables of the prompt's positions, shared by every layer: rc[t][j] =
// cos, rc[t][D/2 + j] = sin of (pos0 + t) * theta^(-2j/D), formed and
// reduced in fp64 exactly as the decode step's k_rope_table.  grid = T.
__global__ __launch_bounds__(64) void k_pf_rope(int pos0, float theta, int D, float *__restrict__ rc) {
    const int t = blockIdx.x, j = threadIdx.x;
    if (j < D / 2) {
        double sd, cd;
        sincos((double)(pos0 + t) * pow((double)theta, -2.0 * j / D), &sd, &cd);
        rc[(long long)t * D + j] = (float)cd;
        rc[(long long)t * D + D / 2 + j] = (float)sd;
    }
}

// grid = (T, ceil((NQ + NKV) / heads per workgroup)); D / 4 lanes per head,
// lane l of them holding elements 2l, 2l + 1 and D/2 + 2l, D/2 + 2l + 1 (the
// rotation's pairs are in one lane), four waves.  qkv row t times rs[t] is the
// true row.  Head hh < NQ: q head hh of token t, normed, rotated and scaled by
// log2(e) / sqrt(D) (the attention's softmax is in powers of two) into qb as
// fp16, the attention's operand; else k head hh - NQ, normed and rotated, and
// the matching v head, written to the layer's cache rows pos0 + t.  One wave
// per head in a workgroup of its own was bound by the workgroups' launch: T =
// 1999, 40 heads of 128: 22.0 -> 16.2 us.
constexpr int PQ_THREADS = 256;
template <int D>
__global__ __launch_bounds__(PQ_THREADS) void k_pf_qk(const float *__restrict__ qkv, int nq, long long qstride,
                                                      const float *__restrict__ rs, const float *__restrict__ qn,
                                                      const float *__restrict__ kn, int NQ, int NKV, int pos0,
                                                      const float *__restrict__ rope, float eps, float *__restrict__ kc,
                                                      float *__restrict__ vc, int max_ctx, _Float16 *__restrict__ qb) {
    constexpr int LPH = D / 4;
    const int t = blockIdx.x, l = threadIdx.x % LPH, h0 = blockIdx.y * (PQ_THREADS / LPH) + threadIdx.x / LPH;
    const bool on = h0 < NQ + NKV;
    const int hh = on ? h0 : NQ + NKV - 1;   // lanes past the last head repeat it and store nothing
    const int QKVR = (NQ + 2 * NKV) * D, pos = pos0 + t;
    const float sc = rs[t];   // row t of qkv is scaled by 1 / rs[t]
    // qkv may be a GEMM's nq split-K slices (slice z at qkv + z * qstride),
    // added in slice order
    auto elem = [&](long long off) {
        float2 a = *reinterpret_cast<const float2 *>(qkv + off);
        for (int z = 1; z < nq; z++) {
            const float2 b = *reinterpret_cast<const float2 *>(qkv + off + z * qstride);
            a.x = a.x + b.x;
            a.y = a.y + b.y;
        }
        return make_float2(a.x * sc, a.y * sc);
    };
    const long long src = (long long)t * QKVR + hh * D + 2 * l;
    float2 x = elem(src), y = elem(src + D / 2);
    const float *w = (hh < NQ ? qn : kn) + 2 * l;
    const float2 cs = *reinterpret_cast<const float2 *>(rope + (long long)t * D + 2 * l);
    const float2 sn = *reinterpret_cast<const float2 *>(rope + (long long)t * D + D / 2 + 2 * l);
    const float ss = group_sum<LPH>(x.x * x.x + x.y * x.y + y.x * y.x + y.y * y.y);
    const float r = 1.0f / sqrtf(ss / (float)D + eps);
    x.x = x.x * r * w[0];
    x.y = x.y * r * w[1];
    y.x = y.x * r * w[D / 2];
    y.y = y.y * r * w[D / 2 + 1];
    const float2 a = make_float2(x.x * cs.x - y.x * sn.x, x.y * cs.y - y.y * sn.y);
    const float2 b = make_float2(x.x * sn.x + y.x * cs.x, x.y * sn.y + y.y * cs.y);
    if (!on) return;
    if (hh < NQ) {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        const float scale = 1.4426950408889634f / sqrtf((float)D);
        h2 *q = reinterpret_cast<h2 *>(qb + ((long long)t * NQ + hh) * D + 2 * l);
        q[0] = h2{(_Float16)(a.x * scale), (_Float16)(a.y * scale)};
        q[D / 4] = h2{(_Float16)(b.x * scale), (_Float16)(b.y * scale)};
    } else {
        const int kvh = hh - NQ;
        const long long row = ((long long)kvh * max_ctx + pos) * D + 2 * l;
        const long long vsrc = (long long)t * QKVR + (NQ + NKV + kvh) * D + 2 * l;
        *reinterpret_cast<float2 *>(kc + row) = a;
        *reinterpret_cast<float2 *>(kc + row + D / 2) = b;
        *reinterpret_cast<float2 *>(vc + row) = elem(vsrc);
        *reinterpret_cast<float2 *>(vc + row + D / 2) = elem(vsrc + D / 2);
    }
}

// The layer's cache rows 0 .. kmax - 1 as the attention's fp16 operands, once
// per layer instead of once per query block: k16[kvh][pos][D], and vt[kvh][D]
// [pos], V transposed, its positions inside each group of 16 in the order 0-3,
// 8-11, 4-7, 12-15 (the order in which the probabilities sit in the
// accumulators).  Both have cp positions per head; rows past kmax up to the
// next multiple of 64 are zeros (their probabilities are 0, and 0 times a
// stale infinity is not).  grid = (NKV, ceil(kmax / 64)).
constexpr int PC_KC = 64;
template <int D>
__global__ __launch_bounds__(256) void k_pf_kv16(const float *__restrict__ kc, const float *__restrict__ vc,
                                                 int max_ctx, int kmax, int cp, _Float16 *__restrict__ k16,
                                                 _Float16 *__restrict__ vt) {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    const int kvh = blockIdx.x, c0 = blockIdx.y * PC_KC, tid = threadIdx.x;
    const float *kb = kc + (long long)kvh * max_ctx * D, *vb = vc + (long long)kvh * max_ctx * D;
#pragma unroll
    for (int i = 0; i < PC_KC * D / 4 / 256; i++) {
        const int f = tid + 256 * i, key = f / (D / 4), c4 = f % (D / 4), p = c0 + key;
        float4 v = *reinterpret_cast<const float4 *>(kb + (long long)min(p, kmax - 1) * D + 4 * c4);
        if (p >= kmax) v = make_float4(0.f, 0.f, 0.f, 0.f);
        *reinterpret_cast<h4 *>(k16 + ((long long)kvh * cp + p) * D + 4 * c4) =
            h4{(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
    }
    // thread = dim tid % D of NP positions
    constexpr int NP = PC_KC * D / 256;
    const int d = tid % D, p0 = c0 + NP * (tid / D);
    float v[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) {
        v[i] = vb[(long long)min(p0 + i, kmax - 1) * D + d];
        if (p0 + i >= kmax) v[i] = 0.f;
    }
    _Float16 *dst = vt + ((long long)kvh * D + d) * cp + p0;
#pragma unroll
    for (int i = 0; i < NP / 8; i++) {
        h8 o;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = (_Float16)v[16 * (i / 2) + 8 * (e / 4) + 4 * (i % 2) + e % 4];
        *reinterpret_cast<h8 *>(dst + 8 * i) = o;
    }
}

// Row t: a = silu(g * s) * (u * s) with gu[t] = [g (F) | u (F)] and s =
// gs[t], then a16[t] = a * 2^e in fp16 (max |a| in [2^14, 2^15)) and
// ainv[t] = 2^-e.  grid = T, 1024 threads, the row read once (up to PS_V
// float4 of g and of u per thread: F <= 16384).
constexpr int PS_THREADS = 1024, PS_V = 4;
__global__ __launch_bounds__(PS_THREADS) void k_pf_swiglu_f16(const float *__restrict__ gu, const float *__restrict__ gs,
                                                              int F, _Float16 *__restrict__ a16,
                                                              float *__restrict__ ainv) {
    __shared__ float red[PS_THREADS / 64];
    const int t = blockIdx.x, tid = threadIdx.x, n4 = F / 4;
    const float4 *g = reinterpret_cast<const float4 *>(gu + (long long)t * 2 * F), *u = g + n4;
    const float s = gs[t];
    float4 a[PS_V];
#pragma unroll
    for (int i = 0; i < PS_V; i++) {
        const int j = min(tid + PS_THREADS * i, n4 - 1);   // clamped: loads stay unconditional
        const float4 gv = g[j], uv = u[j];
        a[i] = make_float4(pro_swiglu(gv.x * s, uv.x * s), pro_swiglu(gv.y * s, uv.y * s),
                           pro_swiglu(gv.z * s, uv.z * s), pro_swiglu(gv.w * s, uv.w * s));
    }
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < PS_V; i++)
        if (tid + PS_THREADS * i < n4)
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(a[i].x), fabsf(a[i].y)), fmaxf(fabsf(a[i].z), fabsf(a[i].w))));
    mx = wave_max(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = 0.f;
#pragma unroll
    for (int i = 0; i < PS_THREADS / 64; i++) mx = fmaxf(mx, red[i]);
    int e = 0;
    frexpf(mx, &e);
    int sh = mx > 0.f ? 15 - e : 0;
    sh = sh > 126 ? 126 : (sh < -126 ? -126 : sh);
    const float sc = ldexpf(1.f, sh);
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    h4 *ar = reinterpret_cast<h4 *>(a16 + (long long)t * F);
#pragma unroll
    for (int i = 0; i < PS_V; i++) {
        const int j = tid + PS_THREADS * i;
        if (j < n4)
            ar[j] = h4{(_Float16)(a[i].x * sc), (_Float16)(a[i].y * sc), (_Float16)(a[i].z * sc),
                       (_Float16)(a[i].w * sc)};
    }
    if (tid == 0) ainv[t] = ldexpf(1.f, -sh);
}

// out[j] = (sum over the ny slices, in slice order, of y[z * ystride + j])
// * ys[0] for one row of n floats (the last token's down output before the
// lm_head).  One element per thread: one workgroup looping over the row took
// 11.7 us for 2560 floats of 5 slices, a chain of dependent trips.
__global__ __launch_bounds__(64) void k_pf_scale_row(const float *__restrict__ y, int ny, long long ystride,
                                                     const float *__restrict__ ys, int n, float *__restrict__ out) {
    const int j = blockIdx.x * 64 + threadIdx.x;
    if (j >= n) return;
    float v[PN_MAXY];
#pragma unroll
    for (int z = 0; z < PN_MAXY; z++) v[z] = y[min(z, ny - 1) * ystride + j];   // past ny: the last again, not added
    float a = v[0];
#pragma unroll
    for (int z = 1; z < PN_MAXY; z++)
        if (z < ny) a = a + v[z];
    out[j] = a * ys[0];
}

// Causal attention on MFMA (v_mfma_f32_32x32x16_f16, fp16 operands, fp32
// accumulate).  grid = (NKV, ceil(T / QB), nsplit), WV waves: the workgroup
// owns QB = 32 WV / G tokens x the G query heads of kv head kvh = 32 WV query
// columns, 32 per wave (query c of a wave: token c / G, head c % G).  K and V
// pass through LDS 64 positions at a time in fp16 (k_pf_kv16's form), copied
// directly from global memory a chunk ahead into one of two stages; the
// 16-byte segments of a row are XOR-swizzled by the copies' source addresses.
// Per chunk a wave forms S^T = K Q^T (64 positions x its 32 queries), so a
// lane holds 32 scores of one query: lane l, block b, register r: query l %
// 32, position 32 b + 8(r/4) + 4(l/32) + r%4.  The query's max needs one
// exchange with lane l ^ 32.  The probabilities, rounded to fp16, are already
// the B operand of O^T += V^T P^T when the 16 positions of a step are taken in
// the order k-slot 8h + i <-> position 8(i/4) + 4h + i%4 (h = l / 32), in which
// vt stores them; O^T's accumulators hold dims 32j + 8(r/4) + 4h + r%4 of the
// lane's query.
//
// Online softmax in powers of two.  The running max m is exact, so the position
// that holds it has p = 1 and no rounding of its weight; the output is rescaled
// in the chunks in which the max of some query of the wave rises.  Raising m
// only past a margin of 2^8 spares most rescalings (0.7% of a 1999-token prompt)
// but rounds the largest weights: the attention's error against 64 bits grew by
// 3 to 4%, the next layer's K and V rows' by 0.3%.  Only chunks that reach past a query's own position are masked.  m
// starts at a large negative number rather than -inf, so a chunk without a
// visible position gives p = 0.
//
// Workgroup i runs on XCD i % 8: with kv heads along x an XCD's L2 holds the K
// and V of NKV / 8 heads.  The query blocks that see most positions start
// first.
//
// Key splits: split z takes positions [z ks, (z + 1) ks) (ks a multiple of
// 64), so the heavy blocks of a causal prompt (whose queries see every earlier
// position) spread over several workgroups.  With nsplit > 1 each writes its
// queries' unnormalised output, running max and denominator to the record
// part[(row * nsplit + z) * pf_rec(D)] (D outputs, max, denominator, two
// floats of padding so that every record starts 16-byte aligned for the float4
// stores), and k_pf_attn_rows merges the splits a row reaches.
//
// Bound by the softmax's VALU work beside the MFMAs.  T = 1999 after 1024
// cached positions, 32 / 8 heads of 128: 293 -> 99 us (0.65 PFLOP/s), T = 512
// from position 0: 25.2 -> 14 to 16 us, against converting the fp32 cache rows in
// every query block, 32 positions at a time between two barriers (and 5 to 11
// us of k_pf_kv16, which that form did without).  Two workgroups of 4 waves
// per CU; 8 waves (half the copies, one workgroup per CU) were 1% slower on the
// whole prefill.
constexpr int PM_KC = PC_KC;
__host__ __device__ constexpr int pf_rec(int D) { return D + 4; }
typedef _Float16 pm_h8 __attribute__((ext_vector_type(8)));
typedef float pm_f16 __attribute__((ext_vector_type(16)));

template <int D>
struct PmLds {
    unsigned char k[2][PM_KC * D * 2];   // [position][dim]
    unsigned char v[2][D * PM_KC * 2];   // [dim][position]
};

template <int D, int G, int WV>
__global__ __launch_bounds__(64 * WV) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_pf_attn(
    const _Float16 *__restrict__ qb, const _Float16 *__restrict__ k16, const _Float16 *__restrict__ vt, int T, int pos0,
    int NQ, int cp, int ks, int nsplit, float *__restrict__ part, float *__restrict__ out) {
    constexpr int QB = 32 * WV / G, NT = D / 32, NS = D / 16, KSEG = D / 8;
    extern __shared__ __attribute__((aligned(1024))) unsigned char pm_lds[];
    PmLds<D> *st = reinterpret_cast<PmLds<D> *>(pm_lds);
    const int kvh = blockIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63,
              li = lane & 31, h = lane >> 5;
    const int yb = gridDim.y - 1 - blockIdx.y;
    const int qc = wave * 32 + li, g = qc % G;
    const int t = yb * QB + qc / G;
    const int tt = min(t, T - 1), qpos = pos0 + tt;
    const int k0 = blockIdx.z * ks;                              // this split's positions k0 .. kend - 1
    const int kend = min(pos0 + min(T, (yb + 1) * QB), k0 + ks);
    if (k0 >= kend) return;   // no position of the split is seen by the block (uniform)
    // the wave's first and last query positions
    const int qlo = pos0 + min(yb * QB + wave * 32 / G, T - 1), qhi = pos0 + min(yb * QB + (wave * 32 + 31) / G, T - 1);
    // Q^T's B fragments: dim step s, lane half h supplies dims 16s + 8h .. + 8
    pm_h8 qf[NS];
    const _Float16 *qsrc = qb + ((long long)tt * NQ + kvh * G + g) * D + 8 * h;
#pragma unroll
    for (int s = 0; s < NS; s++) qf[s] = *reinterpret_cast<const pm_h8 *>(qsrc + 16 * s);
    // copies: KC of K rows (KSEG segments), VC of V rows (8 segments), dealt to the waves
    constexpr int NC = PM_KC * KSEG / 64, CPW = NC / WV;
    static_assert(NC % WV == 0 && D * 8 / 64 == NC, "K and V take the same number of copies");
    const dma_rsrc_t kr = dma_rsrc(k16 + (long long)kvh * cp * D, (uint32_t)((long long)cp * D * 2));
    const dma_rsrc_t vr = dma_rsrc(vt + (long long)kvh * cp * D, (uint32_t)((long long)cp * D * 2));
    auto kswz = [](int row) { return KSEG == 16 ? row & 15 : pf_swz8(row); };
    uint32_t ko[CPW], vo[CPW];
#pragma unroll
    for (int i = 0; i < CPW; i++) {
        const int c = wave + WV * i;
        const int kr_ = c * (64 / KSEG) + lane / KSEG, vr_ = 8 * c + (lane >> 3);
        ko[i] = (uint32_t)(kr_ * D * 2 + 16 * ((lane % KSEG) ^ kswz(kr_)));
        vo[i] = (uint32_t)vr_ * (uint32_t)(cp * 2) + 16u * ((lane & 7) ^ pf_swz8(vr_));
    }
    const uint32_t lk = lds_addr(st->k[0]), lv = lds_addr(st->v[0]);
    auto copy = [&](int buf, int c0) {
#pragma unroll
        for (int i = 0; i < CPW; i++) {
            dma16(lk + buf * (PM_KC * D * 2) + (wave + WV * i) * 1024, ko[i], kr, (uint32_t)c0 * (D * 2));
            dma16(lv + buf * (PM_KC * D * 2) + (wave + WV * i) * 1024, vo[i], vr, (uint32_t)c0 * 2);
        }
    };
    pm_f16 o[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) o[j] = pm_f16{};
    float m = -1e30f, l = 0.f;
    const int ksw = kswz(li), vsw = pf_swz8(li);
    copy(0, k0);
    dma_wait_barrier();
    int buf = 0;
    for (int c0 = k0; c0 < kend; c0 += PM_KC, buf ^= 1) {
        copy(buf ^ 1, c0 + PM_KC < kend ? c0 + PM_KC : c0);   // the last chunk copies itself again, never read
        // V past the block's last query is made zero (past the prompt it is
        // already): its p is 0, and 0 times an infinity or NaN of a later token is not
        if (c0 + PM_KC > kend && kend < pos0 + T) {   // uniform
#pragma unroll
            for (int i = 0; i < D * 8 / (64 * WV); i++) {
                const int f = threadIdx.x + 64 * WV * i, row = f >> 3, seg = f & 7;
                pm_h8 *p = reinterpret_cast<pm_h8 *>(st->v[buf] + row * (PM_KC * 2) + 16 * (seg ^ pf_swz8(row)));
                pm_h8 v = *p;
#pragma unroll
                for (int e = 0; e < 8; e++)   // k_pf_kv16's order of the positions
                    v[e] = c0 + 16 * (seg / 2) + 4 * (seg % 2) + 8 * (e / 4) + e % 4 < kend ? v[e] : (_Float16)0.f;
                *p = v;
            }
            __syncthreads();
        }
        if (c0 <= qhi) {   // uniform per wave
            const unsigned char *Kb = st->k[buf] + li * (D * 2), *Vb = st->v[buf] + li * (PM_KC * 2);
            pm_f16 sc[2] = {pm_f16{}, pm_f16{}};
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    const pm_h8 a = *reinterpret_cast<const pm_h8 *>(Kb + b * (32 * D * 2) + 16 * ((2 * s + h) ^ ksw));
                    sc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[s], sc[b], 0, 0, 0);
                }
            if (c0 + PM_KC - 1 > qlo) {
#pragma unroll
                for (int b = 0; b < 2; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int key = c0 + 32 * b + 8 * (r / 4) + 4 * h + r % 4;
                        sc[b][r] = key <= qpos ? sc[b][r] : -__builtin_huge_valf();
                    }
            }
            float mx = sc[0][0];
#pragma unroll
            for (int r = 1; r < 32; r++) mx = fmaxf(mx, sc[r / 16][r % 16]);
            mx = swap32_max(mx);
            if (__builtin_amdgcn_ballot_w64(mx > m)) {
                const float mn = fmaxf(m, mx), corr = __builtin_amdgcn_exp2f(m - mn);
                m = mn;
                l *= corr;
#pragma unroll
                for (int j = 0; j < NT; j++) o[j] *= corr;
            }
            pm_h8 pb[4];
            float ls = 0.f;
#pragma unroll
            for (int r = 0; r < 32; r++) {
                const float p = __builtin_amdgcn_exp2f(sc[r / 16][r % 16] - m);
                ls += p;
                pb[r / 8][r % 8] = (_Float16)p;
            }
            l += ls;   // this half's positions; the halves are added at the end
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    const pm_h8 a = *reinterpret_cast<const pm_h8 *>(Vb + j * (32 * PM_KC * 2) + 16 * ((2 * u + h) ^ vsw));
                    o[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pb[u], o[j], 0, 0, 0);
                }
        }
        dma_wait_barrier();
    }
    l = swap32_sum(l);
    if (t >= T) return;
    const long long row = (long long)t * NQ + kvh * G + g;
    const float inv = nsplit == 1 ? 1.0f / l : 1.f;
    float *dst = nsplit == 1 ? out + row * D : part + (row * nsplit + blockIdx.z) * pf_rec(D);
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++)
            *reinterpret_cast<float4 *>(dst + 32 * j + 8 * r4 + 4 * h) =
                make_float4(o[j][4 * r4] * inv, o[j][4 * r4 + 1] * inv, o[j][4 * r4 + 2] * inv, o[j][4 * r4 + 3] * inv);
    if (nsplit > 1 && h == 0) {
        dst[D] = m;
        dst[D + 1] = l;
    }
}

// Attention rows to the o GEMM's operand in one pass: row t (all NQ heads,
// QD = NQ * D floats) is the attention output -- att[t] itself when the
// keys were not split, else the merge of the splits z <= (pos0 + t) / ks (at
// most NZ) with 2^(m_z - M) weights and fmaf sums in z order -- and is written as fp16 scaled by
// the power of two that puts its max |value| in [2^14, 2^15), with
// hinv[t] = the inverse scale (k_rows_f16's arithmetic).  grid = T,
// PN_THREADS threads, up to PR_V float4 of the row per thread (QD <= 8192).
constexpr int PR_V = 8;
constexpr int PA_MIN_KS = 128, PA_MAX_SPLIT = 8;   // smallest split size, most splits
template <int D, int NZ>
__global__ __launch_bounds__(PN_THREADS) void k_pf_attn_rows(const float *__restrict__ part,
                                                             const float *__restrict__ att, int NQ, int pos0, int ks,
                                                             int nsplit, _Float16 *__restrict__ h16,
                                                             float *__restrict__ hinv) {
    __shared__ float red[PN_THREADS / 64];
    constexpr int RS = pf_rec(D);
    const int t = blockIdx.x, tid = threadIdx.x, n4 = NQ * D / 4;
    const int nz = (pos0 + t) / ks + 1;
    float4 v[PR_V];
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < PR_V; i++) {
        const int j = tid + PN_THREADS * i;
        if (j >= n4) continue;
        const int hh = 4 * j / D, d = 4 * j % D;
        const long long row = (long long)t * NQ + hh;
        if constexpr (NZ == 1) {
            v[i] = *reinterpret_cast<const float4 *>(att + row * D + d);
        } else {
            // every split's record loaded at once (splits past nz re-read the
            // last one and are skipped), then merged in z order
            const float *p = part + row * nsplit * RS;
            float ml[NZ], ll[NZ];
            float4 o[NZ];
#pragma unroll
            for (int z = 0; z < NZ; z++) {
                const float *r = p + min(z, nz - 1) * RS;
                ml[z] = r[D];
                ll[z] = r[D + 1];
                o[z] = *reinterpret_cast<const float4 *>(r + d);
            }
            float M = -__builtin_huge_valf();
#pragma unroll
            for (int z = 0; z < NZ; z++)
                if (z < nz) M = fmaxf(M, ml[z]);
            float n0 = 0.f, n1 = 0.f, n2 = 0.f, n3 = 0.f, den = 0.f;
#pragma unroll
            for (int z = 0; z < NZ; z++) {
                if (z < nz) {
                    const float f = __builtin_amdgcn_exp2f(ml[z] - M);
                    n0 = fmaf(f, o[z].x, n0);
                    n1 = fmaf(f, o[z].y, n1);
                    n2 = fmaf(f, o[z].z, n2);
                    n3 = fmaf(f, o[z].w, n3);
                    den = fmaf(f, ll[z], den);
                }
            }
            v[i] = make_float4(n0 / den, n1 / den, n2 / den, n3 / den);
        }
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
    }
    mx = pf_block_max(mx, red);
    int e = 0;
    frexpf(mx, &e);
    int sh = mx > 0.f ? 15 - e : 0;
    sh = sh > 126 ? 126 : (sh < -126 ? -126 : sh);
    const float sc = ldexpf(1.f, sh);
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    h4 *hr = reinterpret_cast<h4 *>(h16 + (long long)t * NQ * D);
#pragma unroll
    for (int i = 0; i < PR_V; i++) {
        const int j = tid + PN_THREADS * i;
        if (j < n4)
            hr[j] = h4{(_Float16)(v[i].x * sc), (_Float16)(v[i].y * sc), (_Float16)(v[i].z * sc),
                       (_Float16)(v[i].w * sc)};
    }
    if (tid == 0) hinv[t] = ldexpf(1.f, -sh);
}

// Splits of the positions: as few as give every CU about two workgroups' worth
// of waves (the partial records are written and read once per split), of at
// least PA_MIN_KS positions, a multiple of the chunk.
static int pf_split_size(int kmax, int wgs, int n_cu) {
    int n = std::max(1, std::min(PA_MAX_SPLIT, (2 * n_cu + wgs - 1) / wgs));
    n = std::min(n, (kmax + PA_MIN_KS - 1) / PA_MIN_KS);
    return ((kmax + n - 1) / n + PM_KC - 1) / PM_KC * PM_KC;
}

template <int D, int G, int WV>
static hipError_t launch_pf_attn_g(const _Float16 *qb, const _Float16 *k16, const _Float16 *vt, int T, int pos0, int NQ,
                                   int NKV, int cp, int ks, int nsplit, float *part, float *out, hipStream_t st) {
    constexpr int QB = 32 * WV / G;
    static const hipError_t a = hipFuncSetAttribute((const void *)k_pf_attn<D, G, WV>,
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(PmLds<D>));
    if (a != hipSuccess) return a;
    hipLaunchKernelGGL((k_pf_attn<D, G, WV>), dim3(NKV, (T + QB - 1) / QB, nsplit), dim3(64 * WV), sizeof(PmLds<D>), st,
                       qb, k16, vt, T, pos0, NQ, cp, ks, nsplit, part, out);
    return hipGetLastError();
}

constexpr int PA_WV = 4;   // waves per attention workgroup
template <int D>
static hipError_t launch_pf_attn(int G, const _Float16 *qb, const float *kc, const float *vc, int T, int pos0, int NQ,
                                 int NKV, int max_ctx, _Float16 *k16, _Float16 *vt, int cp, float *part, float *out,
                                 _Float16 *h16, float *hinv, int n_cu, hipStream_t st) {
    const int kmax = pos0 + T, qb_tokens = 32 * PA_WV / G;
    hipLaunchKernelGGL(k_pf_kv16<D>, dim3(NKV, (kmax + PC_KC - 1) / PC_KC), dim3(256), 0, st, kc, vc, max_ctx, kmax, cp,
                       k16, vt);
    const int ks = pf_split_size(kmax, NKV * ((T + qb_tokens - 1) / qb_tokens), n_cu), nsplit = (kmax + ks - 1) / ks;
    hipError_t err;
    switch (G) {
    case 1: err = launch_pf_attn_g<D, 1, PA_WV>(qb, k16, vt, T, pos0, NQ, NKV, cp, ks, nsplit, part, out, st); break;
    case 2: err = launch_pf_attn_g<D, 2, PA_WV>(qb, k16, vt, T, pos0, NQ, NKV, cp, ks, nsplit, part, out, st); break;
    case 4: err = launch_pf_attn_g<D, 4, PA_WV>(qb, k16, vt, T, pos0, NQ, NKV, cp, ks, nsplit, part, out, st); break;
    case 8: err = launch_pf_attn_g<D, 8, PA_WV>(qb, k16, vt, T, pos0, NQ, NKV, cp, ks, nsplit, part, out, st); break;
    default: return hipErrorNotSupported;
    }
    if (err != hipSuccess) return err;
#define TBQ_PFR(NZ)                                                                                                 \
    hipLaunchKernelGGL((k_pf_attn_rows<D, NZ>), dim3(T), dim3(PN_THREADS), 0, st, part, out, NQ, pos0, ks, nsplit, \
                       h16, hinv)
    if (nsplit == 1) TBQ_PFR(1);
    else if (nsplit == 2) TBQ_PFR(2);
    else if (nsplit <= 4) TBQ_PFR(4);
    else TBQ_PFR(8);
#undef TBQ_PFR
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
static size_t pf_up(size_t n) { return (n + 255) & ~(size_t)255; }

// Every model with hidden <= 8192, n_heads * head_dim <= 8192 and ffn <=
// 16384 (the rows the norm, attention-row and SwiGLU kernels hold) takes the batched path for T >= 2.  Q4_K matrices go
// straight into the GEMM (dequantised in its registers); every other
// format and layout is dequantised to fp16 first (one matrix at a time) and
// multiplied by the same GEMM.
bool dense_prefill_batched(const tbq_dense_model *m) {
    return m->hidden <= PN_THREADS * PN_V * 4 && m->ffn <= PS_THREADS * PS_V * 4 &&
           m->n_heads * m->head_dim <= PN_THREADS * PR_V * 4;
}

struct PfWs {
    float *x, *y, *qkv, *att, *gu, *sa, *sb, *part, *rope, *gpart;
    _Float16 *h16, *wh, *qb, *k16, *vt;
    size_t gpart_bytes;
    int cp;   // positions per head of k16 and vt
    int *tok;
    void *dec;
};

// *total: the bytes used, without gpart's, which is what the caller's ws_bytes leave.
static PfWs pf_ws(const tbq_dense_model *m, int T, void *ws, size_t ws_bytes, size_t *total) {
    const size_t H = m->hidden, QD = (size_t)m->n_heads * m->head_dim, F = m->ffn;
    const size_t QKVR = (size_t)(m->n_heads + 2 * m->n_kv_heads) * m->head_dim;
    const size_t wide = std::max(std::max(H, QD), F);
    const size_t wmax = std::max(std::max(QKVR * H, H * QD), std::max(2 * F * H, H * F));
    char *p = (char *)ws;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        void *r = p + off;
        off += pf_up(bytes);
        return r;
    };
    PfWs w{};
    w.dec = take(dense_workspace_bytes(m));
    w.tok = (int *)take((size_t)T * 4);
    if (dense_prefill_batched(m) && T >= 2) {
        w.x = (float *)take((size_t)T * H * 4);
        w.y = (float *)take((size_t)T * H * 4);
        w.qkv = (float *)take((size_t)T * QKVR * 4);
        w.qb = (_Float16 *)take((size_t)T * QD * 2);
        // fp16 K and V of one layer (a prefill reaches position kmax - 1 < max_ctx)
        w.cp = (m->max_ctx + PC_KC - 1) / PC_KC * PC_KC;
        w.k16 = (_Float16 *)take((size_t)m->n_kv_heads * w.cp * m->head_dim * 2);
        w.vt = (_Float16 *)take((size_t)m->n_kv_heads * w.cp * m->head_dim * 2);
        w.att = (float *)take((size_t)T * QD * 4);
        w.gu = (float *)take((size_t)T * 2 * F * 4);
        w.h16 = (_Float16 *)take((size_t)T * wide * 2);
        w.sa = (float *)take((size_t)T * 4);
        w.sb = (float *)take((size_t)T * 4);
        w.wh = (_Float16 *)take(wmax * 2);
        w.rope = (float *)take((size_t)T * m->head_dim * 4);
        // attention split partials: a prefill reaching position kmax - 1 uses
        // at most min(PA_MAX_SPLIT, ceil(kmax / PA_MIN_KS)) splits, and kmax <= max_ctx
        const int ns = std::min(PA_MAX_SPLIT, (m->max_ctx + PA_MIN_KS - 1) / PA_MIN_KS);
        w.part = ns > 1 ? (float *)take((size_t)T * m->n_heads * ns * pf_rec(m->head_dim) * 4) : nullptr;
        // a product's split-K partials until their consumer has added them.  (A
        // region of their own: with the attention's records in the same memory a
        // prefill of 200 tokens took 250 us instead of 241)
        w.gpart_bytes = ws_bytes > off ? ws_bytes - off : 0;
        w.gpart = w.gpart_bytes ? (float *)(p + off) : nullptr;
    }
    if (total) *total = off;
    return w;
}

size_t dense_prefill_workspace_min(const tbq_dense_model *m, int T) {
    size_t t = 0;
    pf_ws(m, T, nullptr, 0, &t);
    return t;
}

// With room for the partial sums of the products that split K (a gate|up
// matrix's does not) at any T up to this one: never less for a larger T.
size_t dense_prefill_workspace_bytes(const tbq_dense_model *m, int T) {
    const size_t base = dense_prefill_workspace_min(m, T);
    if (!dense_prefill_batched(m) || T < 2) return base;
    const int H = m->hidden, QD = m->n_heads * m->head_dim, KD = m->n_kv_heads * m->head_dim, F = m->ffn, cu = hgemm_cus();
    bool qkv = false, q_k_v = false, gate_up = false;
    for (int l = 0; l < m->n_layers; l++) {
        (m->layers[l].wqkv ? qkv : q_k_v) = true;
        gate_up = gate_up || !m->layers[l].wgu;
    }
    size_t gp = std::max(hgemm_partial_upto(T, H, QD, cu), hgemm_partial_upto(T, H, F, cu));
    if (qkv) gp = std::max(gp, hgemm_partial_upto(T, QD + 2 * KD, H, cu));
    if (q_k_v) gp = std::max(gp, std::max(hgemm_partial_upto(T, QD, H, cu), hgemm_partial_upto(T, KD, H, cu)));
    if (gate_up) gp = std::max(gp, hgemm_partial_upto(T, F, H, cu));
    return base + gp;
}

// tokens: T device ints (in range); T >= 2.
static hipError_t pf_batched(const tbq_dense_model *m, const PfWs &w, int T, int pos0, float *logits,
                             hipStream_t st) {
    const int H = m->hidden, D = m->head_dim, NQ = m->n_heads, NKV = m->n_kv_heads, G = NQ / NKV, F = m->ffn;
    const int QD = NQ * D, KD = NKV * D, QKVR = QD + 2 * KD;
    auto qt_of = [m](int q) { return canon_qt(q ? q : m->qtype_layers); };
    const int cu = hgemm_cus();
    // C[T][rows] (row stride ldc) = h16 . W^T: Q4_K rows directly, any other
    // format through its fp16 form in wh
    // (with ns set, the K slices' partial sums stay in w.gpart for the
    // consumer to add: k_pf_qk, k_pf_norm and k_pf_scale_row take them)
    auto gemm = [&](int qt, const void *W, int rows, int K, float *C, int ldc, int *ns = nullptr) {
        if (qt == QT_Q4_K) return launch_hgemm(QT_Q4_K, W, w.h16, T, rows, K, C, ldc, w.gpart, w.gpart_bytes, cu, st, ns);
        const hipError_t e = launch_dequant_f16(qt, W, (long long)rows * K, w.wh, st);
        if (e != hipSuccess) return e;
        return launch_hgemm(QT_F16, w.wh, w.h16, T, rows, K, C, ldc, w.gpart, w.gpart_bytes, cu, st, ns);
    };
    const float *ysrc = w.y;   // the previous sublayer's output, as yns slices
    int yns = 1;
    hipLaunchKernelGGL(k_pf_rope, dim3(T), dim3(64), 0, st, pos0, m->rope_theta, D, w.rope);
    hipError_t err = launch_dequant_rows(canon_qt(m->qtype_embd), m->tok_embd, w.tok, T, H, w.x, st);
    for (int l = 0; l < m->n_layers && err == hipSuccess; l++) {
        const tbq_dense_layer &L = m->layers[l];
        const size_t kvoff = (size_t)l * NKV * m->max_ctx * D;
        float *kc = m->k_cache + kvoff, *vc = m->v_cache + kvoff;
        err = launch_pf_norm(T, w.x, l ? ysrc : nullptr, yns, (long long)T * H, l ? w.sb : nullptr, L.attn_norm, H,
                             m->norm_eps, w.h16, w.sa, st);
        if (err != hipSuccess) break;
        int qns = 1;
        if (L.wqkv) {
            err = gemm(qt_of(L.qt_qkv), L.wqkv, QKVR, H, w.qkv, QKVR, &qns);
        } else {
            err = gemm(qt_of(L.qt_q), L.wq, QD, H, w.qkv, QKVR);
            if (err == hipSuccess) err = gemm(qt_of(L.qt_k), L.wk, KD, H, w.qkv + QD, QKVR);
            if (err == hipSuccess) err = gemm(qt_of(L.qt_v), L.wv, KD, H, w.qkv + QD + KD, QKVR);
        }
        if (err != hipSuccess) break;
        const float *qsrc = qns > 1 ? w.gpart : w.qkv;
        if (D == 128) {
            hipLaunchKernelGGL(k_pf_qk<128>, dim3(T, (NQ + NKV + 7) / 8), dim3(PQ_THREADS), 0, st, qsrc, qns,
                               (long long)T * QKVR, w.sa, L.q_norm, L.k_norm, NQ, NKV, pos0, w.rope, m->norm_eps, kc,
                               vc, m->max_ctx, w.qb);
            err = launch_pf_attn<128>(G, w.qb, kc, vc, T, pos0, NQ, NKV, m->max_ctx, w.k16, w.vt, w.cp, w.part, w.att,
                                     w.h16, w.sb, cu, st);
        } else {
            hipLaunchKernelGGL(k_pf_qk<64>, dim3(T, (NQ + NKV + 15) / 16), dim3(PQ_THREADS), 0, st, qsrc, qns,
                               (long long)T * QKVR, w.sa, L.q_norm, L.k_norm, NQ, NKV, pos0, w.rope, m->norm_eps, kc,
                               vc, m->max_ctx, w.qb);
            err = launch_pf_attn<64>(G, w.qb, kc, vc, T, pos0, NQ, NKV, m->max_ctx, w.k16, w.vt, w.cp, w.part, w.att,
                                     w.h16, w.sb, cu, st);
        }
        if (err != hipSuccess) break;
        if ((err = gemm(qt_of(L.qt_o), L.wo, H, QD, w.y, H, &yns)) != hipSuccess) break;
        ysrc = yns > 1 ? w.gpart : w.y;
        if ((err = launch_pf_norm(T, w.x, ysrc, yns, (long long)T * H, w.sb, L.ffn_norm, H, m->norm_eps, w.h16,
                                  w.sa, st)) != hipSuccess)
            break;
        // a fused gate|up matrix: SwiGLU in the GEMM's epilogue, then the
        // activation rows to fp16; otherwise the gate and up products and
        // k_pf_swiglu_f16
        if (L.wgu) {
            const int qt = qt_of(L.qt_gu);
            const void *Wg = L.wgu;
            if (qt != QT_Q4_K && (err = launch_dequant_f16(qt, L.wgu, (long long)2 * F * H, w.wh, st)) != hipSuccess)
                break;
            if (qt != QT_Q4_K) Wg = w.wh;
            err = launch_hgemm_glu(qt == QT_Q4_K ? QT_Q4_K : QT_F16, Wg, w.h16, w.sa, T, F, H, w.gu, F, cu, st);
            if (err == hipSuccess) err = launch_rows_f16(w.gu, T, F, w.h16, w.sb, st);
        } else {
            err = gemm(qt_of(L.qt_gate), L.wgate, F, H, w.gu, 2 * F);
            if (err == hipSuccess) err = gemm(qt_of(L.qt_up), L.wup, F, H, w.gu + F, 2 * F);
            if (err != hipSuccess) break;
            hipLaunchKernelGGL(k_pf_swiglu_f16, dim3(T), dim3(PS_THREADS), 0, st, w.gu, w.sa, F, w.h16, w.sb);
        }
        if (err != hipSuccess) break;
        err = gemm(qt_of(L.qt_down), L.wdown, H, F, w.y, H, &yns);
        ysrc = yns > 1 ? w.gpart : w.y;
    }
    if (err != hipSuccess) return err;
    float *ylast = w.y + (size_t)(T - 1) * H;
    hipLaunchKernelGGL(k_pf_scale_row, dim3((H + 63) / 64), dim3(64), 0, st, ysrc + (size_t)(T - 1) * H, yns, (long long)T * H,
                       w.sb + (T - 1), H, ylast);
    if ((err = hipGetLastError()) != hipSuccess) return err;
    return dense_final_logits(m, w.x + (size_t)(T - 1) * H, ylast, logits, w.dec, st);
}

hipError_t launch_dense_prefill(const tbq_dense_model *m, const int *tokens_host, int T, int pos0, float *logits,
                                void *ws, size_t ws_bytes, hipStream_t st) {
    const PfWs w = pf_ws(m, T, ws, ws_bytes, nullptr);
    if (!dense_prefill_batched(m) || T < 2) {
        // one token, or a row wider than the norm kernel: the decode step per token
        for (int t = 0; t < T; t++) {
            const hipError_t err = launch_dense_decode(m, tokens_host[t], pos0 + t, logits, w.dec, st);
            if (err != hipSuccess) return err;
        }
        return hipSuccess;
    }
    const hipError_t err = hipMemcpyAsync(w.tok, tokens_host, (size_t)T * 4, hipMemcpyHostToDevice, st);
    if (err != hipSuccess) return err;
    return pf_batched(m, w, T, pos0, logits, st);
}

}  // namespace tbq

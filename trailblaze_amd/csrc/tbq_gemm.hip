// tbq_gemm.hip -- the batched prefill's weight products on gfx950:
//
//   C[T][N] = X[T][K] . W[N][K]^T      X fp16 rows (a power-of-two scale per
//                                      row, undone by the consumer), W fp16
//                                      rows or Q4_K rows, fp32 accumulate and
//                                      output
//
// Both kernels own a tile of weight rows x tokens in blocks of
// v_mfma_f32_32x32x16_f16 (A = 32 weight rows x 16 k, B = 16 k x 32 tokens),
// advance K by 64 columns a step, and bring their operands into two LDS
// stages with direct global-to-LDS copies (tbq_dma.hpp): a step's copies are
// issued at the start of the step before and waited for at its end, so no
// register holds data in flight.  LDS rows are 128 bytes (64 halves) without
// padding; the 16-byte segment of row r sits at slot seg ^ (r & 7) ^ (r >> 3
// & 1), so the 32 rows of a column read spread over all banks (the copies'
// per-lane source addresses place them there).
//
// What bounds them (MI355X): on random operands the matrix cores alone reach
// 1.6 PFLOP/s here (2.16 on zeros: the power limit sets the clock), and every
// VALU instruction beside an MFMA costs clock as well (1.28 PFLOP/s at 4 per
// MFMA).  k_hgemm_q4k without its copies and without the dequantisation runs
// at 1.18 PFLOP/s.
//
// k_hgemm_q4k (Q4_K rows, reference layout).  Wave w owns 64 weight rows and
// all of the tile's tokens, so a weight is dequantised once per tile by the
// one wave that uses it and never passes through LDS as fp16: only the packed
// bytes are staged (4.5 bits a weight), each lane reads its own row's 16
// quant bytes of a step and makes its A fragments in registers between the
// MFMAs of the fragments before (the k order inside a step is permuted: lane
// half h covers columns 32 h .. + 31, for both operands).  64 x 128 blocks
// per wave read 4 KiB of LDS per 8 MFMAs.  Two workgroups of 256 x 128 per CU
// overlap each other's barriers: one workgroup of 256 x 256 that dequantises
// into LDS (8 waves in step) was slower on every shape (T = 1999: 19456 x
// 2560 295 against 198 us).  Against the kernel this replaces (128 x 128
// tiles, operands through registers into padded LDS): T = 512: 6144 x 2560
// 45.1 -> 26.8 us, 2560 x 4096 37.0 -> 22.9, 2560 x 9728 67.4 -> 39.8, gate |
// up 19456 x 2560 106.1 -> 66.1 (SwiGLU included); T = 1999: 124.6 -> 72.4,
// 102.6 -> 56.4, 211.3 -> 126.0 and 330.8 -> 198.2 us (1.0 PFLOP/s).
//
// k_hgemm_f16 (fp16 rows).  Both operands through LDS, waves in a WN x WT
// grid.  Here the L2-to-LDS traffic bounds the tile: 256 x 256 (64 KiB a
// step) beats two workgroups of 256 x 128 (T = 1999, 19456 x 2560: 240
// against 274 us); a ring of three or four 32-column stages with counted
// waits was slower than these two of 64 (261 us).  T = 512: 40.3 -> 26.5,
// 33.3 -> 21.3, 59.5 -> 38.6 and 89.8 -> 67.4 us on the shapes above; T =
// 1999: 95.9 -> 69.1, 85.9 -> 56.3, 204.7 -> 120.4 and 338.9 -> 239.9 us.
//
// Split K.  When the tiles are too few for the CUs, K is split over
// gridDim.y slices; slice z writes its partial sums to P[z][T][N] and
// k_gemm_reduce (or the consumer) adds the slices in slice order.
#include <algorithm>

#include "tbq_dma.hpp"
#include "tbq_kernels.h"
#include "tbq_kquant.hpp"

namespace tbq {

namespace {

typedef _Float16 hg_f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 hg_f16x2 __attribute__((ext_vector_type(2)));
typedef float hg_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned hg_u32x4 __attribute__((ext_vector_type(4)));

// Slot swizzles: 128-byte rows of eight 16-byte segments, and 64-byte rows of
// four.  Any 8 consecutive rows of a column read fall on 8 different 16-byte
// bank groups of 128 bytes, any 16 on 16 of 256.
__device__ __forceinline__ int swz8(int r) { return (r & 7) ^ ((r >> 3) & 1); }
__device__ __forceinline__ int swz4(int r) { return (((r >> 2) & 1) << 1) | (((r >> 1) ^ (r >> 3)) & 1); }

// blockIdx.x -> tile.  Workgroup i runs on XCD i % 8, so each XCD takes a
// contiguous range of tiles (token tiles fastest): the token tiles of a
// weight row block meet in one L2.  -1: no tile (grid rounded up to 8).
__device__ __forceinline__ int hg_tile(int ntile) {
    const int per = (ntile + 7) >> 3, i = blockIdx.x >> 3, tile = (blockIdx.x & 7) * per + i;
    return tile < ntile && i < per ? tile : -1;
}

// Accumulator register r of lane l: weight row 8(r/4) + 4(l/32) + r%4 of the
// 32-row block, token l % 32 of the 32-token block.  Row blocks of one wave
// start at output row nb + 32 i, its token blocks at tb + 32 j.  GLU: block 2p
// holds gate and block 2p + 1 up rows of outputs nb + 32 p .. of F = N / 2,
// out[t][c] = silu(g xs[t]) (u xs[t]).
template <bool GLU, int NA, int NB>
__device__ __forceinline__ void hg_store(const hg_f32x16 (&acc)[NA][NB], int nb, int tb, int T, int N,
                                         float *__restrict__ out, int ldo, const float *__restrict__ xs) {
    const int lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5;
    static_assert(!GLU || NA % 2 == 0, "GLU pairs the wave's 32-row blocks");
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int t = tb + 32 * j + li;
        if (t >= T) continue;
        float *o = out + (long long)t * ldo;
        float sx = 1.f;
        if constexpr (GLU) sx = xs[t];
#pragma unroll
        for (int i = 0; i < (GLU ? NA / 2 : NA); i++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int n = nb + 32 * i + 8 * g + 4 * lh;
                if (n >= (GLU ? N / 2 : N)) continue;   // rows past the end (clamped loads) are not stored
                float r[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if constexpr (GLU) r[e] = pro_swiglu(acc[2 * i][j][4 * g + e] * sx, acc[2 * i + 1][j][4 * g + e] * sx);
                    else r[e] = acc[i][j][4 * g + e];
                }
                *reinterpret_cast<float4 *>(o + n) = make_float4(r[0], r[1], r[2], r[3]);
            }
    }
}

template <int NW, int NB>
struct HqLds {
    static constexpr int ROWS = 64 * NW, TOK = 32 * NB;
    unsigned char act[2][TOK * 128];   // two 64-column steps of the activation rows
    unsigned char q[2][ROWS * 64];     // quants of a super-block's two 128-column halves
    unsigned char hdr[ROWS * 16];      // its first 16 bytes: d, dmin and the scale bytes
};

template <int WN, int WT, int NA, int NB>
struct HfLds {
    static constexpr int ROWS = WN * NA * 32, TOK = WT * NB * 32;
    unsigned char s[2][(ROWS + TOK) * 128];   // two 64-column steps: weight rows, then activation rows
};

}  // namespace

// kper = K columns per slice (a multiple of 256); out = C with row stride ldo
// (one slice) or the slice partials P[z][T][N] (ldo = N).  The weights' decode:
// a nibble q becomes the fp16 number 1 + q/16 by placing it in the mantissa
// (0x3C00 | q << 6, both nibbles of a byte from one 24-bit multiply and one
// v_bitop3 (a & b) | c), and one packed fp16 fma with (16 S, C = -16 S - M)
// gives 16 S (1 + q/16) + C = S q - M, exact before its one rounding: 1.5 VALU
// per weight, with the fp16 roundings of 16 S, C and the result (16 d 63 +
// dmin 63 must stay below 65504).
template <int NW, int NB, bool GLU>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) void k_hgemm_q4k(
    const uint8_t *__restrict__ W, const _Float16 *__restrict__ X, int T, int N, int K, int nt, int ntile, int kper,
    float *__restrict__ out, int ldo, const float *__restrict__ xs) {
    using L = HqLds<NW, NB>;
    constexpr int ROWS = L::ROWS, TOK = L::TOK;
    extern __shared__ __attribute__((aligned(1024))) unsigned char hq_lds[];
    L *st = reinterpret_cast<L *>(hq_lds);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31,
              lh = lane >> 5;
    const int tile = hg_tile(ntile);
    if (tile < 0) return;   // uniform
    const int n0 = (tile / nt) * ROWS, t0 = (tile % nt) * TOK;
    const int kb = blockIdx.y * kper, nsb = (min(K, kb + kper) - kb) >> 8;   // super-blocks of this slice
    const uint32_t rb = (uint32_t)(K >> 8) * 144u;

    // rows of this wave's two 32-row blocks
    const int F = N >> 1;
    const int rbase0 = GLU ? (n0 >> 1) + 32 * wave : n0 + 64 * wave;
    const int rbase1 = GLU ? F + rbase0 : rbase0 + 32;
    const int rmax0 = GLU ? F - 1 : N - 1, rmax1 = N - 1;
    // descriptor bases at the (clamped) first rows of each block
    const int rs0 = min(rbase0, rmax0), rs1 = min(rbase1, rmax1);
    const dma_rsrc_t w0 = dma_rsrc(W + (long long)rs0 * rb + (long long)(kb >> 8) * 144, 0x7FFFFFFFu);
    const dma_rsrc_t w1 = dma_rsrc(W + (long long)rs1 * rb + (long long)(kb >> 8) * 144, 0x7FFFFFFFu);
    const dma_rsrc_t xr = dma_rsrc(X + kb, 0x7FFFFFFFu);
    // quant copies: 16 rows x 4 segments each; group g of 4 covers rows 16 g .. of the wave's 64
    uint32_t qv[4], hv;
    {
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int rr = 16 * (g & 1) + (lane >> 2);   // row in its 32-row block
            const int row = g < 2 ? min(rbase0 + rr, rmax0) - rs0 : min(rbase1 + rr, rmax1) - rs1;
            qv[g] = (uint32_t)row * rb + 16u + 16u * ((lane & 3) ^ swz4(rr));
        }
    }
    // header copy: lane = row (0..31 of block 0, then of block 1), all through block 0's descriptor
    {
        const long long row = lane < 32 ? min(rbase0 + li, rmax0) : min(rbase1 + li, rmax1);
        hv = (uint32_t)((row - rs0) * (long long)rb);
    }
    // activation copies: 8 tokens x 8 segments each; the 4 NB copies of a step are dealt to the waves round-robin
    constexpr int AC = 4 * NB, APW = (AC + NW - 1) / NW;
    uint32_t av[APW];
#pragma unroll
    for (int i = 0; i < APW; i++) {
        const int tok = 8 * (wave + NW * i) + (lane >> 3);
        av[i] = (uint32_t)min(t0 + tok, T - 1) * (uint32_t)(K * 2) + 16u * ((lane & 7) ^ swz8(tok));
    }
    const uint32_t la = lds_addr(st->act[0]), lq = lds_addr(st->q[0]) + wave * 4096, lhd = lds_addr(st->hdr) + wave * 1024;
    auto copy_act = [&](int buf, int step) {   // step: 64-column step of the slice
#pragma unroll
        for (int i = 0; i < APW; i++) {
            const int c = wave + NW * i;
            if (AC % NW == 0 || c < AC) dma16(la + buf * (TOK * 128) + c * 1024, av[i], xr, step * 128);
        }
    };
    auto copy_q = [&](int half, int g, int sb) {   // group g of super-block sb's 128-column half
        dma16(lq + half * (ROWS * 64) + g * 1024, qv[g], g < 2 ? w0 : w1, (uint32_t)(sb * 144 + half * 64));
    };

    hg_f32x16 acc[2][NB];
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[b][j] = hg_f32x16{};

    // LDS read offsets
    const int fq = swz4(li), fa = swz8(li);
    hg_u32x4 hd[2], q[2];
    uint32_t mhi[2];
    float d[2], dm[2];
    hg_f16x2 S16[2], C[2];
    hg_f16x8 a[2][2];   // [kk parity][block]
    const unsigned char *qbase = st->q[0] + (wave * 64 + li) * 64;
    // raw quants of step s (0..3) of the super-block whose halves are in LDS
    auto raw = [&](int s) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const unsigned char *qrow = qbase + (s >> 1) * (ROWS * 64) + 32 * b * 64;
            if (s == 0) {
                hd[b] = *reinterpret_cast<const hg_u32x4 *>(st->hdr + (wave * 64 + 32 * b + li) * 16);
                mhi[b] = *reinterpret_cast<const uint32_t *>(qrow + 16 * fq);
            }
            q[b] = *reinterpret_cast<const hg_u32x4 *>(qrow + 16 * (((s & 1) * 2 + lh) ^ fq));
        }
    };
    // scale and constant of step s
    auto scales = [&](int s) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            if (s == 0) {
                d[b] = (hd[b].x & 0x7C00u) ? (float)__builtin_bit_cast(_Float16, (uint16_t)(hd[b].x & 0xFFFFu)) : 0.f;
                dm[b] = (hd[b].x & 0x7C000000u) ? (float)__builtin_bit_cast(_Float16, (uint16_t)(hd[b].x >> 16)) : 0.f;
            }
            const uint32_t sw = s < 2 ? hd[b].y : hd[b].w, mw = s < 2 ? hd[b].z : mhi[b];
            const int jb = 16 * (s & 1) + 8 * lh;
            const float S = d[b] * (float)((sw >> jb) & 63), M = dm[b] * (float)((mw >> jb) & 63);
            const _Float16 s16 = (_Float16)(16.f * S), cc = (_Float16)(-(float)s16 - M);
            S16[b] = hg_f16x2{s16, s16};
            C[b] = hg_f16x2{cc, cc};
        }
    };
    auto frag = [&](int b, int kk) {
        unsigned w[4];
        const unsigned qd = kk == 0 ? q[b].x : kk == 1 ? q[b].y : kk == 2 ? q[b].z : q[b].w;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const unsigned y = (qd >> (8 * i)) & 0xFFu;
            const unsigned t = __builtin_amdgcn_bitop3_b32(__umul24(y, 0x40040u), 0x03C003C0u, 0x3C003C00u, 0xEA);
            w[i] = __builtin_bit_cast(unsigned, __builtin_elementwise_fma(__builtin_bit_cast(hg_f16x2, t), S16[b], C[b]));
        }
        return __builtin_bit_cast(hg_f16x8, hg_u32x4{w[0], w[1], w[2], w[3]});
    };

    copy_act(0, 0);
    dma16(lhd, hv, w0, 0);
#pragma unroll
    for (int g = 0; g < 4; g++) { copy_q(0, g, 0); copy_q(1, g, 0); }
    dma_wait_barrier();
    raw(0);
    scales(0);
#pragma unroll
    for (int b = 0; b < 2; b++) a[0][b] = frag(b, 0);
    lds_read_wait();   // step 0's copies go to other slots, but every copy follows the reads before it
    for (int sb = 0; sb < nsb; sb++) {
        const int nx = min(sb + 1, nsb - 1);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            // copies of the next step (past the end: the last again, never read)
            copy_act((s + 1) & 1, min(4 * sb + s + 1, 4 * nsb - 1));
            if (s == 0) { copy_q(1, 2, sb); copy_q(1, 3, sb); }
            if (s == 1) { copy_q(0, 0, nx); copy_q(0, 1, nx); }
            if (s == 2) { copy_q(0, 2, nx); copy_q(0, 3, nx); dma16(lhd, hv, w0, (uint32_t)(nx * 144)); }
            if (s == 3) { copy_q(1, 0, nx); copy_q(1, 1, nx); }
            const unsigned char *ab = st->act[s & 1] + li * 128;
            hg_f16x8 bf[2][NB];
#pragma unroll
            for (int j = 0; j < NB; j++) bf[0][j] = *reinterpret_cast<const hg_f16x8 *>(ab + j * 4096 + 16 * ((4 * lh) ^ fa));
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                if (kk < 3) {
#pragma unroll
                    for (int j = 0; j < NB; j++)
                        bf[(kk + 1) & 1][j] = *reinterpret_cast<const hg_f16x8 *>(ab + j * 4096 + 16 * ((4 * lh + kk + 1) ^ fa));
                    if (kk == 2) {
                        // fragment 3 first: the raw registers are then free
                        a[1][0] = frag(0, 3);
                        a[1][1] = frag(1, 3);
                        raw((s + 1) & 3);
                    } else {
                        a[(kk + 1) & 1][0] = frag(0, kk + 1);
                        a[(kk + 1) & 1][1] = frag(1, kk + 1);
                    }
                } else {
                    scales((s + 1) & 3);
                    a[0][0] = frag(0, 0);
                    a[0][1] = frag(1, 0);
                }
#pragma unroll
                for (int j = 0; j < NB; j++)
#pragma unroll
                    for (int b = 0; b < 2; b++)
                        acc[b][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[kk & 1][b], bf[kk & 1][j], acc[b][j], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 2 * NB; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);
                }
            }
            dma_wait_barrier();
        }
    }
    hg_store<GLU>(acc, GLU ? rbase0 : n0 + 64 * wave, t0, T, N, out + (long long)blockIdx.y * T * N, ldo, xs);
}

// The same product for fp16 rows; GLU's 32-row blocks alternate gate and up.
template <int WN, int WT, int NA, int NB, bool GLU>
__global__ __launch_bounds__(64 * WN * WT) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_hgemm_f16(
    const _Float16 *__restrict__ W, const _Float16 *__restrict__ X, int T, int N, int K, int nt, int ntile, int kper,
    float *__restrict__ out, int ldo, const float *__restrict__ xs) {
    using L = HfLds<WN, WT, NA, NB>;
    constexpr int NW = WN * WT, ROWS = L::ROWS, TOK = L::TOK, SB = (ROWS + TOK) * 128;
    constexpr int NC = (ROWS + TOK) / 8, CPW = NC / NW;   // 1 KiB copies per stage, per wave
    static_assert(NC % NW == 0 && (ROWS / 8) % NW == 0, "");
    extern __shared__ __attribute__((aligned(1024))) unsigned char hf_lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31,
              lh = lane >> 5;
    const int tile = hg_tile(ntile);
    if (tile < 0) return;   // uniform
    const int n0 = (tile / nt) * ROWS, t0 = (tile % nt) * TOK;
    const int kb = blockIdx.y * kper, nst = (min(K, kb + kper) - kb) >> 6;
    const int F = N >> 1;
    auto wrow = [&](int rho) {
        if constexpr (GLU) return min((rho & 32 ? F : 0) + min((n0 >> 1) + 32 * (rho >> 6) + (rho & 31), F - 1), N - 1);
        else return min(n0 + rho, N - 1);
    };
    const int base = wrow(0);
    const dma_rsrc_t wr = dma_rsrc(W + (long long)base * K + kb, 0xFFFFFFFFu), xr = dma_rsrc(X + kb, 0x7FFFFFFFu);
    const uint32_t l0 = lds_addr(hf_lds);
    // 8 rows x 8 segments per copy, swizzled as the quant copies
    uint32_t vo[CPW];
#pragma unroll
    for (int i = 0; i < CPW; i++) {
        const int c = wave + NW * i, r = 8 * c + (lane >> 3);
        const uint32_t seg = 16u * ((lane & 7) ^ swz8(r));
        if (i < ROWS / 8 / NW) vo[i] = (uint32_t)(wrow(r) - base) * (uint32_t)(K * 2) + seg;
        else vo[i] = (uint32_t)min(t0 + r - ROWS, T - 1) * (uint32_t)(K * 2) + seg;
    }
    auto copy = [&](int slot, int step) {
#pragma unroll
        for (int i = 0; i < CPW; i++)
            dma16(l0 + slot * SB + (wave + NW * i) * 1024, vo[i], i < ROWS / 8 / NW ? wr : xr, step * 128);
    };
    const int wn = NA * 32 * (wave % WN), wt = NB * 32 * (wave / WN);
    const int fr = swz8(li);
    hg_f32x16 acc[NA][NB];
#pragma unroll
    for (int b = 0; b < NA; b++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[b][j] = hg_f32x16{};
    const int last = nst - 1;
    copy(0, 0);
    dma_wait_barrier();
    const unsigned char *A = hf_lds + (wn + li) * 128, *B = hf_lds + (ROWS + wt + li) * 128;
    for (int s0 = 0; s0 < nst; s0 += 2) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            copy(s ^ 1, min(s0 + s + 1, last));
            const unsigned char *As = A + s * SB, *Bs = B + s * SB;
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                const int o = 16 * ((2 * kk + lh) ^ fr);
                hg_f16x8 a[NA], b[NB];
#pragma unroll
                for (int i = 0; i < NA; i++) a[i] = *reinterpret_cast<const hg_f16x8 *>(As + i * 4096 + o);
#pragma unroll
                for (int i = 0; i < NB; i++) b[i] = *reinterpret_cast<const hg_f16x8 *>(Bs + i * 4096 + o);
#pragma unroll
                for (int j = 0; j < NB; j++)
#pragma unroll
                    for (int i = 0; i < NA; i++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], acc[i][j], 0, 0, 0);
            }
            // every read of the next k group goes out behind the first MFMAs of this one
            __builtin_amdgcn_sched_group_barrier(0x100, NA + NB, 0);
#pragma unroll
            for (int i = 0; i < 4 * NA * NB; i++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            dma_wait_barrier();
        }
    }
    hg_store<GLU>(acc, GLU ? (n0 + wn) >> 1 : n0 + wn, t0 + wt, T, N, out + (long long)blockIdx.y * T * N, ldo, xs);
}

// C[t][n] (row stride ldc) = sum over the S slices of P[z][t][n], in slice order.
__global__ __launch_bounds__(256) void k_gemm_reduce(const float *__restrict__ P, int S, int T, int N,
                                                     float *__restrict__ C, int ldc) {
    const long long n4 = (long long)T * N / 4;
    const int N4 = N / 4;
    for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n4; i += (long long)gridDim.x * 256) {
        float4 a = reinterpret_cast<const float4 *>(P)[i];
        for (int z = 1; z < S; z++) {
            const float4 b = reinterpret_cast<const float4 *>(P)[z * n4 + i];
            a.x = a.x + b.x;
            a.y = a.y + b.y;
            a.z = a.z + b.z;
            a.w = a.w + b.w;
        }
        const long long t = i / N4, c = i - t * N4;
        *reinterpret_cast<float4 *>(C + t * ldc + 4 * c) = a;
    }
}

// CUs the slicing plans for (the device's, at most 256, so that workspace
// sizes computed before and after initialisation agree on this part).
int hgemm_cus() {
    const int c = tbq_cu_count();
    return c > 0 && c < 256 ? c : 256;
}

namespace {

// Tile choice.  A launch of W workgroups runs n = ceil(W / CUs) of them on
// its busiest CU, so its time is about
//   c0 + steps * (n == 1 ? ke + (k1 - ke) W / CUs : n k2 / 2) + partial sums
// in us, with steps = 64-column steps per workgroup: ke is a step of one
// workgroup on an otherwise idle chip, k1 with one on every CU (clock and L2
// shared), k2 a step of two on every CU.  The constants were fitted to 585
// measured launches (every tile, T 20..1999, N 2560..19456, K 2560..9728, 1
// to 8 slices; 4-12% rms; prefills of 1024- and 2048-wide models, N and K from
// 1024, are 8 to 44% faster with its choice than on fixed 128 x 128 tiles), and
// the launch takes the tile and slice count with
// the least; partial sums are priced at 0.25 us a MB written plus 0.2 read.
struct HgTile {
    int rows, tok;
    float c0, ke, k1, k2;
};
constexpr HgTile HG_Q4K[] = {{256, 128, 3.2f, 0.635f, 1.011f, 1.502f}, {128, 128, 4.0f, 0.577f, 0.709f, 1.116f},
                             {256, 64, 1.7f, 0.587f, 0.828f, 1.075f}, {128, 64, 3.0f, 0.466f, 0.625f, 0.764f},
                             {128, 32, 4.1f, 0.381f, 0.451f, 0.544f}};
constexpr HgTile HG_F16[] = {{256, 256, 2.7f, 1.106f, 1.520f, 3.559f}, {128, 128, 1.1f, 0.551f, 0.776f, 0.973f},
                             {128, 64, 1.0f, 0.466f, 0.635f, 0.678f}};

struct HgPlan {
    int tile, S, per;   // index into the table, slices, super-blocks per slice
};

// max_slices and part_bytes (room for the partial sums) limit the slices.
template <int NT>
HgPlan hg_plan(const HgTile (&tab)[NT], int T, int N, int K, int n_cu, int max_slices, size_t part_bytes) {
    HgPlan best{0, 1, K / 256};
    float bt = 1e30f;
    for (int i = 0; i < NT; i++) {
        const long long tiles = (long long)((N + tab[i].rows - 1) / tab[i].rows) * ((T + tab[i].tok - 1) / tab[i].tok);
        for (int s = 1; s <= std::min(max_slices, K / 256); s++) {
            const int per = (K / 256 + s - 1) / s, S = (K / 256 + per - 1) / per;
            if (S != s) continue;
            if (s > 1 && (size_t)s * T * N * 4 > part_bytes) break;
            const long long W = tiles * S, n = (W + n_cu - 1) / n_cu;
            const float steps = 4.f * per, mb = (float)T * N * 4e-6f;
            const float step = n == 1 ? tab[i].ke + (tab[i].k1 - tab[i].ke) * W / n_cu : n * tab[i].k2 * 0.5f;
            const float t = tab[i].c0 + steps * step + 0.25f * mb * S + (S > 1 ? 0.2f * mb * S : 0.f);
            if (t < bt) {
                bt = t;
                best = {i, S, per};
            }
        }
    }
    return best;
}

constexpr int HG_MAX_SLICES = 8;   // the consumers add at most this many

template <int NW, int NB, bool GLU>
hipError_t go_q4k(const void *W, const _Float16 *X, int T, int N, int K, const HgPlan &p, float *out, int ldo,
                  const float *xs, hipStream_t st) {
    using L = HqLds<NW, NB>;
    // more than 64 KiB of dynamic LDS is opted into once per kernel
    static const hipError_t a = hipFuncSetAttribute((const void *)k_hgemm_q4k<NW, NB, GLU>,
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(L));
    if (a != hipSuccess) return a;
    const int nt = (T + L::TOK - 1) / L::TOK, ntile = nt * ((N + L::ROWS - 1) / L::ROWS);
    hipLaunchKernelGGL((k_hgemm_q4k<NW, NB, GLU>), dim3((ntile + 7) / 8 * 8, p.S), dim3(64 * NW), sizeof(L), st,
                       (const uint8_t *)W, X, T, N, K, nt, ntile, p.per * 256, out, ldo, xs);
    return hipGetLastError();
}

template <int WN, int WT, int NA, int NB, bool GLU>
hipError_t go_f16(const void *W, const _Float16 *X, int T, int N, int K, const HgPlan &p, float *out, int ldo,
                  const float *xs, hipStream_t st) {
    using L = HfLds<WN, WT, NA, NB>;
    static const hipError_t a = hipFuncSetAttribute((const void *)k_hgemm_f16<WN, WT, NA, NB, GLU>,
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(L));
    if (a != hipSuccess) return a;
    const int nt = (T + L::TOK - 1) / L::TOK, ntile = nt * ((N + L::ROWS - 1) / L::ROWS);
    hipLaunchKernelGGL((k_hgemm_f16<WN, WT, NA, NB, GLU>), dim3((ntile + 7) / 8 * 8, p.S), dim3(64 * WN * WT),
                       sizeof(L), st, (const _Float16 *)W, X, T, N, K, nt, ntile, p.per * 256, out, ldo, xs);
    return hipGetLastError();
}

template <bool GLU>
hipError_t go(int wqt, const void *W, const _Float16 *X, int T, int N, int K, const HgPlan &p, float *out, int ldo,
              const float *xs, hipStream_t st) {
    if (wqt == QT_F16) {
        switch (p.tile) {
        case 0: return go_f16<4, 2, 2, 4, GLU>(W, X, T, N, K, p, out, ldo, xs, st);
        case 1: return go_f16<2, 2, 2, 2, GLU>(W, X, T, N, K, p, out, ldo, xs, st);
        default: return go_f16<2, 2, 2, 1, GLU>(W, X, T, N, K, p, out, ldo, xs, st);
        }
    }
    switch (p.tile) {
    case 0: return go_q4k<4, 4, GLU>(W, X, T, N, K, p, out, ldo, xs, st);
    case 1: return go_q4k<2, 4, GLU>(W, X, T, N, K, p, out, ldo, xs, st);
    case 2: return go_q4k<4, 2, GLU>(W, X, T, N, K, p, out, ldo, xs, st);
    case 3: return go_q4k<2, 2, GLU>(W, X, T, N, K, p, out, ldo, xs, st);
    default: return go_q4k<2, 1, GLU>(W, X, T, N, K, p, out, ldo, xs, st);
    }
}

HgPlan hg_plan_for(int wqt, int T, int N, int K, int n_cu, int max_slices, size_t part_bytes) {
    return wqt == QT_F16 ? hg_plan(HG_F16, T, N, K, n_cu, max_slices, part_bytes)
                         : hg_plan(HG_Q4K, T, N, K, n_cu, max_slices, part_bytes);
}

// Slices that either weight format's plan would take, given room.
int hg_slices(int T, int N, int K, int n_cu) {
    return std::max(hg_plan_for(QT_F16, T, N, K, n_cu, HG_MAX_SLICES, SIZE_MAX).S,
                    hg_plan_for(QT_Q4_K, T, N, K, n_cu, HG_MAX_SLICES, SIZE_MAX).S);
}

}  // namespace

// Partial sums of a T x N product over K, whichever weight format runs it.
size_t hgemm_partial_bytes(int T, int N, int K, int n_cu) {
    const int s = hg_slices(T, N, K, n_cu);
    return s > 1 ? (size_t)s * T * N * 4 : 0;
}

// The most that any product of 1 .. T rows wants.  Within 32 rows the tile
// counts stay and only the price of the partial sums grows, so the slices are
// at most those of the first row.
size_t hgemm_partial_upto(int T, int N, int K, int n_cu) {
    size_t most = 0;
    for (int t = 1; t <= T; t += 32) {
        const int s = hg_slices(t, N, K, n_cu);
        if (s > 1) most = std::max(most, (size_t)s * std::min(t + 31, T) * N * 4);
    }
    return most;
}

bool hgemm_supported(int wqt, int N, int K) {
    return (wqt == QT_F16 || wqt == QT_Q4_K) && N > 0 && N % 4 == 0 && K > 0 && K % 256 == 0;
}

bool hgemm_plan(int wqt, int T, int N, int K, bool glu, int n_cu, int plan[3]) {
    if (!hgemm_supported(wqt, N, K) || T <= 0 || (glu && N % 128)) return false;
    const HgPlan p = hg_plan_for(wqt, T, N, K, n_cu, glu ? 1 : HG_MAX_SLICES, SIZE_MAX);
    plan[0] = wqt == QT_F16 ? HG_F16[p.tile].rows : HG_Q4K[p.tile].rows;
    plan[1] = wqt == QT_F16 ? HG_F16[p.tile].tok : HG_Q4K[p.tile].tok;
    plan[2] = p.S;
    return true;
}

// The gate/up product with SwiGLU in the epilogue: W holds 2F rows (gate then
// up), A[T][F] (row stride lda) = silu(g xs) (u xs).  K is never split here
// (the SwiGLU of partial sums is not defined).  hipErrorNotSupported where F
// is not a multiple of 64.
hipError_t launch_hgemm_glu(int wqt, const void *W, const _Float16 *X, const float *xs, int T, int F, int K,
                            float *A, int lda, int n_cu, hipStream_t st) {
    const int N = 2 * F;
    if (!hgemm_supported(wqt, N, K) || F % 64 || T <= 0 || (long long)T * K * 2 >= (1ll << 31))
        return hipErrorNotSupported;
    return go<true>(wqt, W, X, T, N, K, hg_plan_for(wqt, T, N, K, n_cu, 1, 0), A, lda, xs, st);
}

// wqt: QT_F16 (IEEE fp16 rows, as k_dequant_f16 writes them) or QT_Q4_K.
// C: T rows of N floats at row stride ldc.  part: part_bytes of device memory
// for the slices' partial sums, which limit them (hgemm_partial_bytes() do not).
hipError_t launch_hgemm(int wqt, const void *W, const _Float16 *X, int T, int N, int K, float *C, int ldc,
                        float *part, size_t part_bytes, int n_cu, hipStream_t st, int *nslices) {
    if (!hgemm_supported(wqt, N, K) || T <= 0 || (long long)T * K * 2 >= (1ll << 31)) return hipErrorNotSupported;
    const HgPlan p = hg_plan_for(wqt, T, N, K, n_cu, HG_MAX_SLICES, part ? part_bytes : 0);
    if (nslices && p.S > 1 && ldc != N) return hipErrorInvalidValue;   // slices are packed at row stride N
    const hipError_t err = go<false>(wqt, W, X, T, N, K, p, p.S > 1 ? part : C, p.S > 1 ? N : ldc, nullptr, st);
    if (nslices) *nslices = p.S;
    if (err != hipSuccess || p.S == 1 || nslices) return err;
    const long long n4 = (long long)T * N / 4;
    const int g = (int)std::min<long long>((n4 + 255) / 256, 4096);
    hipLaunchKernelGGL(k_gemm_reduce, dim3(g), dim3(256), 0, st, part, p.S, T, N, C, ldc);
    return hipGetLastError();
}

}  // namespace tbq

// tbq_moe_prefill.hip -- batched (prefill) MoE experts on gfx950 fp16 MFMA.
//
// After routing (exact, as in decode), the (token, slot) pairs are grouped by
// expert and every expert's products run as dense tiles:
//
//   k_dispatch        per-expert histogram, prefix sum and permutation of the
//                     pairs in LDS (one workgroup), plus a tile list of
//                     (expert, first pair, pairs in tile) entries of <= 128
//                     pairs; order inside an expert does not affect results.
//   k_rows_f16        a matrix of fp32 rows to fp16, each row scaled by a
//                     power of two that puts its max |value| in [2^14, 2^15)
//                     (exact, undone in the GEMM epilogues): x for gate/up,
//                     the SwiGLU activations for down.
//   k_moe_f16<0>      act[p] = swiglu(x_t . W_gate[e], x_t . W_up[e]) for a
//                     tile of <= 128 pairs x 64 or 128 columns (as many gate
//                     and as many up rows), K = H, fp32 out.
//   k_moe_f16<1>      y[p] = act[p] . W_down[e] for <= 128 pairs x 128 or 256
//                     rows, K = F.
//   (k_combine)       out = resid + sum over slots in slot order (tbq_moe.hip).
//
// Weights never pass through LDS as fp16: their packed bytes are staged and
// each lane dequantises its own MFMA A operands in registers.
//
// Dequantisation to fp16.  A nibble q becomes the fp16 number 1 + q/16 by
// placing q in the mantissa (0x3C00 | q << 6), for two weights per dword:
// one 24-bit multiply spreads a quant byte's two nibbles into the two
// halves, one three-input bit operation (v_bitop3, (a & b) | c) masks them
// and sets the exponent; one v_pk_fma_f16 with (16 S, C = -16 S - M) gives
// 16 S (1 + q/16) + C = S q - M: three VALU per two weights.  The fma's
// product and sum are exact before its one rounding, so the fp16 roundings
// are those of 16 S, of C (at most ulp(16 S + M) / 2, a per-sub-block
// constant) and of the result.
//
// Accuracy: fp16 weights and activations (11-bit mantissa), fp32
// accumulation; outputs land within 1e-2 relative L2 of the fp32 reference.
// The weights' fp16 form needs 16 * 63 * d + 63 * dmin below 65504.
#include "tbq_dma.hpp"
#include "tbq_kernels.h"
#include "tbq_kquant.hpp"

namespace tbq {

// The int8 prefill decodes Q4_K in the reference's layout for all three
// expert tensors; the fp16 one also takes all three in ggml's layout.
static bool prefill_q4k_layer(const MoeArgs &a) { return a.qg == QT_Q4_K && a.qu == QT_Q4_K && a.qd == QT_Q4_K; }
static bool prefill_gq4k_layer(const MoeArgs &a) {
    return a.qg == QT_GQ4_K && a.qu == QT_GQ4_K && a.qd == QT_GQ4_K;
}

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
// native vectors: HIP's uint4 struct is copied with memcpy, which keeps
// register arrays in scratch memory
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int PF_MT = 128;         // pairs per tile (four 32-pair MFMA sub-tiles)
constexpr int PF_KC = 128;         // K columns per chunk (half a Q4_K super-block)
#ifndef PF_WAVES
#define PF_WAVES 8
#endif
constexpr int PF_THREADS = 64 * PF_WAVES;   // 32 weight rows per wave
constexpr int PF_ROWS = 32 * PF_WAVES;      // weight rows per workgroup
constexpr int PF_COLS = PF_ROWS / 2;        // gate/up columns per workgroup

struct PfTile {
    int e, n;
};

// a tile's count of 32-pair sub-tiles as a type, for the per-count copies of
// the expert GEMM's chunk loop
template <int N>
struct PfSub {
    static constexpr int value = N;
};

// ---------------------------------------------------------------------------
// Dispatch: one workgroup of 1024 threads.  pairs p = t*k + s.  Tiles are
// listed heaviest first (by 32-pair sub-tile count), so the
// longest workgroups start first and the grid's tail is short; tile T's
// pairs are tpair[128T .. 128T + n) (-1 after), its activation rows ttok
// (= pair / k, the token).
// ---------------------------------------------------------------------------
constexpr int PF_MAX_TILES = 65536 * 8 / PF_MT + 256;
// NE > 0 (up to 1024 NE pairs): a thread keeps its NE pairs' expert indices in
// registers (read once) and the permutation is in LDS (16 bits a pair); NE = 0:
// any number, the permutation in global memory, read back after its own stores
// by a loop of dependent round trips (15992 pairs: 31 -> 19.5 us with NE = 16).
// One workgroup of code that no other launch keeps in the instruction cache is
// bound by its length as well, hence an instance per range: in one kernel with
// both forms and sixteen pairs a thread 4096 pairs took 10.9 us, with eight 8.9,
// and NE = 4 takes 8.5 (2400 pairs: 6.3, 5.3 and 5.0).
template <int NE>
__global__ __launch_bounds__(1024) void k_dispatch(const int *__restrict__ sel_idx, int T, int k, int E,
                                                   int *__restrict__ perm, PfTile *__restrict__ tiles,
                                                   int *__restrict__ ntiles, int *__restrict__ tpair,
                                                   int *__restrict__ ttok) {
    constexpr int NQ = PF_MT / 32;   // sub-tile count classes 1..NQ
    static_assert(PF_MT == 128 && NQ == 4, "tile classes");
    __shared__ int hist[256], off[257], cur[256], wsum[4];
    __shared__ int qcnt[NQ + 1], qbase[NQ + 2];
    constexpr int TILES = NE ? NE * 1024 / PF_MT + 256 : PF_MAX_TILES;
    __shared__ int t_e[TILES], t_start[TILES];
    __shared__ unsigned short perm_s[NE ? NE * 1024 : 1];
    const int tid = threadIdx.x, P = T * k;
    if (tid < 256) { hist[tid] = 0; cur[tid] = 0; }
    if (tid <= NQ) qcnt[tid] = 0;
    int es[NE ? NE : 1];
    if constexpr (NE > 0) {
#pragma unroll
        for (int m = 0; m < NE; m++) {
            const int p = tid + 1024 * m;
            es[m] = p < P ? sel_idx[(p / k) * 8 + p % k] : -1;
        }
    }
    __syncthreads();
    // a pair whose expert index is outside [0, E) (never produced by the
    // router) joins no tile; the combine skips its slot
    if constexpr (NE > 0) {
#pragma unroll
        for (int m = 0; m < NE; m++)
            if ((unsigned)es[m] < (unsigned)E) atomicAdd(&hist[es[m]], 1);
    } else {
        for (int p = tid; p < P; p += 1024) {
            const int e = sel_idx[(p / k) * 8 + p % k];
            if ((unsigned)e < (unsigned)E) atomicAdd(&hist[e], 1);
        }
    }
    __syncthreads();
    // exclusive prefix sum of hist over 256 experts: a scan within each of
    // the first four waves (shuffles, no barrier), then the wave totals.
    // Tiles counted per sub-tile class: expert e has n >> 7 full tiles
    // (class 4) and, if n % 128 > 0, one of class (n % 128 + 31) / 32;
    // per wave by ballot counts, one LDS atomic per wave and class.
    int incl = 0;
    if (tid < 256) {   // four whole waves
        const int lane = tid & 63, n = hist[tid];   // 0 for experts >= E
        incl = n;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        if (lane == 63) wsum[tid >> 6] = incl;
        const int rem = n & (PF_MT - 1), rq = (rem + 31) >> 5;   // 0 when rem = 0
        int c4 = (n >> 7) + (rq == NQ ? 1 : 0);
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) c4 += __shfl_xor(c4, d, 64);
        int cq[NQ + 1];
#pragma unroll
        for (int q = 1; q < NQ; q++) cq[q] = (int)__builtin_popcountll(__builtin_amdgcn_ballot_w64(rq == q));
        cq[NQ] = c4;
        if (lane == 0) {
#pragma unroll
            for (int q = 1; q <= NQ; q++)
                if (cq[q]) atomicAdd(&qcnt[q], cq[q]);
        }
    }
    __syncthreads();
    if (tid < 256) {
        int add = 0;
        for (int w = 0; w < (tid >> 6); w++) add += wsum[w];
        off[tid + 1] = incl + add;
    }
    if (tid == 0) {
        off[0] = 0;
        // classes NQ (heaviest) first
        int b = 0;
        for (int q = NQ; q >= 1; q--) {
            qbase[q] = b;
            b += qcnt[q];
            ntiles[3 + NQ - q] = qcnt[q];   // tiles of NQ, NQ - 1 .. 1 sub-tiles (k_moe_i8's items)
            qcnt[q] = 0;
        }
        *ntiles = b;
        // item tickets of the two expert GEMMs (k_moe_f16), taken from 0
        ntiles[1] = 0;
        ntiles[2] = 0;
        qbase[0] = b;
    }
    __syncthreads();
    if (tid < E) {
        const int n = hist[tid];
        for (int s0 = 0; s0 < n; s0 += PF_MT) {
            const int q = (min(PF_MT, n - s0) + 31) / 32;
            const int t = qbase[q] + atomicAdd(&qcnt[q], 1);
            t_e[t] = tid | min(PF_MT, n - s0) << 16;   // expert | pairs in the tile
            t_start[t] = off[tid] + s0;
        }
    }
    if constexpr (NE > 0) {
#pragma unroll
        for (int m = 0; m < NE; m++) {
            const int e = es[m];
            if ((unsigned)e < (unsigned)E) perm_s[off[e] + atomicAdd(&cur[e], 1)] = (unsigned short)(tid + 1024 * m);
        }
    } else {
        for (int p = tid; p < P; p += 1024) {
            const int e = sel_idx[(p / k) * 8 + p % k];
            if ((unsigned)e < (unsigned)E) perm[off[e] + atomicAdd(&cur[e], 1)] = p;
        }
    }
    __syncthreads();
    const int nt = qbase[0];
    // the tile's record and first pair are two independent LDS reads
#pragma unroll 4
    for (int i = tid; i < nt * PF_MT; i += 1024) {
        const int t = i >> 7, j = i & (PF_MT - 1), te = t_e[t], st = t_start[t];
        const int e = te & 0xFFFF, n = te >> 16;
        if (j == 0) tiles[t] = PfTile{e, n};
        int p = -1;
        if (j < n) p = NE ? perm_s[st + j] : perm[st + j];
        tpair[i] = p;
        ttok[i] = p >= 0 ? p / k : -1;
    }
}

static void launch_dispatch(const MoeArgs &a, int *perm, PfTile *tiles, int *ntiles, int *tpair, int *ttok, hipStream_t st) {
#define TBQ_DISPATCH(NE)                                                                                            \
    hipLaunchKernelGGL(k_dispatch<NE>, dim3(1), dim3(1024), 0, st, a.sel_idx, a.T, a.k, a.E, perm, tiles, ntiles, \
                       tpair, ttok)
    const long long P = (long long)a.T * a.k;
    if (P <= 4096) TBQ_DISPATCH(4);
    else if (P <= 8192) TBQ_DISPATCH(8);
    else if (P <= 16384) TBQ_DISPATCH(16);
    else TBQ_DISPATCH(0);
#undef TBQ_DISPATCH
}

// ---------------------------------------------------------------------------
// Rows of n floats to fp16: one workgroup per row; s = 2^(15 - e) with
// max |row| = f * 2^e (f in [0.5, 1)), so |row| * s < 2^15; inv[row] = 1/s.
// n a multiple of 4.  swap: every four elements are stored in the order 0, 2,
// 1, 3 (the k order of the ggml layout's fragments).
// ---------------------------------------------------------------------------
// RV > 0: the row is held in registers (n <= 1024 RV), read once with
// every load issued before the max; RV = 0: two passes over the row.
template <int RV>
__global__ __launch_bounds__(256) void k_rows_f16(const float *__restrict__ in, int n, _Float16 *__restrict__ out,
                                                  float *__restrict__ inv, bool swap) {
    __shared__ float part[4];
    const int row = blockIdx.x, tid = threadIdx.x, n4 = n / 4;
    const float4 *r = reinterpret_cast<const float4 *>(in + (long long)row * n);
    float4 v[RV > 0 ? RV : 1];
    float mx = 0.f;
    if constexpr (RV > 0) {
#pragma unroll
        for (int i = 0; i < RV; i++) v[i] = r[min(tid + 256 * i, n4 - 1)];   // clamped: unconditional
#pragma unroll
        for (int i = 0; i < RV; i++)
            if (tid + 256 * i < n4)
                mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
    } else {
        for (int i = tid; i < n4; i += 256) {
            const float4 w = r[i];
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(w.x), fabsf(w.y)), fmaxf(fabsf(w.z), fabsf(w.w))));
        }
    }
    mx = wave_max(mx);
    if ((tid & 63) == 0) part[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
    int e = 0;
    frexpf(mx, &e);
    int sh = mx > 0.f ? 15 - e : 0;
    sh = sh > 126 ? 126 : (sh < -126 ? -126 : sh);
    const float s = ldexpf(1.f, sh);
    uint2 *o = reinterpret_cast<uint2 *>(out + (long long)row * n);
    auto put = [&](int i, float4 w) {
        const f16x2 a = {(_Float16)(w.x * s), (_Float16)((swap ? w.z : w.y) * s)};
        const f16x2 b = {(_Float16)((swap ? w.y : w.z) * s), (_Float16)(w.w * s)};
        o[i] = make_uint2(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
    };
    if constexpr (RV > 0) {
#pragma unroll
        for (int i = 0; i < RV; i++)
            if (tid + 256 * i < n4) put(tid + 256 * i, v[i]);
    } else {
        for (int i = tid; i < n4; i += 256) put(i, r[i]);
    }
    if (tid == 0) inv[row] = ldexpf(1.f, -sh);
}

__device__ __forceinline__ float h2f(unsigned bits) {
    return (float)__builtin_bit_cast(_Float16, (unsigned short)(bits & 0xFFFFu));
}

// Both halves with subnormals made zero: the reference's layout reads one as
// m * 2^-136 (f16_ref), which no sum here can hold, ggml's as IEEE does.
__device__ __forceinline__ unsigned f16x2_no_subnormal(unsigned h) {
    const unsigned lo = (h & 0x7C00u) ? h & 0xFFFFu : 0u;
    return (h & 0x7C000000u) ? lo | (h & 0xFFFF0000u) : lo;
}

// ---------------------------------------------------------------------------
// Expert tile GEMM.  Work items are (tile, row block) pairs, tile-major (ncb =
// F / (64 NA) row blocks of columns for MODE 0, H / (128 NA) of rows for MODE 1;
// NA by mf_two_blocks, from the tiles that the dispatch made),
// the tiles heaviest first.  The grid is persistent (two workgroups of four
// waves per CU): workgroup b starts with item b, then takes tickets from the
// counter ntiles[1 + MODE] (zeroed by k_dispatch): item grid + ticket, the
// ticket taken two steps before the end of the current item (taken an item
// ahead, with the next item's lists copied to LDS meanwhile, T = 512 was 9%
// slower: with little more than one item per workgroup the second ones then go
// to the workgroups with the heaviest first).  Items thus go out heaviest first
// to whichever workgroup is about to be free (greedy list scheduling); a fixed stride over the items left the workgroups that drew
// heavy items 30% busier than the mean.
//
// Wave w owns NA 32-row blocks of weight rows and all of the tile's pairs, in NB
// 32-pair sub-tiles.  MODE 0: NA = 2 gate and up of 32 columns, one block each;
// NA = 1 gate (rows 0..15) and up (16..31) of 16 columns; either way SwiGLU pairs
// accumulators of one lane.  MODE 1: 32 NA down rows.  X rows are tokens (ttok)
// of x in MODE 0, pairs (tpair) of act in MODE 1; xinv[X row] undoes the row's
// fp16 scaling.
//
// K advances 64 columns (two Q4_K sub-blocks) a step.  Packed quants (32 bytes
// a row), headers and activation rows are copied directly to LDS (tbq_dma.hpp)
// into rings of D steps, with counted waits: a tile of few pairs is bound by
// the weights' latency, and D = 5 at one sub-tile keeps four steps (32 KiB) of
// weights in flight per workgroup; D = 3 where four sub-tiles' activations
// need the room.  Quants run one step ahead of the activations, so a lane reads
// its rows' bytes during the step before and its first MFMA finds the fragment
// made.  Each lane dequantises its own rows' fragments between the MFMAs
// of the fragments before (half h = lane / 32 covers columns 32 h .. + 31 of a
// step, one sub-block; the k order inside a step is the same for both
// operands).  LDS rows are swizzled by the copies' source addresses: slot seg
// ^ swizzle(row), so column reads spread over all banks.
//
// Against one 8-wave workgroup per CU whose lanes loaded their own rows' bytes
// (a cache line per lane and load), whole layer of 128 experts, top 8, H 2048, F
// 768, in us: 40 tokens 150 -> 145, 512 Zipf-skewed 164 -> 155, 900 even 238 -> 229,
// 1999 of ggml's layout 427 -> 374; 8% over 300 random layers, 11 of them slower by
// more than 1% (at most 7%, nearly all of H = 1536).  Left at 512 tokens: 183 + 140
// MB read (35 + 27 us at the copy rate) while the heaviest experts' tiles, which
// set the end, wait for the same memory; at NA = 2 the two GEMMs took 127 us,
// without copies 88, without the dequantisation as well 71.
// ---------------------------------------------------------------------------
constexpr int MF_WAVES = 4, MF_ROWS = 64 * MF_WAVES;   // rows at two blocks per wave
constexpr int mf_depth(int nb) { return nb == 1 ? 5 : nb == 2 ? 4 : 3; }
// header slots: at D = 5 the next super-block's copy is issued in the step that
// reads the current one's, at D <= 4 after it
constexpr int mf_hdrs(int nb) { return mf_depth(nb) > 4 ? 2 : 1; }
constexpr int mf_lds(int nb) { return mf_hdrs(nb) * MF_ROWS * 16 + mf_depth(nb) * (MF_ROWS * 32 + nb * 32 * 128); }
// behind the rings: this item's pair ids and row scales, and the next item
struct MfLists {
    int tp[PF_MT];
    float xsc[PF_MT];
    int next, pad[3];
};
constexpr int MF_RING = mf_lds(4) > mf_lds(1) ? mf_lds(4) : mf_lds(1);
constexpr int MF_LDS = MF_RING + (int)sizeof(MfLists);
static_assert(mf_lds(2) <= MF_RING && mf_lds(3) <= MF_RING && 2 * MF_LDS <= 160 * 1024, "two workgroups per CU");

__device__ __forceinline__ int mf_swz8(int r) { return (r & 7) ^ ((r >> 3) & 1); }    // 128-byte rows
__device__ __forceinline__ int mf_swz2(int r) { return ((r >> 2) ^ (r >> 3)) & 1; }   // 32-byte rows

// One item for a compile-time count of sub-tiles.  w0, w1: the wave's blocks'
// rows (32 rows of rb bytes each); xrows: the tile's X rows; tp, xsc: its pair
// ids and X row scales in LDS.
template <int MODE, bool GG, int NA, int NB>
__device__ __forceinline__ void mf_item(unsigned char *lds, const uint8_t *w0, const uint8_t *w1, uint32_t rb, int K,
                                        const _Float16 *X, uint32_t xbytes, const int *xrows, const int *tp,
                                        const float *xsc, int n, int col, int ldo, float *out, int *ticket, int &nxt) {
    constexpr int D = mf_depth(NB), HD = mf_hdrs(NB), XS = NB * 32 * 128, QS = MF_WAVES * NA * 32 * 32;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31,
              lh = lane >> 5;
    unsigned char *const lh_p = lds, *const lq_p = lds + HD * MF_ROWS * 16, *const lx_p = lq_p + D * QS;
    const int nst = K >> 6;
    // activation copies: 8 rows x 8 segments each, NB per wave and step; rows
    // past the tile's pairs (id -1) copy row 0, whose results are not stored
    uint32_t xv[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const int r = 8 * (wave + MF_WAVES * i) + (lane >> 3);
        xv[i] = (uint32_t)max(xrows[r], 0) * (uint32_t)(K * 2) + 16u * ((lane & 7) ^ mf_swz8(r));
    }
    const dma_rsrc_t xr = dma_rsrc(X, xbytes);
    const dma_rsrc_t r0 = dma_rsrc(w0, 32 * rb), r1 = dma_rsrc(w1, 32 * rb);
    // quant copies: 32 rows x 2 segments each, one per block and step
    const uint32_t qv = (uint32_t)(lane >> 1) * rb + 16u + 16u * ((lane & 1) ^ mf_swz2(lane >> 1));
    // header copy: lane = row of block 0, then of block 1 (NA = 1: of the one
    // block again).  NA = 1, MODE 0: the block's rows are 16 of w0, then 16 of w1
    constexpr bool MIX = NA == 1 && MODE == 0;
    const uint8_t *hp = MIX ? (li < 16 ? w0 : w1) + (uint32_t)(li & 15) * rb
                            : (lane < 32 || NA == 1 ? w0 : w1) + (uint32_t)li * rb;
    const uint8_t *qp = (lane < 32 ? w0 : w1) + (uint32_t)((lane >> 1) & 15) * rb + 16 + 16 * ((lane & 1) ^ mf_swz2(lane >> 1));
    const uint32_t ax = lds_addr(lx_p) + wave * 1024, aq = lds_addr(lq_p) + wave * (NA * 1024), ah = lds_addr(lh_p) + wave * 1024;
    auto copy_x = [&](int slot, int step) {
#pragma unroll
        for (int i = 0; i < NB; i++) dma16(ax + slot * XS + MF_WAVES * i * 1024, xv[i], xr, min(step, nst - 1) * 128);
    };
    auto copy_q = [&](int slot, int step) {   // steps past the end copy bytes of the last super-block again, never read
        const uint32_t so = (min(step, nst - 1) >> 2) * 144 + (step & 3) * 32;
        if constexpr (MIX) dma16_ptr(aq + slot * QS, qp + so);
        else dma16(aq + slot * QS, qv, r0, so);
        if constexpr (NA == 2) dma16(aq + slot * QS + 1024, qv, r1, so);
    };
    auto copy_h = [&](int sb) { dma16_ptr(ah + sb % HD * (MF_ROWS * 16), hp + min(sb, (nst >> 2) - 1) * 144); };

    f32x16 acc[NA][NB];
#pragma unroll
    for (int b = 0; b < NA; b++)
#pragma unroll
        for (int t = 0; t < NB; t++) acc[b][t] = f32x16{};

    constexpr int QR = GG ? 2 : 1;   // 16-byte quant reads per lane and step
    u32x4 hd[NA], q[NA][QR];
    uint32_t mhi[NA];
    f16x2 S16[NA], C[NA];
    f16x8 a[2][NA];
    const int wrow = wave * (32 * NA) + li, qsw = mf_swz2(li);
    // the raw bytes of step s (of its super-block), whose quants sit in slot
    auto raw = [&](int s, int slot, int sb) {
#pragma unroll
        for (int b = 0; b < NA; b++) {
            const unsigned char *qrow = lq_p + slot * QS + (wrow + 32 * b) * 32;
            if (s == 0) {
                hd[b] = *reinterpret_cast<const u32x4 *>(lh_p + sb % HD * (MF_ROWS * 16) + (wave * 64 + 32 * b + li) * 16);
                if constexpr (!GG) {
                    // the reference's mins of sub-blocks 4..7 are quant bytes 0..3 (layer4/tb_gguf.c:163-168)
                    mhi[b] = *reinterpret_cast<const uint32_t *>(qrow + 16 * qsw);
                    hd[b].x = f16x2_no_subnormal(hd[b].x);
                }
            }
            if constexpr (GG) {
                q[b][0] = *reinterpret_cast<const u32x4 *>(qrow + 16 * qsw);
                q[b][QR - 1] = *reinterpret_cast<const u32x4 *>(qrow + 16 * (qsw ^ 1));
            } else {
                q[b][0] = *reinterpret_cast<const u32x4 *>(qrow + 16 * (lh ^ qsw));
            }
        }
    };
    // 16 S and C = -16 S - M of the lane's sub-block 2 s + lh
    auto scales = [&](int s) {
#pragma unroll
        for (int b = 0; b < NA; b++) {
            const int jb = 16 * (s & 1) + 8 * lh;
            uint32_t sc, mn;
            if constexpr (GG) {   // ggml's get_scale_min_k4
                const uint32_t y = hd[b].y >> jb, z = hd[b].z >> jb, w = hd[b].w >> jb;
                sc = s < 2 ? y & 63 : (w & 15) | ((y >> 2) & 48);
                mn = s < 2 ? z & 63 : ((w >> 4) & 15) | ((z >> 2) & 48);
            } else {
                sc = ((s < 2 ? hd[b].y : hd[b].w) >> jb) & 63;
                mn = ((s < 2 ? hd[b].z : mhi[b]) >> jb) & 63;
            }
            const float S = h2f(hd[b].x) * (float)sc, M = h2f(hd[b].x >> 16) * (float)mn;
            const _Float16 s16 = (_Float16)(16.f * S), cc = (_Float16)(-(float)s16 - M);
            S16[b] = f16x2{s16, s16};
            C[b] = f16x2{cc, cc};
        }
    };
    const int gsh0 = 6 - 4 * lh, gsh1 = 2 + 4 * lh;   // ggml: nibble lh of bytes 0, 2 and of bytes 1, 3 to bit 6
    // fragment kk: the weights of columns 32 lh + 8 kk .. + 7 of the step.
    // Reference layout: weights 2i, 2i + 1 in the nibbles of quant byte i, a
    // byte spread into the two halves by one 24-bit multiply.  ggml's: weight i
    // of sub-block lh in nibble lh of byte i; one shift and one v_bitop3 take
    // bytes 0 and 2 (then 1 and 3) of a dword, so k runs 0, 2, 1, 3 in every
    // four columns, an order in which the activation rows are stored
    // (launch_rows_f16).
    auto frag = [&](int b, int kk) {
        unsigned w[4];
        if constexpr (GG) {
            const u32x4 v = q[b][kk >> 1 & (QR - 1)];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const unsigned d = i < 2 ? (kk & 1 ? v.z : v.x) : (kk & 1 ? v.w : v.y);
                // nibble lh of bytes 0 and 2 (i even) or 1 and 3 to bits 6..9 and 22..25
                const unsigned y = i & 1 ? d >> gsh1 : d << gsh0;
                const unsigned t = __builtin_amdgcn_bitop3_b32(y, 0x03C003C0u, 0x3C003C00u, 0xEA);
                w[i] = __builtin_bit_cast(unsigned, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, t), S16[b], C[b]));
            }
        } else {
            const u32x4 v = q[b][0];
            const unsigned qd = kk == 0 ? v.x : kk == 1 ? v.y : kk == 2 ? v.z : v.w;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const unsigned y = (qd >> (8 * i)) & 0xFFu;
                const unsigned t = __builtin_amdgcn_bitop3_b32(__umul24(y, 0x40040u), 0x03C003C0u, 0x3C003C00u, 0xEA);   // (a & b) | c
                w[i] = __builtin_bit_cast(unsigned, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, t), S16[b], C[b]));
            }
        }
        return __builtin_bit_cast(f16x8, u32x4{w[0], w[1], w[2], w[3]});
    };

    // Step i issues the activations of step i + D - 1 and the quants (and at a
    // super-block's first step the header) of step i + D.  Before step s the
    // activations of step s and the quants of step s + 1 must have landed:
    // everything issued up to step s - D + 1, so the D - 2 steps issued after
    // it may stay in flight (any other memory operation in between only makes
    // the wait longer).
    copy_x(0, 0);
    copy_q(0, 0);
    copy_h(0);
    copy_q(1, 1);
#pragma unroll
    for (int i = 1; i <= D - 2; i++) {
        copy_x(i, i);
        copy_q(i + 1, i + 1);
        if (i + 1 == 4) copy_h(1);
    }
    dma_wait_barrier_n<(D - 2) * (NB + NA) + (D >= 5 ? 1 : 0)>();
    raw(0, 0, 0);
    scales(0);
#pragma unroll
    for (int b = 0; b < NA; b++) a[0][b] = frag(b, 0);
    // step 0 copies into quant slot 0, and at D = 4 into the only header slot:
    // rows this wave alone reads, whose first reads the step's copies must not pass
    lds_read_wait();
    int xs = 0, qs = 0;   // slots of this step's activations and quants
    const unsigned char *const xb0 = lx_p + li * 128;
    const int xsw = mf_swz8(li);
    for (int s0 = 0; s0 < nst; s0 += 4) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            copy_x(xs == 0 ? D - 1 : xs - 1, s0 + s + D - 1);
            copy_q(qs, s0 + s + D);
            if ((s + D) % 4 == 0) copy_h((s0 + s + D) >> 2);
            const int qn = qs == D - 1 ? 0 : qs + 1;
            if (s == 2 && s0 + 4 >= nst && tid == 0) nxt = atomicAdd(ticket, 1) + (int)gridDim.x;
            const unsigned char *xb = xb0 + xs * XS;
            f16x8 bf[2][NB];
#pragma unroll
            for (int t = 0; t < NB; t++) bf[0][t] = *reinterpret_cast<const f16x8 *>(xb + t * 4096 + 16 * ((4 * lh) ^ xsw));
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                if (kk < 3) {
#pragma unroll
                    for (int t = 0; t < NB; t++)
                        bf[(kk + 1) & 1][t] = *reinterpret_cast<const f16x8 *>(xb + t * 4096 + 16 * ((4 * lh + kk + 1) ^ xsw));
#pragma unroll
                    for (int b = 0; b < NA; b++) a[(kk + 1) & 1][b] = frag(b, kk + 1);
                    if (kk == 2) raw((s + 1) & 3, qn, (s0 + s + 1) >> 2);
                } else {
                    scales((s + 1) & 3);
#pragma unroll
                    for (int b = 0; b < NA; b++) a[0][b] = frag(b, 0);
                }
#pragma unroll
                for (int t = 0; t < NB; t++)
#pragma unroll
                    for (int b = 0; b < NA; b++)
                        acc[b][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[kk & 1][b], bf[kk & 1][t], acc[b][t], 0, 0, 0);
                // keep the decode between the MFMAs: run ahead, it spills in the loop
                // (the few registers that still do hold per-item state)
                if constexpr (!GG && NA == 2 && NB >= 3) {
#pragma unroll
                    for (int i = 0; i < NA * NB; i++) {
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x2, 7, 0);
                    }
                }
            }
            // steps s - D + 3 .. s (of the unrolled four) stay in flight
            constexpr int base = (D - 2) * (NB + NA);
            bool hdr = false;
#pragma unroll
            for (int i = 0; i < D - 2; i++) hdr = hdr || (s - i + D + 4) % 4 == 0;
            if (hdr) dma_wait_barrier_n<base + 1>();
            else dma_wait_barrier_n<base>();
            xs = xs == D - 1 ? 0 : xs + 1;
            qs = qn;
        }
    }
    // accumulator register r of lane l: row 8(r/4) + 4(l/32) + r%4 of the
    // 32-row block, pair 32 t + l % 32 of the tile
#pragma unroll
    for (int t = 0; t < NB; t++) {
        if (32 * t + li >= n) continue;
        const float sc = xsc[32 * t + li];
        float *o = out + (long long)tp[32 * t + li] * ldo + col + 4 * lh;
        if constexpr (MODE == 0) {
#pragma unroll
            for (int g4 = 0; g4 < 2 * NA; g4++) {   // NA = 1: the up rows are the block's second half
                float v[4];
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const float g = acc[0][t][4 * g4 + c] * sc, u = acc[NA - 1][t][4 * g4 + c + (NA == 1 ? 8 : 0)] * sc;
                    v[c] = g * u * __builtin_amdgcn_rcpf(1.0f + __expf(-g));
                }
                *reinterpret_cast<float4 *>(o + 8 * g4) = make_float4(v[0], v[1], v[2], v[3]);
            }
        } else {
#pragma unroll
            for (int b = 0; b < NA; b++)
#pragma unroll
                for (int g4 = 0; g4 < 4; g4++)
                    *reinterpret_cast<float4 *>(o + 32 * b + 8 * g4) =
                        make_float4(acc[b][t][4 * g4] * sc, acc[b][t][4 * g4 + 1] * sc, acc[b][t][4 * g4 + 2] * sc,
                                    acc[b][t][4 * g4 + 3] * sc);
        }
    }
}

// Row blocks per wave, by the items that two blocks would make (a) for the slots
// (two workgroups per CU) and the pairs per tile (p).  Two read the activations
// half as often and decode between twice the MFMAs; one halves the items, which
// shortens the last round and fills a chip with few of them.  Two are better
// from 40 (down: 32) pairs per tile on, but not where few items, or a last round
// nearly empty, leave slots idle; below that they gain where one round is just
// filled (gate/up: up to a second round's start), and otherwise the weights'
// lines of twice the rows in flight do not stay in L2.  Fitted over 194 layers of
// H 1024..3072, F 512..1536, E 32..128, k 2..8 and 33..2048 tokens, half of them
// Zipf-skewed: 0.5% from the best choice for each, one block everywhere 1.5%,
// two everywhere 5.9% (2048 x 768, 128 experts, 900 tokens: 246 us with one, 227
// with two; 700 Zipf-skewed: 198 and 213).  Over 120 other layers 4 were more
// than 1% slower than on the 8-wave workgroups of 256 rows before these kernels.
template <int MODE>
__device__ __forceinline__ bool mf_two_blocks(int a, int pairs, int tiles, int slots) {
    if (a > slots && 10 * a < (MODE == 0 ? 13 : 15) * slots) return false;
    if constexpr (MODE == 0) {
        if (pairs >= 40 * tiles) return 5 * a >= 4 * slots;
        return 8 * a >= 7 * slots && 5 * a <= 8 * slots;
    } else {
        if (pairs >= 32 * tiles) return 2 * a >= slots && (2 * a < 5 * slots || pairs >= 64 * tiles);
        return 10 * a >= 9 * slots && a <= slots;
    }
}

template <int MODE, bool GG>
__global__ __launch_bounds__(64 * MF_WAVES) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_moe_f16(
    const uint8_t *__restrict__ W0, const uint8_t *__restrict__ W1, const _Float16 *__restrict__ X, int x_rows,
    const float *__restrict__ xinv, const int *__restrict__ tpair, const int *__restrict__ ttok,
    const PfTile *__restrict__ tiles, int *__restrict__ ntiles, int pairs, int slots, int H, int F, float *__restrict__ out) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char mf_lds_p[];
    const int K = MODE == 0 ? H : F, nt = *ntiles;
    const uint32_t rb = (uint32_t)(K >> 8) * 144u;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    MfLists &ml = *reinterpret_cast<MfLists *>(mf_lds_p + MF_RING);
    const dma_rsrc_t sr = dma_rsrc(xinv, (uint32_t)x_rows * 4u);
    const int lane = threadIdx.x & 63;
    const int n2 = MODE == 0 ? F / (MF_ROWS / 2) : H / MF_ROWS;   // row blocks at NA = 2
    auto run = [&](auto na) {
        constexpr int NA = decltype(na)::value;
        const int ncb = NA == 1 ? 2 * n2 : n2, nitems = nt * ncb;
        for (int item = blockIdx.x; item < nitems;) {
            const int tix = item / ncb, cb = item % ncb;
            const PfTile tl = tiles[tix];
            const int *xrows = (MODE == 0 ? ttok : tpair) + (long long)tix * PF_MT;
            // the tile's pair ids and row scales to LDS for the epilogue (rows
            // past its pairs: row 0's scale, not used)
            if (wave < 2) {
                const uint32_t r = (uint32_t)max(xrows[64 * wave + lane], 0);
                dma4(lds_addr(ml.tp) + 256 * wave, 4u * (64 * wave + lane), dma_rsrc(tpair + (long long)tix * PF_MT, PF_MT * 4));
                dma4(lds_addr(ml.xsc) + 256 * wave, 4u * r, sr);
            }
            const int e = __builtin_amdgcn_readfirstlane(tl.e), n = __builtin_amdgcn_readfirstlane(tl.n);
            const int col = (cb * MF_WAVES + wave) * (MODE == 0 ? 16 : 32) * NA;
            const uint8_t *w0 = W0 + ((long long)e * (MODE == 0 ? F : H) + col) * rb;
            const uint8_t *w1 = MODE == 0 ? W1 + ((long long)e * F + col) * rb : w0 + 32ll * rb;
            int nxt = 0;
            auto body = [&](auto nb) {
                mf_item<MODE, GG, NA, decltype(nb)::value>(mf_lds_p, w0, w1, rb, K, X, (uint32_t)x_rows * (uint32_t)(K * 2),
                                                       xrows, ml.tp, ml.xsc, n, col, MODE == 0 ? F : H, out,
                                                       ntiles + 1 + MODE, nxt);
            };
            switch ((n + 31) / 32) {   // uniform
            case 1: body(PfSub<1>{}); break;
            case 2: body(PfSub<2>{}); break;
            case 3: body(PfSub<3>{}); break;
            default: body(PfSub<4>{}); break;
            }
            // every wave is past its last read of the rings and lists when all
            // have passed this barrier
            if (threadIdx.x == 0) ml.next = nxt;
            dma_wait_barrier();
            item = __builtin_amdgcn_readfirstlane(ml.next);
        }
    };
    if (mf_two_blocks<MODE>(nt * n2, pairs, nt, slots)) run(PfSub<2>{});   // uniform
    else run(PfSub<1>{});
}

// ---------------------------------------------------------------------------
// int8 MFMA variant (TBQ_MOE_I8): Q8_K-quantised activations against the
// Q4_K nibbles on v_mfma_i32_32x32x32_i8.
//
// Activations.  k_rows_q8 quantises rows of n floats per 256-element block
// as the Q8_K activation quantiser (tbo_quantize_q8k): d = max|x| / 127,
// q1 = rint(x / d) clamped to +-127 (computed as x * (1/d)).  For the
// prefill it adds a second int8 level for the residual, q2 = rint((x - q1 d)
// * 256 / d) clamped to +-127, so x = d (q1 + q2 / 256) to 2^-16 of the
// block's max: with the first level alone the layer's MoE delta lands 1-2%
// from the fp32 reference on N(0,1) activations (the SwiGLU outputs are
// heavy-tailed), above the 1e-2 bound.  Each level keeps Q8_K's 16-element
// sums (fp16: |sum| <= 2032 is exact).  The int8 rows store the elements of
// every 16-element group in the order 0,2,4,6,1,3,5,7,8,10,12,14,9,11,13,15:
// the order in which one Q4_K quant dword unpacks with two AND masks and a
// shift (the reference's layout puts weights 2i and 2i+1 in the low and high
// nibbles of byte i, layer4/tb_gguf.c:148-180).  The sum over k does not
// depend on the order, which both operands share.
//
// Weights.  Per 32-weight sub-block j of a row the 6-bit scale is split
// sc_j = 8 a_j + b_j (a_j, b_j < 8) and folded into the int8 operands q a_j
// and q b_j (<= 105), so int8 MFMAs accumulate a whole super-block in int32
// with no per-output scaling: four per sub-block, (q a, q b) x (q1, q2).  The
// mins enter once per super-block through two fp16 MFMAs of the row's m_j
// (each twice) against the pair's 16-element sums of q1 and q2 (exact
// integers in fp32).  Per super-block and output, with F_l = 8 acc_a,l +
// acc_b,l and M_l = sum_j m_j S_j,l:
//   y += dx (d (F_1 + F_2 / 256) - dmin (M_1 + M_2 / 256))
// with d, dmin the row's fp16 super-block scales (a1's reading of the
// scale bytes) and dx the pair's block scale; fp32 accumulation.  The
// activations are the MFMAs' A operand and the weights B, so a lane's
// accumulators all belong to its own weight row (its d and dmin, no lane
// exchange per flush) and to 16 pairs, whose block scales are staged in LDS
// per item.
//
// Items: (tile, 32-pair sub-tile, row block), on an 8-wave workgroup (32 weight
// rows per wave, MODE 0 rows i < 16 gate and i >= 16 up of column 16 w + i %
// 16); SwiGLU takes a gate row's up partner from lane li + 16.  Packed rows and
// activations are copied directly to LDS (tbq_dma.hpp), a super-block a step:
// weights two steps ahead into the wave's own rows of a stage (one ahead where
// K > 2048 leaves room for two stages only), activations one ahead, one barrier
// a step.  Lanes that loaded their own rows' bytes touched a cache line per lane
// and load, five loads per 128 columns.  At 512 Zipf-skewed tokens of E = 128, k
// = 8, H = 2048, F = 768 the gate/up launch went 168 -> 146 us and the down
// launch 82 -> 76, at 1999 tokens the layer 750 -> 701.  The rest is the SIMDs'
// own time: two 8-bit levels times two scale parts make four integer MFMAs per
// fragment, their operands some 330 vector instructions per super-block, at two
// waves per SIMD.
// ---------------------------------------------------------------------------
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr int I8_MT = 32;                 // pairs per item

// Position of element e (< 16) of a 16-element group in the stored order.
__device__ __forceinline__ int q8_pos(int e) {
    const int h = e & 8, r = e & 7;
    return h + ((r & 1) << 2) + (r >> 1);
}

// One wave per 256-element block of a float array (blocks of 256
// consecutive floats).  BLOCKS = false: the prefill operand form of a row of
// n floats (int8 levels [row][2][n] in the MFMA order above, block scales
// [row][n/256], fp16 group sums [row][2][n/16]); BLOCKS = true: the
// reference's Q8_K block of the first level only (layer4/tb_gguf.c:281-288:
// f32 d at 0, int8 qs[256] in element order at 4, int16 bsums[16] at 260;
// 292 bytes), written to q8 with n, dq and bs16 unused.
template <bool BLOCKS>
__global__ __launch_bounds__(256) void k_rows_q8(const float *__restrict__ in, int n, long long nblocks,
                                                 int8_t *__restrict__ q8, float *__restrict__ dq,
                                                 _Float16 *__restrict__ bs16) {
    __shared__ int8_t stage[4][2][256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long long b0 = (long long)blockIdx.x * 4 + wave;
    const bool valid = b0 < nblocks;   // past the end: redo the last block, store nothing
    const long long b = valid ? b0 : nblocks - 1;
    const float4 v = reinterpret_cast<const float4 *>(in + b * 256)[lane];
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    amax = wave_max(amax);
    const float d = amax / 127.0f;
    const float id = d > 0.0f ? 1.0f / d : 0.0f;
    const float xs[4] = {v.x, v.y, v.z, v.w};
    int s1 = 0, s2 = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float r = rintf(xs[i] * id);
        r = fminf(fmaxf(r, -127.0f), 127.0f);
        const int q1 = (int)r;
        float r2 = rintf((xs[i] - r * d) * (id * 256.0f));
        r2 = fminf(fmaxf(r2, -127.0f), 127.0f);
        const int q2 = (int)r2;
        s1 += q1;
        s2 += q2;
        const int e = 4 * (lane & 3) + i;   // element within the lane's 16-element group
        const int pos = 16 * (lane >> 2) + (BLOCKS ? e : q8_pos(e));
        stage[wave][0][pos] = (int8_t)q1;
        stage[wave][1][pos] = (int8_t)q2;
    }
    // the group's sums over its four lanes
    s1 += __shfl_xor(s1, 1);
    s1 += __shfl_xor(s1, 2);
    s2 += __shfl_xor(s2, 1);
    s2 += __shfl_xor(s2, 2);
    __syncthreads();
    if (!valid) return;
    if constexpr (BLOCKS) {
        uint8_t *blk = reinterpret_cast<uint8_t *>(q8) + b * 292;   // 4-byte aligned
        reinterpret_cast<int *>(blk + 4)[lane] = reinterpret_cast<const int *>(stage[wave][0])[lane];
        if ((lane & 3) == 0) reinterpret_cast<int16_t *>(blk + 260)[lane >> 2] = (int16_t)s1;
        if (lane == 0) *reinterpret_cast<float *>(blk) = d;
    } else {
        const int nb = n / 256;
        const long long row = b / nb, blk = b % nb;
        int8_t *qr = q8 + row * 2 * n + blk * 256;
        reinterpret_cast<int *>(qr)[lane] = reinterpret_cast<const int *>(stage[wave][0])[lane];
        reinterpret_cast<int *>(qr + n)[lane] = reinterpret_cast<const int *>(stage[wave][1])[lane];
        if ((lane & 3) == 0) {
            _Float16 *sr = bs16 + row * 2 * (n / 16) + blk * 16 + (lane >> 2);
            sr[0] = (_Float16)(float)s1;
            sr[n / 16] = (_Float16)(float)s2;
        }
        if (lane == 0) dq[b] = d;
    }
}

template <int MODE, int NS>
__global__ __launch_bounds__(PF_THREADS) void k_moe_i8(const uint8_t *__restrict__ W0, const uint8_t *__restrict__ W1,
                                                       const int8_t *__restrict__ X, const float *__restrict__ XD,
                                                       const _Float16 *__restrict__ XB, int x_rows,
                                                       const int *__restrict__ tpair, const int *__restrict__ ttok,
                                                       const PfTile *__restrict__ tiles, const int *__restrict__ ntiles,
                                                       int ncb, int H, int F, float *__restrict__ out) {
    constexpr int K = NS * PF_KC;
    constexpr int NSB = K / 256;
    constexpr int NQ = PF_MT / I8_MT;   // sub-tiles per tile, as k_dispatch counts them
    static_assert(I8_MT == 32, "sub-tile classes");
    constexpr int WS = PF_WAVES * 32 * 144, XS = 2 * I8_MT * 256;   // a stage: 256 packed rows; 32 rows of two levels, two halves
    constexpr int D = NSB <= 8 ? 3 : 2;   // weight stages that fit beside the group sums
    __shared__ __attribute__((aligned(16))) unsigned char lds[D * WS + 2 * XS + I8_MT * (K / 4) + I8_MT * 4 * NSB + I8_MT * 8];
    static_assert(sizeof(lds) <= 160 * 1024, "LDS");
    unsigned char *const lx_p = lds + D * WS;
    _Float16 *const xb_s = reinterpret_cast<_Float16 *>(lx_p + 2 * XS);          // [I8_MT][K/8] group sums
    float *const dx_s = reinterpret_cast<float *>(xb_s + I8_MT * (K / 8));       // [NSB][I8_MT] block scale of pair slot
    int *const po_s = reinterpret_cast<int *>(dx_s + NSB * I8_MT), *const px_s = po_s + I8_MT;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31, lh = lane >> 5;
    constexpr int rb = NSB * 144;
    const dma_rsrc_t xrs = dma_rsrc(X, (uint32_t)(x_rows * 2 * K));
    const uint32_t aw = lds_addr(lds) + wave * (32 * 144), ax = lds_addr(lx_p) + wave * 1024;
    unsigned char *const lw_p = lds + wave * (32 * 144) + li * 144;
    // Items are the sub-tiles that exist, tiles in their heaviest-first order (c[i]
    // tiles of NQ - i sub-tiles each): with NQ item slots per tile, the stride
    // over mostly empty slots left some workgroups twice the mean's items.  E = 128,
    // k = 8, H = 2048, F = 768 (layer): 512 tokens, Zipf routing 370 -> 279 us; 40
    // tokens 329 -> 187; 1999 tokens, tiles nearly full, 814 -> 750.
    int c[NQ], nsub = 0;
#pragma unroll
    for (int i = 0; i < NQ; i++) {
        c[i] = ntiles[3 + i];
        nsub += (NQ - i) * c[i];
    }
    const int nitems = nsub * ncb;
    for (int item = blockIdx.x; item < nitems; item += gridDim.x) {
        const int cb = item % ncb;
        int s = item / ncb, tix = 0, qt = 0;
        bool found = false;
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            if (!found && s < (NQ - i) * c[i]) {
                tix += s / (NQ - i);
                qt = s % (NQ - i);
                found = true;
            } else if (!found) {
                tix += c[i];
                s -= (NQ - i) * c[i];
            }
        }
        const PfTile tl = tiles[tix];
        const int n = min(tl.n - I8_MT * qt, I8_MT);   // pairs of this sub-tile (uniform, > 0)
        const int *xrows = (MODE == 0 ? ttok : tpair) + tix * PF_MT + I8_MT * qt;
        // activation copies: slot tid >> 4 of a 128-column half, its 16 segments
        // (two levels of eight) at segment ^ (slot & 15); slots past the tile's
        // pairs (id -1) copy row 0, whose results are not stored
        const int xsg = (tid & 15) ^ ((tid >> 4) & 15);
        const uint32_t xv = (uint32_t)((max(xrows[tid >> 4], 0) * 2 + (xsg >> 3)) * K + 16 * (xsg & 7));
        if (tid < I8_MT) {
            po_s[tid] = tpair[tix * PF_MT + I8_MT * qt + tid];
            px_s[tid] = xrows[tid];
        }
        // weight copies: the wave's 32 rows of 144 bytes as 288 segments of 16
        const uint8_t *r0, *r1;   // rows 0..15 and 16..31
        if (MODE == 0) {
            const long long ro = ((long long)tl.e * F + cb * PF_COLS + 16 * wave) * rb;
            r0 = W0 + ro;
            r1 = W1 + ro;
        } else {
            r0 = W0 + ((long long)tl.e * H + cb * PF_ROWS + 32 * wave) * rb;
            r1 = r0 + 16 * rb;
        }
        const uint8_t *wp[5];
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const int g = min(64 * i + lane, 287), row = g / 9;
            wp[i] = (row < 16 ? r0 : r1) + (row & 15) * rb + 16 * (g % 9);
        }
        auto copy_w = [&](int st, int sb) {
#pragma unroll
            for (int i = 0; i < 4; i++) dma16_ptr(aw + st * WS + 1024 * i, wp[i] + sb * 144);
            if (lane < 32) dma16_ptr(aw + st * WS + 4096, wp[4] + sb * 144);
        };
        auto copy_x = [&](int st, int sb) {
            dma16(ax + st * XS, xv, xrs, sb * 256);
            dma16(ax + st * XS + XS / 2, xv, xrs, sb * 256 + 128);
        };
        copy_w(0, 0);
        copy_x(0, 0);
        if (D == 3 && NSB > 1) copy_w(1, 1);
        __syncthreads();   // po_s / px_s written
        // the pair slots' block scales and group sums into LDS (ordered
        // before the first flush by chunk 0's barrier): the flushes then
        // wait for no global load
        if (tid < NSB * I8_MT) {
            const int ps = tid % I8_MT, sbi = tid / I8_MT, xrw = px_s[ps];
            dx_s[tid] = xrw >= 0 ? XD[(long long)xrw * NSB + sbi] : 0.f;
        }
        {
            constexpr int SEG = K / 64;   // 16-byte segments of a slot's K / 8 halves
#pragma unroll
            for (int i0 = 0; i0 < I8_MT * SEG; i0 += PF_THREADS) {
                const int i = i0 + tid, ps = min(i / SEG, I8_MT - 1), sg = i % SEG, xrw = px_s[ps];
                const u32x4 v = *reinterpret_cast<const u32x4 *>(XB + (long long)(xrw >= 0 ? xrw : 0) * (K / 8) + 8 * sg);
                if (i < I8_MT * SEG)
                    *reinterpret_cast<u32x4 *>(xb_s + ps * (K / 8) + 8 * sg) = xrw >= 0 ? v : u32x4{0u, 0u, 0u, 0u};
            }
        }
        i32x16 aa1 = {}, ab1 = {}, aa2 = {}, ab2 = {};
        f32x16 y = {};
        // The MFMAs take the activations as the A operand and the weights as
        // B, so accumulator register r of lane l holds pair slot
        // 8(r/4) + 4(l/32) + r%4 and the lane's own weight row l%32: the
        // row's d and dmin are the lane's, the pairs' block scales come from
        // LDS.  Super-block flush:
        //   y += dx (d (F1 + F2/256) - dmin (M1 + M2/256))
        auto flush = [&](unsigned dd, unsigned wmw, int sb) {
            f16x8 am;   // this lane's row's mins m_{4 lh + i}, each twice
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const _Float16 m = (_Float16)(float)((wmw >> (8 * i)) & 63u);
                am[2 * i] = m;
                am[2 * i + 1] = m;
            }
            const _Float16 *bsr = xb_s + li * (K / 8) + 16 * sb + 8 * lh;   // pair slot li's sums
            const f16x8 b1 = *reinterpret_cast<const f16x8 *>(bsr);
            const f16x8 b2 = *reinterpret_cast<const f16x8 *>(bsr + K / 16);
            const f32x16 m1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(b1, am, f32x16{}, 0, 0, 0);
            const f32x16 m2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(b2, am, f32x16{}, 0, 0, 0);
            const float dw = f16_ref((uint16_t)(dd & 0xFFFFu)), mw = f16_ref((uint16_t)(dd >> 16));
            const float4 *dxs = reinterpret_cast<const float4 *>(dx_s + sb * I8_MT);
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float4 dx4 = dxs[2 * c + lh];   // pair slots 8c + 4lh + 0..3
                const float dxv[4] = {dx4.x, dx4.y, dx4.z, dx4.w};
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int r = 4 * c + q;
                    const float f = fmaf((float)(8 * aa2[r] + ab2[r]), 1.0f / 256.0f, (float)(8 * aa1[r] + ab1[r]));
                    const float mm = fmaf(m2[r], 1.0f / 256.0f, m1[r]);
                    y[r] = fmaf(dxv[q], fmaf(dw, f, -mw * mm), y[r]);
                }
            }
            aa1 = i32x16{};
            ab1 = i32x16{};
            aa2 = i32x16{};
            ab2 = i32x16{};
        };
        // half c of a super-block, whose packed row and activations are in LDS
        auto half = [&](const unsigned char *wr, const unsigned char *xb, int c) {
            const unsigned sw = *reinterpret_cast<const unsigned *>(wr + (c ? 12 : 4));
            const uint4 wq[2] = {*reinterpret_cast<const uint4 *>(wr + 16 + 64 * c + 16 * lh),
                                 *reinterpret_cast<const uint4 *>(wr + 16 + 64 * c + 16 * (2 + lh))};
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const uint4 q4 = wq[ks >> 1];
                const uint2 q = (ks & 1) ? make_uint2(q4.z, q4.w) : make_uint2(q4.x, q4.y);
                const unsigned sc = (sw >> (8 * (2 * (ks >> 1) + lh))) & 63u;   // sub-block 2(ks>>1) + lh
                const unsigned short a = (unsigned short)(sc >> 3), b = (unsigned short)(sc & 7u);
                const unsigned n0 = q.x & 0x0F0F0F0Fu, n1 = (q.x >> 4) & 0x0F0F0F0Fu;
                const unsigned n2 = q.y & 0x0F0F0F0Fu, n3 = (q.y >> 4) & 0x0F0F0F0Fu;
                const u16x2 va = {a, a}, vb = {b, b};
                auto mul = [](unsigned v, u16x2 f) {
                    return __builtin_bit_cast(unsigned, __builtin_bit_cast(u16x2, v) * f);
                };
                const i32x4 Aa = {(int)mul(n0, va), (int)mul(n1, va), (int)mul(n2, va), (int)mul(n3, va)};
                const i32x4 Ab = {(int)mul(n0, vb), (int)mul(n1, vb), (int)mul(n2, vb), (int)mul(n3, vb)};
                // 16-element group 4(ks >> 1) + 2 lh + (ks & 1) of the chunk
                const int sg = (4 * (ks >> 1) + (ks & 1) + 2 * lh) ^ (li & 15);
                const i32x4 bv1 = *reinterpret_cast<const i32x4 *>(xb + 16 * sg);
                const i32x4 bv2 = *reinterpret_cast<const i32x4 *>(xb + 16 * (sg ^ 8));
                aa1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(bv1, Aa, aa1, 0, 0, 0);
                ab1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(bv1, Ab, ab1, 0, 0, 0);
                aa2 = __builtin_amdgcn_mfma_i32_32x32x32_i8(bv2, Aa, aa2, 0, 0, 0);
                ab2 = __builtin_amdgcn_mfma_i32_32x32x32_i8(bv2, Ab, ab2, 0, 0, 0);
            }
        };
        for (int sb = 0; sb < NSB; sb++) {
            // this super-block's copies have landed; with three weight stages the
            // next one's weights, issued last, stay in flight
            if (D == 3 && sb + 1 < NSB) dma_wait_barrier_n<5>();
            else dma_wait_barrier();
            if (sb + 1 < NSB) copy_x((sb + 1) & 1, sb + 1);
            if (sb + D - 1 < NSB) copy_w((sb + D - 1) % D, sb + D - 1);
            const unsigned char *wr = lw_p + sb % D * WS, *xb = lx_p + (sb & 1) * XS + li * 256;
            const unsigned dd = *reinterpret_cast<const unsigned *>(wr);
            const unsigned mw = *reinterpret_cast<const unsigned *>(wr + (lh ? 16 : 8));   // mins 4..7 sit in quant bytes 0..3
            half(wr, xb, 0);
            half(wr, xb + XS / 2, 1);
            flush(dd, mw, sb);
        }
        // accumulator register r of lane l: pair slot 8(r/4) + 4 lh + r%4 of
        // the sub-tile, the wave's weight row li
        if (MODE == 0) {
            // gate (rows li < 16) and up (li + 16) of column 16 wave + li%16:
            // the up value from lane li + 16
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float uv = __shfl_xor(y[r], 16);
                const int pr = 8 * (r >> 2) + 4 * lh + (r & 3);
                if (li < 16 && pr < n) {
                    const float g = y[r];
                    const float o = g * uv * __builtin_amdgcn_rcpf(1.0f + __expf(-g));
                    out[(long long)po_s[pr] * F + cb * PF_COLS + 16 * wave + li] = o;
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int pr = 8 * (r >> 2) + 4 * lh + (r & 3);
                if (pr < n) out[(long long)po_s[pr] * H + cb * PF_ROWS + 32 * wave + li] = y[r];
            }
        }
        __syncthreads();   // the next item rewrites the pair lists and the activation buffers
    }
}

template <int MODE>
static hipError_t launch_moe_i8(int ns, unsigned nwg, hipStream_t st, const uint8_t *W0, const uint8_t *W1,
                                const int8_t *X, const float *XD, const _Float16 *XB, int x_rows, const int *tpair,
                                const int *ttok, const PfTile *tiles, const int *ntiles, int ncb, int H, int F,
                                float *out) {
#define TBQ_NS(N)                                                                                                   \
    case N:                                                                                                         \
        hipLaunchKernelGGL((k_moe_i8<MODE, N>), dim3(nwg), dim3(PF_THREADS), 0, st, W0, W1, X, XD, XB,   \
                           x_rows, tpair, ttok, tiles, ntiles, ncb, H, F, out);                                     \
        break;
    switch (ns) {
        TBQ_NS(2) TBQ_NS(4) TBQ_NS(6) TBQ_NS(8) TBQ_NS(12) TBQ_NS(16) TBQ_NS(24) TBQ_NS(32)
    default:
        return hipErrorNotSupported;
    }
#undef TBQ_NS
    return hipGetLastError();
}

size_t prefill_workspace_bytes(int T, int k, int E, int H, int F) {
    const size_t P = (size_t)T * k;
    const size_t max_tiles = (P + PF_MT - 1) / PF_MT + E;
    auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
    return up(P * 4) + up(max_tiles * sizeof(PfTile)) + 256 + 2 * up(max_tiles * PF_MT * 4) + up(P * F * 2) +
           up((size_t)T * H * 2) + up(P * 4) + up((size_t)T * 4);
}

// Persistent grid of the int8 expert GEMMs: one workgroup per CU (130 to 157 KiB
// of its LDS: a second would only queue behind the first), never more than the
// item count bound.
static unsigned pf_grid(unsigned max_items) {
    const unsigned g = (unsigned)(tbq_cu_count() > 0 ? tbq_cu_count() : 256);
    return max_items < g ? max_items : g;
}

template <int MODE, bool GG>
static hipError_t launch_moe_f16(const MoeArgs &a, int max_tiles, hipStream_t st, const uint8_t *W0, const uint8_t *W1, const _Float16 *X,
                                 int x_rows, const float *xinv, const int *tpair, const int *ttok, const PfTile *tiles,
                                 int *ntiles, int H, int F, float *out) {
    // more than 64 KiB of dynamic LDS is opted into once per kernel
    static const hipError_t attr =
        hipFuncSetAttribute((const void *)k_moe_f16<MODE, GG>, hipFuncAttributeMaxDynamicSharedMemorySize, MF_LDS);
    if (attr != hipSuccess) return attr;
    const unsigned slots = 2u * (unsigned)(tbq_cu_count() > 0 ? tbq_cu_count() : 256);   // two workgroups per CU
    const unsigned items = 2u * (unsigned)max_tiles * (unsigned)(MODE == 0 ? F / (MF_ROWS / 2) : H / MF_ROWS);   // at NA = 1
    hipLaunchKernelGGL((k_moe_f16<MODE, GG>), dim3(items < slots ? items : slots), dim3(64 * MF_WAVES), MF_LDS, st, W0, W1, X,
                       x_rows, xinv, tpair, ttok, tiles, ntiles, a.T * a.k, (int)slots, H, F, out);
    return hipGetLastError();
}

// K values the MFMA kernel is instantiated for (K = 128 * NS).
bool gemm_k_supported(int K) {
    const int n = K / PF_KC;
    return K % 256 == 0 && (n == 2 || n == 4 || n == 6 || n == 8 || n == 12 || n == 16 || n == 24 || n == 32);
}

// int8 mode workspace: the dispatch lists of the fp16 mode, then the
// two-level Q8_K activations of x ([T][2][H] int8, block scales [T][H/256],
// fp16 16-element sums [T][2][H/16]) and of the SwiGLU output ([P][2][F],
// the same three).
size_t prefill_i8_workspace_bytes(int T, int k, int E, int H, int F) {
    const size_t P = (size_t)T * k;
    const size_t max_tiles = (P + PF_MT - 1) / PF_MT + E;
    auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
    return up(P * 4) + up(max_tiles * sizeof(PfTile)) + 256 + 2 * up(max_tiles * PF_MT * 4) +
           up((size_t)T * H * 2) + up((size_t)T * H / 256 * 4) + up((size_t)T * H / 16 * 4) + up(P * F * 2) +
           up(P * F / 256 * 4) + up(P * F / 16 * 4);
}

// Rows of n floats (n a multiple of 256) to Q8_K blocks in the int8 MFMA
// operand order (k_rows_q8).
hipError_t launch_rows_q8(const float *in, long long rows, int n, int8_t *q8, float *dq, _Float16 *bs16,
                          hipStream_t st) {
    const long long nb = rows * (n / 256);
    hipLaunchKernelGGL(k_rows_q8<false>, dim3((unsigned)((nb + 3) / 4)), dim3(256), 0, st, in, n, nb, q8, dq, bs16);
    return hipGetLastError();
}

// n floats (a multiple of 256) to n / 256 Q8_K blocks of 292 bytes.
hipError_t launch_quantize_q8k(const float *in, long long n, void *blocks, hipStream_t st) {
    const long long nb = n / 256;
    hipLaunchKernelGGL(k_rows_q8<true>, dim3((unsigned)((nb + 3) / 4)), dim3(256), 0, st, in, 256, nb,
                       (int8_t *)blocks, nullptr, nullptr);
    return hipGetLastError();
}

hipError_t launch_moe_prefill_q4k_i8(const MoeArgs &a, void *scratch, hipStream_t st) {
    if (!prefill_q4k_layer(a) || !gemm_k_supported(a.H) || !gemm_k_supported(a.F) || a.H % PF_ROWS ||
        a.F % PF_COLS || a.T > 65536 || a.E > 256)
        return hipErrorNotSupported;
    const size_t P = (size_t)a.T * a.k;
    const int max_tiles = (int)((P + PF_MT - 1) / PF_MT + a.E);
    auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
    char *w = (char *)scratch;
    int *perm = (int *)w; w += up(P * 4);
    PfTile *tiles = (PfTile *)w; w += up((size_t)max_tiles * sizeof(PfTile));
    int *ntiles = (int *)w; w += 256;
    int *tpair = (int *)w; w += up((size_t)max_tiles * PF_MT * 4);
    int *ttok = (int *)w; w += up((size_t)max_tiles * PF_MT * 4);
    int8_t *x8 = (int8_t *)w; w += up((size_t)a.T * a.H * 2);
    float *xd = (float *)w; w += up((size_t)a.T * a.H / 256 * 4);
    _Float16 *xb = (_Float16 *)w; w += up((size_t)a.T * a.H / 16 * 4);
    int8_t *a8 = (int8_t *)w; w += up(P * a.F * 2);
    float *ad = (float *)w; w += up(P * a.F / 256 * 4);
    _Float16 *ab = (_Float16 *)w;
    hipError_t err = launch_rows_q8(a.xn, a.T, a.H, x8, xd, xb, st);
    if (err != hipSuccess) return err;
    launch_dispatch(a, perm, tiles, ntiles, tpair, ttok, st);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
    const int ncb0 = a.F / PF_COLS, ncb1 = a.H / PF_ROWS;
    err = launch_moe_i8<0>(a.H / PF_KC, pf_grid((unsigned)(PF_MT / I8_MT * max_tiles * ncb0)), st, (const uint8_t *)a.gate,
                           (const uint8_t *)a.up, x8, xd, xb, a.T, tpair, ttok, tiles, ntiles, ncb0, a.H, a.F, a.act);
    if (err != hipSuccess) return err;
    err = launch_rows_q8(a.act, (long long)P, a.F, a8, ad, ab, st);
    if (err != hipSuccess) return err;
    return launch_moe_i8<1>(a.F / PF_KC, pf_grid((unsigned)(PF_MT / I8_MT * max_tiles * ncb1)), st, (const uint8_t *)a.down,
                            nullptr, a8, ad, ab, (int)P, tpair, ttok, tiles, ntiles, ncb1, a.H, a.F, a.y);
}

// Short rows (n <= 64 * 4 * RW floats): one wave per row, four rows per
// workgroup, the row's max by a wave reduction with no LDS or barrier; the
// same scale and conversion as k_rows_f16.
template <int RW>
__global__ __launch_bounds__(256) void k_rows_f16_wave(const float *__restrict__ in, int rows, int n,
                                                       _Float16 *__restrict__ out, float *__restrict__ inv, bool swap) {
    const int lane = threadIdx.x & 63;
    const int row = min((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6), rows - 1);   // past the end: redo the last
    const bool store = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6) < rows;
    const int n4 = n / 4;
    const float4 *r = reinterpret_cast<const float4 *>(in + (long long)row * n);
    float4 v[RW];
#pragma unroll
    for (int i = 0; i < RW; i++) v[i] = r[min(lane + 64 * i, n4 - 1)];   // clamped: unconditional
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < RW; i++)
        if (lane + 64 * i < n4)
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
    mx = wave_max(mx);
    int e = 0;
    frexpf(mx, &e);
    int sh = mx > 0.f ? 15 - e : 0;
    sh = sh > 126 ? 126 : (sh < -126 ? -126 : sh);
    const float s = ldexpf(1.f, sh);
    if (!store) return;
    uint2 *o = reinterpret_cast<uint2 *>(out + (long long)row * n);
#pragma unroll
    for (int i = 0; i < RW; i++) {
        if (lane + 64 * i < n4) {
            const f16x2 a = {(_Float16)(v[i].x * s), (_Float16)((swap ? v[i].z : v[i].y) * s)};
            const f16x2 b = {(_Float16)((swap ? v[i].y : v[i].z) * s), (_Float16)(v[i].w * s)};
            o[lane + 64 * i] = make_uint2(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
        }
    }
    if (lane == 0) inv[row] = ldexpf(1.f, -sh);
}

hipError_t launch_rows_f16(const float *in, int rows, int n, _Float16 *out, float *inv, hipStream_t st, bool swap) {
    const int rw = (n / 4 + 63) / 64;   // float4 per lane with a wave per row
    const unsigned wgs = (unsigned)((rows + 3) / 4);
    if (rw <= 4) {
        if (rw <= 1) hipLaunchKernelGGL(k_rows_f16_wave<1>, dim3(wgs), dim3(256), 0, st, in, rows, n, out, inv, swap);
        else if (rw <= 2) hipLaunchKernelGGL(k_rows_f16_wave<2>, dim3(wgs), dim3(256), 0, st, in, rows, n, out, inv, swap);
        else if (rw <= 3) hipLaunchKernelGGL(k_rows_f16_wave<3>, dim3(wgs), dim3(256), 0, st, in, rows, n, out, inv, swap);
        else hipLaunchKernelGGL(k_rows_f16_wave<4>, dim3(wgs), dim3(256), 0, st, in, rows, n, out, inv, swap);
        return hipGetLastError();
    }
    const int rv = (n / 4 + 255) / 256;
    switch (rv) {
    case 1: hipLaunchKernelGGL(k_rows_f16<1>, dim3(rows), dim3(256), 0, st, in, n, out, inv, swap); break;
    case 2: hipLaunchKernelGGL(k_rows_f16<2>, dim3(rows), dim3(256), 0, st, in, n, out, inv, swap); break;
    case 3: case 4: hipLaunchKernelGGL(k_rows_f16<4>, dim3(rows), dim3(256), 0, st, in, n, out, inv, swap); break;
    case 5: case 6: case 7: case 8: hipLaunchKernelGGL(k_rows_f16<8>, dim3(rows), dim3(256), 0, st, in, n, out, inv, swap); break;
    case 9: case 10: case 11: case 12: hipLaunchKernelGGL(k_rows_f16<12>, dim3(rows), dim3(256), 0, st, in, n, out, inv, swap); break;
    case 13: case 14: case 15: case 16: hipLaunchKernelGGL(k_rows_f16<16>, dim3(rows), dim3(256), 0, st, in, n, out, inv, swap); break;
    default: hipLaunchKernelGGL(k_rows_f16<0>, dim3(rows), dim3(256), 0, st, in, n, out, inv, swap); break;
    }
    return hipGetLastError();
}

// Experts on MFMA for Q4_K weights; routing already in a.sel_idx/a.sel_w.
// Uses a.act (pairs x F fp32), a.y (pairs x H fp32) and `scratch`
// (prefill_workspace_bytes).  H and F must be 256, 512, 768, 1024, 1536,
// 2048, 3072 or 4096, H a multiple of PF_ROWS and F of PF_COLS; T <= 65536.
void prefill_x16(const MoeArgs &a, void *scratch, _Float16 **x16, float **xinv, bool *swap) {
    *swap = prefill_gq4k_layer(a);
    const size_t P = (size_t)a.T * a.k;
    const size_t max_tiles = (P + PF_MT - 1) / PF_MT + a.E;
    auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
    char *w = (char *)scratch;
    w += up(P * 4) + up(max_tiles * sizeof(PfTile)) + 256 + 2 * up(max_tiles * PF_MT * 4) + up(P * a.F * 2);
    *x16 = (_Float16 *)w;
    w += up((size_t)a.T * a.H * 2) + up(P * 4);
    *xinv = (float *)w;
}

hipError_t launch_moe_prefill_q4k(const MoeArgs &a, void *scratch, hipStream_t st, bool x16_done) {
    const bool gg = prefill_gq4k_layer(a);
    if (!(prefill_q4k_layer(a) || gg) || !gemm_k_supported(a.H) || !gemm_k_supported(a.F) || a.H % MF_ROWS || a.F % (MF_ROWS / 2) ||
        a.T > 65536 || a.E > 256)
        return hipErrorNotSupported;
    const size_t P = (size_t)a.T * a.k;
    const int max_tiles = (int)((P + PF_MT - 1) / PF_MT + a.E);
    auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
    char *w = (char *)scratch;
    int *perm = (int *)w; w += up(P * 4);
    PfTile *tiles = (PfTile *)w; w += up((size_t)max_tiles * sizeof(PfTile));
    int *ntiles = (int *)w; w += 256;
    int *tpair = (int *)w; w += up((size_t)max_tiles * PF_MT * 4);
    int *ttok = (int *)w; w += up((size_t)max_tiles * PF_MT * 4);
    _Float16 *act16 = (_Float16 *)w; w += up(P * a.F * 2);
    _Float16 *x16 = (_Float16 *)w; w += up((size_t)a.T * a.H * 2);
    float *ainv = (float *)w; w += up(P * 4);
    float *xinv = (float *)w;
    if (!x16_done) {
        const hipError_t e = launch_rows_f16(a.xn, a.T, a.H, x16, xinv, st, gg);
        if (e != hipSuccess) return e;
    }
    launch_dispatch(a, perm, tiles, ntiles, tpair, ttok, st);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    const uint8_t *wg = (const uint8_t *)a.gate, *wu = (const uint8_t *)a.up, *wd = (const uint8_t *)a.down;
    err = gg ? launch_moe_f16<0, true>(a, max_tiles, st, wg, wu, x16, a.T, xinv, tpair, ttok, tiles, ntiles, a.H, a.F, a.act)
             : launch_moe_f16<0, false>(a, max_tiles, st, wg, wu, x16, a.T, xinv, tpair, ttok, tiles, ntiles, a.H, a.F, a.act);
    if (err != hipSuccess) return err;
    err = launch_rows_f16(a.act, (int)P, a.F, act16, ainv, st, gg);
    if (err != hipSuccess) return err;
    return gg ? launch_moe_f16<1, true>(a, max_tiles, st, wd, nullptr, act16, (int)P, ainv, tpair, ttok, tiles, ntiles, a.H, a.F, a.y)
              : launch_moe_f16<1, false>(a, max_tiles, st, wd, nullptr, act16, (int)P, ainv, tpair, ttok, tiles, ntiles, a.H, a.F, a.y);
}

}  // namespace tbq

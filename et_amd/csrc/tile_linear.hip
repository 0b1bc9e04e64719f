// Tensor-tile pruned linear (and the dense row-compacted linear) for gfx950.
//
// Computes Y[M x N] = X[M x K] * W^T + bias (optionally followed by GELU) where
// W[N x K] is stored as its surviving 16x16 tiles (tile_mat: CSR over
// block-rows of 16 output features, kernels/linear.cu:54-101 in the
// reference), or dense row-major for the row-pruned linear
// (kernels/linear.cu:18-34).
//
// Mapping.  A workgroup of 8 waves owns 32 rows of X (two 16-row MFMA
// subtiles) and a group of 8*NB consecutive block-rows of W.  The 32 x KC
// panel of X lives in LDS; each wave walks the tile list of its NB block-rows
// and issues v_mfma_f32_16x16x32_f16 with TWO arbitrary surviving tiles
// concatenated along k (a surviving tile is exactly one k=16 slice): lanes
// 0-31 carry the first tile of the pair, lanes 32-63 the second.  The W
// operand of a pair is one coalesced 1 KB global read reused for both row
// subtiles; the X operand is gathered from LDS at the tile's column offset.
// The product is formed transposed (D = W_tile * X^T) so that a lane ends up
// with four consecutive output features of one row, which makes the
// half-precision staging write 8 bytes wide.  Results are staged in LDS and
// written with 16-byte row-contiguous stores, because at >= 80 % sparsity a
// linear on its own is bound by the Y write.
// K larger than the LDS panel is walked in chunks of KC columns; plans sort
// each block-row's tiles by column and carry a per-chunk CSR so a chunk only
// touches its own tiles (TL_PLAN); raw unsorted input with K > one panel falls
// back to filtering the whole list per chunk (TL_FILTER).
//
// Kernels in this file: tile_linear_resident_kernel (K in one panel: persistent
// workgroups, 32- or 64-row panels, optional LayerNorm epilogue),
// tile_linear_plan_kernel (K in chunks), tile_linear_chunked_kernel (K in
// chunks, double-buffered panels with fetching waves, optional LayerNorm
// epilogue), tile_ffn_fused_kernel (feed-forward block / whole layer tail in one
// launch, hidden activations in LDS), tile_linear_generic_kernel (raw and dense
// input).  Whole rows in LDS (tile_rows.hip) and the dense product
// (dense_gemm.hip) are launched from here where they are the shorter launch.
#include "tile_plan.h"
#include "tile_walk.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <numeric>
#include <vector>

namespace et {

void set_attn_variant(int v);
void set_attn_vwin(int v);
void set_attn_packed(int v);
void set_ln_rows(int v);
void set_tail_pair(int v);
void set_tail_spin(int v);
void set_dense_form(int v);
// tile_rows.hip
bool tile_rows_fits(int K);
double tile_rows_estimate(int M, int K, int nbr_max, int nlin, double pairs, double w_mb);
int tile_rows_launch(const LfLinear *lins, f16 *const *Ys, int nlin, const f16 *X, int M, int K, double pairs, bool gelu,
                     bool raw, hipStream_t st);
void set_flow_rows(int v);
void set_qkv_attention(int v);
void set_row_layernorm(int v);
int tail_spin();

constexpr int TL_THREADS = 512;
constexpr int TL_WAVES = 8;
constexpr int TL_BM = 32;
constexpr int TL_PAD = 16;       // halves; LDS row stride == 32 (mod 64) bytes: measured conflict-free for ds_read_b128
constexpr int TL_MAX_PANEL = 1024;      // plans: single-panel K limit, two 16-byte pieces per lane and row
constexpr int TL_MAX_RAW_PANEL = 992;   // generic kernel: 32*(992+16)*2 B < 64 KB
constexpr int TL_CHUNK = 768;
constexpr int TL_MAX_LIN = 4;

// TL_PLAN: plan layout (see et_tile_plan_create): tiles ordered (chunk,
//          block-row, column), every (chunk, block-row) segment padded to an
//          even tile count with an all-zero tile, cptr[c*nbr + bn] in tiles.
// TL_RAW:  caller's tile_mat as is (any order inside a block-row, odd counts),
//          K fits one LDS panel; cptr is row_ptr.
// TL_FILTER: caller's tile_mat, K walked in chunks by filtering every list.
// TL_DENSE: W row-major [N x K] (the row-pruned linear's compacted rows).
enum { TL_PLAN = 0, TL_RAW = 1, TL_FILTER = 2, TL_DENSE = 3 };

struct TlProblem {
    f16 *Y;
    const int *cptr;
    const int *row_offset; // element column offset per tile
    const f16 *data;       // tile data, or dense row-major W for TL_DENSE
    const f16 *bias;
    int N;
    int nbr; // N / 16
    int ntile = 0; // surviving tiles where known (plans), 0 otherwise
    int npair = 0; // index of an all-zero pair (plans)
};

// kernel arguments; per-linear fields as separate arrays that are only ever
// indexed with constants (a dynamically indexed by-value struct would be
// copied to scratch memory)
struct TlArgs {
    f16 *Y[TL_MAX_LIN];
    const int *cptr[TL_MAX_LIN];
    const int *row_offset[TL_MAX_LIN];
    const f16 *data[TL_MAX_LIN];
    const f16 *bias[TL_MAX_LIN];
    int N[TL_MAX_LIN];
    const f16 *X;
    int nlin, M, K, KC, nchunk, ncg, per_xcd;
    int ipw;      // resident kernel: consecutive items of a row panel per workgroup
    int nwg, div; // workgroups; those of a panel (by_group: of a column group)
    unsigned div_magic, ncg_magic; // magic_of(div), magic_of(ncg)
    int by_group; // consecutive workgroups walk the panels of one column group (tl_order)
    // fused skip + LayerNorm epilogue (plan kernels with LN = true)
    const f16 *skip, *gamma, *beta;
    const f16 *gamma2, *beta2; // second LayerNorm of the fused layer tail
    int *status;               // fused feed-forward kernels: set when a bounded LDS wait gives up
    int spin;                  // ... after this many polls
};
// What a workgroup needs before its first requests stands in front of the struct as parameters of its own: the hardware
// loads the first fourteen dwords of scalar parameters into registers while it starts a wave (build.py asks for it), a
// struct is fetched from memory by the wave.  0.3-0.6 us a launch: 80 %, 37 rows 768->768 4.50 -> 4.12, 1536 rows
// 768->768 + skip + LayerNorm 6.24 -> 5.90, 1000 rows 3072->768 10.5 -> 9.8.  (The fused feed-forward kernel runs for
// 50 us and has no register to spare: its arguments stay in the struct.)
#define TL_HOT_PARAMS                                                                             \
    const f16 *hot_X, const int *hot_cptr, int hot_M, int hot_K, int hot_n, int hot_per_xcd, int hot_nwg, int hot_div,       \
        unsigned hot_div_magic, unsigned hot_ncg_magic, int hot_ncg, int hot_ipw
// (hot_n: outputs of the first linear for the resident kernel, whose one chunk is K wide, else the chunk's width)
#define TL_HOT(a_, n_)                                                                            \
    (a_).X, (a_).cptr[0], (a_).M, (a_).K, (a_).n_, (a_).per_xcd, (a_).nwg, (a_).div, (a_).div_magic, (a_).ncg_magic, (a_).ncg,  \
        (a_).ipw | (a_).nlin << 24 | ((a_).by_group ? 1 << 30 : 0)
constexpr int TL_HOT_BYTES = 2 * 8 + 10 * 4; // (the struct starts behind them)
#define TL_HOT_TAKE(a_, args_, n_)                                                                \
    TlArgs a_ = args_;                                                                            \
    a_.X = hot_X;                                                                                 \
    a_.cptr[0] = hot_cptr;                                                                        \
    a_.M = hot_M;                                                                                 \
    a_.K = hot_K;                                                                                 \
    a_.n_ = hot_n;                                                                                \
    a_.per_xcd = hot_per_xcd;                                                                     \
    a_.nwg = hot_nwg;                                                                             \
    a_.div = hot_div;                                                                             \
    a_.div_magic = hot_div_magic;                                                                 \
    a_.ncg_magic = hot_ncg_magic;                                                                 \
    a_.ncg = hot_ncg;                                                                             \
    a_.by_group = hot_ipw >> 30;                                                                  \
    a_.nlin = hot_ipw >> 24 & 63;                                                                 \
    a_.ipw = hot_ipw & 0xFFFFFF;
#define TL_SEL(f) (lin == 0 ? a.f[0] : lin == 1 ? a.f[1] : lin == 2 ? a.f[2] : a.f[3])

// tanh-form GELU of kernels/linear.cu:36-48: x^3 in half, the tanh argument
// and 0.5(1+tanh u) in fp32, rounded to half, times x in half.
// 0.5(1+tanh u) == 1 - 1/(exp(2u)+1).
__device__ __forceinline__ f16 gelu_h(f16 v) {
    const f16 x2 = v * v;
    const f16 x3 = v * x2;
    const float x = (float)v;
    const float u2 = 1.5957691216057308f * (x + 0.044715f * (float)x3); // 2u
    const float e = __builtin_amdgcn_exp2f(u2 * 1.4426950408889634f);
    const float t = 1.0f - __builtin_amdgcn_rcpf(e + 1.0f);
    return v * (f16)t;
}

// A workgroup's first item.  The hardware deals consecutive workgroup ids round robin over the 8 XCDs; consecutive
// virtual ids run on ONE of them.  They are the column groups of a row panel, which then enters one L2 only while W
// enters all eight - or, by_group, the panels of a column group: W enters one L2 and the panels all of them.  The
// launcher takes the order that moves fewer bytes (tl_order).
__device__ __forceinline__ bool tl_place(const TlArgs &a, int &rp, int &lin, int &cg) {
    const int vid = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    if (vid >= a.nwg)
        return false;
    const QuotRem of = quot_rem(vid, a.div, a.div_magic);
    rp = a.by_group ? of.r : of.q;
    const QuotRem rest = quot_rem((a.by_group ? of.q : of.r) * a.ipw, a.ncg, a.ncg_magic);
    lin = rest.q;
    cg = rest.r;
    return true;
}

// what every variant shares: workgroup -> (row panel, linear, column group)
struct TlCtx {
    int lin, cg, m0, wave, lane, c16, g4, khalf8, hi, ldx, bn_wg, bn0, ld_r, ld_c;
};

__device__ __forceinline__ bool tl_context(const TlArgs &a, int nb, TlCtx &x) {
    int rp;
    if (!tl_place(a, rp, x.lin, x.cg))
        return false;
    x.m0 = rp * TL_BM;
    x.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    x.lane = threadIdx.x & 63;
    x.c16 = x.lane & 15;
    x.g4 = x.lane >> 4;
    x.khalf8 = (x.g4 & 1) * 8;
    x.hi = x.lane >> 5;
    x.ldx = a.KC + ((a.KC & 31) ? 0 : TL_PAD);
    x.bn_wg = x.cg * (TL_WAVES * nb);
    x.bn0 = x.bn_wg + x.wave * nb;
    x.ld_r = threadIdx.x >> 4; // 0..31: panel row this thread stages
    x.ld_c = threadIdx.x & 15;
    return true;
}

// bias (+GELU), round to half, stage in LDS (the X panel's storage), then
// 16-byte row-contiguous stores
template <int NB, bool GELU>
__device__ __forceinline__ void tl_epilogue(const TlArgs &a, const TlCtx &x, f16 *xs, f16 *Y, int N,
                                            int nbr, const f32x4 (&acc)[NB][2], const f16x4 (&b4)[NB]) {
    __syncthreads(); // every wave is done reading the X panel
    constexpr int BNW = TL_WAVES * NB * 16; // output columns per workgroup
    constexpr int ldy = BNW + TL_PAD;
    f16 *ys = xs;
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int bn = x.bn0 + j;
        if (bn >= nbr)
            continue;
        const int ncol = (bn - x.bn_wg) * 16 + x.g4 * 4;
#pragma unroll
        for (int ms = 0; ms < 2; ms++) {
            f16x4 o;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const f16 v = (f16)(acc[j][ms][r] + (float)b4[j][r]);
                o[r] = GELU ? gelu_h(v) : v;
            }
            *reinterpret_cast<f16x4 *>(ys + (ms * 16 + x.c16) * ldy + ncol) = o;
        }
    }
    __syncthreads();
    const int col0 = x.bn_wg * 16;
    const int wcols = min(BNW, N - col0);
    const int cpr = wcols >> 3;
    if (x.m0 + x.ld_r < a.M) {
        u32x4 *dst = reinterpret_cast<u32x4 *>(Y + (size_t)(x.m0 + x.ld_r) * N + col0);
        const u32x4 *src = reinterpret_cast<const u32x4 *>(ys + x.ld_r * ldy);
        for (int cc = x.ld_c; cc < cpr; cc += 16)
            dst[cc] = src[cc];
    }
}

// Per-wave epilogue: bias (+GELU), round to half, transpose through a
// wave-private LDS tile (32 rows x 16*NB columns, no barrier: a wave's LDS
// operations execute in order), then 16-byte stores of 32*NB contiguous bytes
// per row.  Waves never wait for each other here, so one wave's stores overlap
// the other waves' MFMAs.
template <int NB> constexpr int tl_wave_stage_halves() { return TL_BM * (16 * NB + 8); }

template <int NB, bool GELU, bool STORE = true>
__device__ __forceinline__ void tl_epilogue_wave(const TlArgs &a, const TlCtx &x, f16 *stage, f16 *Y,
                                                 int N, int nbr, const f32x4 (&acc)[NB][2],
                                                 const f16x4 (&b4)[NB]) {
    constexpr int lds = 16 * NB + 8; // halves per staged row
#pragma unroll
    for (int j = 0; j < NB; j++) {
#pragma unroll
        for (int ms = 0; ms < 2; ms++) {
            f16x4 o;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const f16 v = (f16)(acc[j][ms][r] + (float)b4[j][r]);
                o[r] = GELU ? gelu_h(v) : v;
            }
            *reinterpret_cast<f16x4 *>(stage + (ms * 16 + x.c16) * lds + j * 16 + x.g4 * 4) = o;
        }
    }
    if (!STORE)
        return;
    // valid block-rows of this wave (the last column group may be partial)
    const int nvalid = min(NB, nbr - x.bn0);
    if (nvalid <= 0)
        return;
    const int cpr = 2 * nvalid; // 16-byte chunks per row
    f16 *ybase = Y + (size_t)x.m0 * N + x.bn0 * 16;
#pragma unroll
    for (int t = 0; t < NB; t++) {
        const int i = x.lane + 64 * t;
        const int r = i / (2 * NB), c = i - r * (2 * NB);
        if (c < cpr && x.m0 + r < a.M) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(stage + r * lds + c * 8);
            *reinterpret_cast<u32x4 *>(ybase + (size_t)r * N + c * 8) = v;
        }
    }
}

// ---------------------------------------------------------------------------
// The pair stream shared by the plan kernels.
//
// A wave owns NB CONSECUTIVE block-rows, and the plan stores tiles in (chunk,
// block-row) order with even segments, so the wave's work for a chunk is ONE
// contiguous run of tile pairs [q0, qend): 1 KB of W per pair at an address
// linear in the pair index, plus one int per half-wave giving the LDS byte
// offset of that tile's X columns.  The run is consumed through a TL_DEPTH-stage
// register pipeline (stage = pair index mod TL_DEPTH) with unconditional loads
// in the main loop, so TL_DEPTH pairs are always in flight per wave and the
// waits are counted, not drained; only the last stages of a run test whether
// there is still a pair to request.  X operands are read from LDS one stage
// ahead.  Products accumulate into one running 32x16 accumulator; when the
// stream crosses a block-row boundary (a scalar compare per pair) flush(j,
// cur0, cur1) receives block-row j's finished sums.  All control flow in here
// is wave-uniform and straight-line per stage: loops or conditional loads
// would make the compiler drain every load instead of counting.
// ---------------------------------------------------------------------------
#ifndef TL_DEPTH
#define TL_DEPTH 4
#endif
// Wave priority while a stream runs (0 outside and inside a flush): waves that
// are streaming issue their loads and MFMAs ahead of waves that sit in the
// vector-ALU work of a GELU flush or a LayerNorm (layer tail: -2 %).
#ifndef TL_PRIO
#define TL_PRIO 1
#endif
static_assert(TL_DEPTH % 2 == 0, "the X operand ping-pong needs an even pipeline depth");

template <int I> using tl_ic = std::integral_constant<int, I>;
template <int B, int E, class F>
__device__ __forceinline__ void tl_static_for(F &&f) {
    if constexpr (B < E) {
        f(tl_ic<B>());
        tl_static_for<B + 1, E>(f);
    }
}

// the first TL_DEPTH pairs of a stream (an empty stream still loads pair q0:
// the plan keeps a spare pair behind the last one)
// One pair's operands: 16 bytes of W per lane and the lane's X offset.  The
// pair's address is wave-uniform (scalar registers) and the lane's part a
// 32-bit offset, so the loads need no vector address arithmetic.
// lo / lw: the lane's byte offsets into a pair's two ints and its 1 KB of W
__device__ __forceinline__ void tl_load_pair_at(const char *wq, const char *oq, unsigned &lo,
                                                unsigned &lw, f16x8 &w, int &o) {
    // (the empty asm, in place on variables that live across the whole stream,
    // makes the lane offsets look freshly computed: otherwise the compiler folds
    // them into loop-invariant 64-bit vector addresses and pays two 64-bit
    // vector adds per pair instead of using scalar base + 32-bit lane offset)
    asm("" : "+v"(lo), "+v"(lw));
    o = *reinterpret_cast<const int *>(oq + lo);
    w = *reinterpret_cast<const f16x8 *>(wq + lw);
}
__device__ __forceinline__ void tl_load_pair(const f16 *data, const int *poff, int q, unsigned lane_w,
                                             unsigned hi, f16x8 &w, int &o) {
    unsigned lo = hi * 4u, lw = lane_w * 2u;
    tl_load_pair_at(reinterpret_cast<const char *>(data) + (size_t)q * 1024,
                    reinterpret_cast<const char *>(poff) + (size_t)q * 8, lo, lw, w, o);
}

__device__ __forceinline__ void tl_preload(const f16 *data, const int *poff, unsigned lane_w, unsigned hi,
                                           int q0, int qlast, f16x8 (&w)[TL_DEPTH], int (&o)[TL_DEPTH]) {
#pragma unroll
    for (int i = 0; i < TL_DEPTH; i++)
        tl_load_pair(data, poff, min(q0 + i, qlast), lane_w, hi, w[i], o[i]);
}


// Ends of a wave's block-rows: [k] is the first pair of block-row k, [NB] the end of the last one.  In scalar registers
// throughout: kept in the lanes of a vector register, every block-row end cost reads of single lanes, and filling it a
// select per end, all of them vector instructions, which is what the fused layer tail is bound by (8192 rows, 80 %:
// 50.5 -> 48.4 us; 90 %: 42.5 -> 40.5; the Q/K/V launch of 64-row panels 15.7 -> 15.4).
template <int NB> struct TlBounds {
    int at[NB + 1];
};
// (bvec: lane k holds [k])
template <int NB> __device__ __forceinline__ TlBounds<NB> tl_bounds(int bvec) {
    TlBounds<NB> b;
#pragma unroll
    for (int k = 0; k <= NB; k++)
        b.at[k] = __builtin_amdgcn_readlane(bvec, k);
    return b;
}

// MS 16-row subtiles per pair: 2 (a 32-row panel), or 4 (64 rows: a W pair feeds four MFMAs, and a stream that is bound by
// delivering W runs faster).  flush(j, sums) receives block-row j's MS sums.
template <int NB, int MS, class Flush>
__device__ __forceinline__ void tl_stream(const char *xlane, int xrow16, const f16 *data, const int *poff, unsigned lane_w,
                                          unsigned hi, TlBounds<NB> bounds, f16x8 (&w)[TL_DEPTH], int (&o)[TL_DEPTH],
                                          Flush &&flush) {
    const int qend = bounds.at[NB];
    int q = bounds.at[0];
    if (q >= qend)
        return;
    __builtin_amdgcn_s_setprio(TL_PRIO);
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 cur[MS];
#pragma unroll
    for (int m = 0; m < MS; m++)
        cur[m] = zero;
    // j: the block-row that runs, ends at bend; the ends behind it move up as block-rows close
    int j = 0, bend = bounds.at[1], ends[NB];
#pragma unroll
    for (int k = 0; k < NB; k++)
        ends[k] = bounds.at[k + 2 < NB ? k + 2 : NB];
    auto next_end = [&] {
        j++;
        bend = ends[0];
#pragma unroll
        for (int k = 0; k < NB - 1; k++)
            ends[k] = ends[k + 1];
    };
#pragma unroll
    for (int t = 0; t < NB - 1; t++) // leading empty block-rows
        if (bend == q)
            next_end();
    f16x8 x[2][MS];
#pragma unroll
    for (int m = 0; m < MS; m++) {
        x[0][m] = *reinterpret_cast<const f16x8 *>(xlane + o[0] + m * xrow16);
        x[1][m] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    // running (wave-uniform) addresses of pair q + TL_DEPTH: a stage adds a
    // constant, which goes into the load's immediate offset
    const char *wp = reinterpret_cast<const char *>(data) + (size_t)(q + TL_DEPTH) * 1024;
    const char *op = reinterpret_cast<const char *>(poff) + (size_t)(q + TL_DEPTH) * 8;
    unsigned lane_lo = hi * 4u, lane_lw = lane_w * 2u;
    auto stage = [&](auto ic, auto always) {
        constexpr int I = decltype(ic)::value;
        constexpr int S = I % TL_DEPTH, SN = (I + 1) % TL_DEPTH, P = I & 1;
#pragma unroll
        for (int m = 0; m < MS; m++)
            x[P ^ 1][m] = *reinterpret_cast<const f16x8 *>(xlane + o[SN] + m * xrow16);
        // keep the reads above the MFMAs: left alone, the scheduler sinks them
        // to the end of the stage and every stage then waits out the LDS latency
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < MS; m++)
            cur[m] = mfma16x16x32(w[S], x[P][m], cur[m]);
        // pair q + I + TL_DEPTH; the last stages of a stream request nothing:
        // a request still in flight when the stream ends would make the next
        // use of these registers wait out a full memory latency
        if (decltype(always)::value || q + I + TL_DEPTH < qend)
            tl_load_pair_at(wp + I * 1024, op + I * 8, lane_lo, lane_lw, w[S], o[S]);
        if (q + I + 1 == bend) { // block-row j is complete
            __builtin_amdgcn_s_setprio(0);
            flush(j, cur);
            __builtin_amdgcn_s_setprio(TL_PRIO);
#pragma unroll
            for (int m = 0; m < MS; m++)
                cur[m] = zero;
            next_end();
#pragma unroll
            for (int t = 0; t < NB - 2; t++) // skip empty block-rows
                if (bend == q + I + 1)
                    next_end();
        }
    };
    for (; q + 2 * TL_DEPTH <= qend; q += TL_DEPTH) { // straight-line body: counted waits
        tl_static_for<0, TL_DEPTH>([&](auto ic) { stage(ic, std::true_type()); });
        wp += TL_DEPTH * 1024;
        op += TL_DEPTH * 8;
    }
    tl_static_for<0, 2 * TL_DEPTH - 1>([&](auto ic) {
        if (q + decltype(ic)::value < qend)
            stage(ic, std::false_type());
    });
    __builtin_amdgcn_s_setprio(0);
}

// flush for kernels that keep NB static accumulators: acc[j] += cur by a
// branch per accumulator.  (A factor of 0 or 1 per accumulator makes NaN of an
// infinite sum in block-rows that it does not belong to; a mask on the sums'
// bits is two instructions for each value of every accumulator.  48-row panels,
// factor / mask / branch, us: 5134 rows 4096 -> 1024 80 % 23.6 / 24.6 / 23.4, 16000
// rows 3072 -> 768 90 % 39.5 / 40.9 / 39.1, 10000 rows 2048 -> 512 50 % 23.1 / 23.4 /
// 23.1.)  Two things keep the compiler from undoing the branches: the adds are
// inline assembly with tied operands (the sum replaces the accumulator in its
// own registers; otherwise every accumulator gets a second set of registers
// behind the branches), and the cases are independent ifs with something opaque
// between them (as an if / else chain they become a switch, whose lowering
// copies the accumulators around or addresses them through scratch memory).
template <int K>
__device__ __forceinline__ void tl_add_tied(f32x4 &a, const f32x4 &c) {
    float a0 = a[0], a1 = a[1], a2 = a[2], a3 = a[3];
    asm volatile("v_add_f32 %0, %0, %4 ; accumulator %8\n\tv_add_f32 %1, %1, %5\n\t"
                 "v_add_f32 %2, %2, %6\n\tv_add_f32 %3, %3, %7"
                 : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
                 : "v"(c[0]), "v"(c[1]), "v"(c[2]), "v"(c[3]), "n"(K));
    a = f32x4{a0, a1, a2, a3};
}
template <int NB, int MS>
__device__ __forceinline__ void tl_flush_acc(f32x4 (&acc)[NB][MS], int j, const f32x4 (&cur)[MS]) {
    if constexpr (NB == 1) {
#pragma unroll
        for (int m = 0; m < MS; m++)
            acc[0][m] += cur[m];
    } else {
        tl_static_for<0, NB>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            if (j == k) {
#pragma unroll
                for (int m = 0; m < MS; m++)
                    tl_add_tied<k>(acc[k][m], cur[m]);
            }
            asm volatile("; after case %0" ::"n"(k));
        });
    }
}

// Fused skip connection + LayerNorm over a workgroup's 32 finished rows (the
// math of skip_layernorm.hip: x = half(y + skip), fp32 mean and biased
// two-pass variance, eps 1e-6).  The workgroup covers the whole row: wave k's
// staging tile holds columns [k*16*NB, (k+1)*16*NB), k < NW.  Wave w of the NLW
// waves that take part normalises rows w, w+NLW, ..., two at a time, each spread
// over 32 lanes in 16-byte pieces (rows wider than 1024: one over 64, for the
// registers).  A row of 768 is one and a half pieces for 64 lanes and three for
// 32, and two rows share the sums' exchanges: 140 vector instructions a wave and
// LayerNorm fewer than row after row, and the layer tail keeps its registers out of
// memory.  Whole layers of 16 x 512 rows 82.4 -> 79.7 us, with pruned values 83.8 ->
// 82.2, the stack of 64 ragged sequences 2287 -> 2226 (inputs that change from pass to
// pass).  The sums are those of skip_layernorm.hip to the bit; those of a row over 64
// lanes differed from them in the last bit of a variance.
// The operands that come from global memory (the skip rows, gamma, beta) are requested
// by tl_ln_fetch, which a wave calls BEFORE the barrier that ends the staging writes, so
// that their latency runs under the wait for the other waves.
template <int NB, int NW, int NLW>
struct TlLnOperands {
    static constexpr int LPR = NW * NB > 64 ? 64 : 32;                         // lanes per row
    static constexpr int NP = (NW * NB * 2 + LPR - 1) / LPR;                   // 16-byte pieces per lane
    static constexpr int STEPS = ((TL_BM + NLW - 1) / NLW * LPR + 63) / 64;    // rows, or pairs of them, per wave
    f16x8 skip[STEPS][NP], gamma[NP], beta[NP];
};

// (skip0 / Y0 point at the panel's first row, in global memory or in LDS, with
// row pitches ldskip / ldy in halves)
template <int NB, int NW, int NLW>
__device__ __forceinline__ void tl_ln_fetch_skip(TlLnOperands<NB, NW, NLW> &op, int M, int wave, int lane,
                                                 int m0, int N, const f16 *skip0, long ldskip) {
    typedef TlLnOperands<NB, NW, NLW> Op;
#pragma unroll
    for (int i = 0; i < Op::NP; i++) {
        const int ch = min((lane & (Op::LPR - 1)) + Op::LPR * i, (N >> 3) - 1); // (clamped pieces are never used)
#pragma unroll
        for (int k = 0; k < Op::STEPS; k++) {
            const long r = min(wave + (64 / Op::LPR * k + lane / Op::LPR) * NLW, min(TL_BM, M - m0) - 1);
            op.skip[k][i] = *reinterpret_cast<const f16x8 *>(skip0 + r * ldskip + ch * 8);
        }
    }
}
// (behind the epilogue: its accumulators' registers are free then)
template <int NB, int NW, int NLW>
__device__ __forceinline__ void tl_ln_fetch_scale(TlLnOperands<NB, NW, NLW> &op, int lane, int N, const f16 *gamma,
                                                  const f16 *beta) {
#pragma unroll
    for (int i = 0; i < TlLnOperands<NB, NW, NLW>::NP; i++) {
        constexpr int LPR = TlLnOperands<NB, NW, NLW>::LPR;
        const int ch = min((lane & (LPR - 1)) + LPR * i, (N >> 3) - 1);
        op.gamma[i] = *reinterpret_cast<const f16x8 *>(gamma + ch * 8);
        op.beta[i] = *reinterpret_cast<const f16x8 *>(beta + ch * 8);
    }
}

template <int NB, int NW, int NLW>
__device__ __forceinline__ void tl_ln_fetch(TlLnOperands<NB, NW, NLW> &op, const TlArgs &a, int wave,
                                            int lane, int m0, int N) {
    tl_ln_fetch_skip(op, a.M, wave, lane, m0, N, a.skip + (long)m0 * N, (long)N);
    tl_ln_fetch_scale(op, lane, N, a.gamma, a.beta);
}

template <int NB, int NW, int NLW>
__device__ __forceinline__ void tl_ln_rows_at(const TlLnOperands<NB, NW, NLW> &op, int M,
                                              const f16 *stage0, int wave, int lane, int m0, int N,
                                              f16 *Y0, long ldy);

template <int NB, int NW, int NLW>
__device__ __forceinline__ void tl_ln_rows(const TlLnOperands<NB, NW, NLW> &op, const TlArgs &a,
                                           const f16 *stage0, int wave, int lane, int m0, f16 *Y, int N) {
    tl_ln_rows_at(op, a.M, stage0, wave, lane, m0, N, Y + (long)m0 * N, (long)N);
}

template <int NB, int NW, int NLW>
__device__ __forceinline__ void tl_ln_rows_at(const TlLnOperands<NB, NW, NLW> &op, int M,
                                              const f16 *stage0, int wave, int lane, int m0, int N,
                                              f16 *Y0, long ldy) {
    constexpr int lds = 16 * NB + 8;
    typedef TlLnOperands<NB, NW, NLW> Op;
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    constexpr int LPR = Op::LPR, HALF = LPR == 32;
    const int npiece = N >> 3;
    const float inv_n = 1.0f / (float)N;
    auto row_sum = [](const float (&v)[2]) { return LPR == 32 ? half_wave_sum(v[0], v[1]) : wave_sum(v[0]); };
    // (a half times 1.0 plus a float is one instruction; the multiplier is opaque, or it is a conversion and an addition)
    float one = 1.0f;
    asm("" : "+s"(one));
#pragma unroll
    for (int k = 0; k < Op::STEPS; k++) {
        if (m0 + wave + 64 / LPR * k * NLW >= M) // (wave-uniform)
            break;
        const int r = wave + (64 / LPR * k + lane / LPR) * NLW, rc = min(r, TL_BM - 1);
        f16x8 xv[Op::NP];
        // (32 lanes: the sums of the pieces that a whole wave would hold in lanes 0..31 and in lanes 32..63 are kept apart,
        // since skip_layernorm.hip adds in that order)
        float sum[2] = {0.f, 0.f}, var[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < Op::NP; i++) {
            const int ch = (lane & (LPR - 1)) + LPR * i;
            const int tile = ch / (2 * NB), c = ch - tile * (2 * NB);
            xv[i] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (ch < npiece)
                xv[i] = *reinterpret_cast<const f16x8 *>(stage0 + tile * tl_wave_stage_halves<NB>() + rc * lds + c * 8) +
                        op.skip[k][i]; // half add, one rounding (kernels/skip_layernorm.cu:20)
            // (pairs of halves summed in fp32 by the dot-product unit: no conversions)
#pragma unroll
            for (int j = 0; j < 8; j += 2)
                sum[i & HALF] = __builtin_amdgcn_fdot2(h2{xv[i][j], xv[i][j + 1]}, h2{(f16)1, (f16)1}, sum[i & HALF], false);
        }
        const float mean = row_sum(sum) * inv_n;
#pragma unroll
        for (int i = 0; i < Op::NP; i++)
            if ((lane & (LPR - 1)) + LPR * i < npiece) {
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float d = __builtin_fmaf((float)xv[i][j], one, -mean);
                    var[i & HALF] += d * d;
                }
            }
        const float rstd = __builtin_amdgcn_rsqf(row_sum(var) * inv_n + 1e-6f); // (never a denormal)
        const float shift = -mean * rstd;
        const bool store = r < min(TL_BM, M - m0);
#pragma unroll
        for (int i = 0; i < Op::NP; i++) {
            const int ch = (lane & (LPR - 1)) + LPR * i;
            f16x8 o;
#pragma unroll
            for (int j = 0; j < 8; j++) // ((x - mean) * rstd) * gamma + beta, the first step as one fma
                o[j] = (f16)(__builtin_fmaf((float)xv[i][j], rstd, shift) * (float)op.gamma[i][j] + (float)op.beta[i][j]);
            if (store && ch < npiece)
                *reinterpret_cast<f16x8 *>(Y0 + r * ldy + ch * 8) = o;
        }
    }
}

// ---------------------------------------------------------------------------
// Plan kernel: K in chunks, one panel buffer.
//
// A workgroup does one (row panel, linear, column group): it fetches a chunk of
// the panel, waits, multiplies and goes on to the next chunk; every wave stages
// its output through a private LDS tile, so one wave's stores overlap the
// others' MFMAs.
//
// A wave owns NB CONSECUTIVE block-rows, and the plan stores
// tiles in (chunk, block-row) order with even segments, so the wave's work for
// a chunk is ONE contiguous stream of tile pairs: 1 KB of W per pair at an
// address that is linear in the pair index, plus one int per half-wave giving
// the LDS byte offset of that tile's X columns.  The stream is consumed
// through a fixed 4-stage register pipeline (stage = pair index mod 4, see
// tl_stream), so four pairs are always in flight per wave and the waits are
// counted, not drained.  Products accumulate
// into one running 32x16 accumulator; when the stream crosses a block-row
// boundary (a scalar compare per pair) it is added into that block-row's
// static accumulator.
// ---------------------------------------------------------------------------

template <int NB, bool GELU, int NW, bool LN>
__global__ void __launch_bounds__(NW * 64) tile_linear_plan_kernel(TL_HOT_PARAMS, const TlArgs args) {
    TL_HOT_TAKE(a, args, KC)
    extern __shared__ __attribute__((aligned(16))) unsigned char tl_smem[];
    f16 *xs = reinterpret_cast<f16 *>(tl_smem);
    TlCtx x;
    int rp;
    if (!tl_place(a, rp, x.lin, x.cg))
        return;
    x.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    x.lane = threadIdx.x & 63;
    x.c16 = x.lane & 15;
    x.g4 = x.lane >> 4;
    x.khalf8 = (x.g4 & 1) * 8;
    x.hi = x.lane >> 5;
    x.ldx = a.KC + ((a.KC & 31) ? 0 : TL_PAD);
    const int hi = x.hi, lane = x.lane;
    const char *xlane = reinterpret_cast<const char *>(xs + x.c16 * x.ldx + x.khalf8);
    const int xrow16 = 16 * x.ldx * 2; // bytes between the two 16-row subtiles
    f16 *const stage0 = xs + TL_BM * x.ldx;
    f16 *const stage = stage0 + x.wave * tl_wave_stage_halves<NB>();

    // X panel staging: global -> LDS directly (global_load_lds_dwordx4: lane L
    // of the issuing wave writes 16 bytes at  base + 16*L, the source address is
    // free per lane).  Wave w fills panel rows 4w..4w+3, each row as one 64-lane
    // and one partial instruction; no VGPRs are held and nothing waits until the
    // barrier.  Rows at or beyond M are left unwritten: a panel row only feeds
    // the output row of the same index, which is never stored.
#define TL_PANEL_LOAD(c_)                                                                         \
    {                                                                                             \
        const int pk0 = (c_) * a.KC;                                                              \
        const int pcpr = min(a.KC, a.K - pk0) >> 3; /* 16-byte chunks per row, <= 96 */           \
        _Pragma("unroll") for (int rr = 0; rr < TL_BM / NW; rr++) {                               \
            const int row = x.wave * (TL_BM / NW) + rr;                                           \
            if (x.m0 + row < a.M) {                                                               \
                const f16 *src = a.X + (size_t)(x.m0 + row) * a.K + pk0;                          \
                f16 *dstrow = xs + row * x.ldx;                                                   \
                if (lane < pcpr)                                                                  \
                    load_lds16(src + lane * 8, dstrow);                                           \
                if (64 + lane < pcpr)                                                             \
                    load_lds16(src + (64 + lane) * 8, dstrow + 512);                              \
            }                                                                                     \
        }                                                                                         \
    }

    const int lin = x.lin;
    x.m0 = rp * TL_BM;
    x.bn_wg = x.cg * (NW * NB);
    x.bn0 = x.bn_wg + x.wave * NB;
    f16 *const Yp = TL_SEL(Y);
    const int *const cptr = TL_SEL(cptr);
    const int *const poff = TL_SEL(row_offset); // LDS byte offset per tile (chunk-local column * 2)
    const f16 *const data = TL_SEL(data);
    const f16 *const bias = TL_SEL(bias);
    const int N = TL_SEL(N);
    const int nbr = N >> 4;

    f32x4 acc[NB][2];
    f16x4 b4[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        acc[j][0] = f32x4{0.f, 0.f, 0.f, 0.f};
        acc[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        b4[j] = f16x4{0, 0, 0, 0};
        if (x.bn0 + j < nbr)
            b4[j] = *reinterpret_cast<const f16x4 *>(bias + (x.bn0 + j) * 16 + x.g4 * 4);
    }
    const unsigned lane_w = hi * 256 + x.c16 * 16 + x.khalf8; // lane's halves inside a 1 KB tile pair

    for (int c = 0; c < a.nchunk; c++) {
        // pair-index boundaries of the wave's block-rows: lane j holds the end
        // of block-row j (read back with v_readlane)
        const int bidx = c * nbr + min(x.bn0 + min(lane, NB), nbr);
        const int bvec = cptr[bidx] >> 1;

        if (c > 0)
            __syncthreads(); // every wave is done with the previous chunk
        TL_PANEL_LOAD(c)
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): this wave's part has landed
        __syncthreads();                    // ... and everyone else's
        // the first pairs of the stream
        const int q0 = __builtin_amdgcn_readfirstlane(bvec);
        const int qend = __builtin_amdgcn_readlane(bvec, NB);
        const int qlast = max(qend - 1, q0);
        f16x8 w[TL_DEPTH];
        int o[TL_DEPTH];
        tl_preload(data, poff, lane_w, hi, q0, qlast, w, o);
        tl_stream<NB, 2>(xlane, xrow16, data, poff, lane_w, hi, tl_bounds<NB>(bvec), w, o,
                         [&](int j, const f32x4 (&c)[2]) { tl_flush_acc(acc, j, c); });
    }
    tl_epilogue_wave<NB, GELU, !LN>(a, x, stage, Yp, N, nbr, acc, b4);
    if constexpr (LN) {
        TlLnOperands<NB, NW, NW> lnop;
        tl_ln_fetch(lnop, a, x.wave, lane, x.m0, N);
        __syncthreads(); // every wave's part of the rows is staged
        tl_ln_rows(lnop, a, stage0, x.wave, lane, x.m0, Yp, N);
    }
#undef TL_PANEL_LOAD
}

// ---------------------------------------------------------------------------
// Resident-panel kernel: the plan kernel for K that fits one LDS panel (every
// BERT-base linear except FFN2).  Same tile stream and 4-stage pipeline as
// above, with three differences that take work off the critical path of a
// wave:
//  * a finished block-row is converted (bias, GELU, half) and written to the
//    wave's staging tile right where the stream crosses its boundary, so there
//    are no per-block-row accumulators to fold into and the conversion work
//    overlaps the weight loads already in flight;
//  * the next item's block-row boundaries and bias are requested before the
//    current item's stream starts, and its first four weight pairs before the
//    current item's output tile is stored - a wave sees one memory latency per
//    item instead of three;
//  * items that share the row panel reuse it without any barrier.
// ---------------------------------------------------------------------------
// Workgroup barrier that orders LDS traffic only.  __syncthreads() also fences
// global memory, which would make every wave drain the weight pairs it has
// just requested; this one is for hand-overs of LDS buffers.
__device__ __forceinline__ void tl_barrier_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

struct TlItem {
    int lin, cg, bn0, nbr, N;
    int q0, qend; // the wave's pairs (scalar loads: a wait for them is none for the panel's requests)
    f16 *Y;
    const int *cptr;
    const int *poff;
    const f16 *data;
    const f16 *bias;
};

// one finished 32x16 block-row tile -> wave-private staging tile
template <bool GELU>
__device__ __forceinline__ void tl_stage_tile(f16 *dst, int lds, f32x4 c0, f32x4 c1, f16x4 bj) {
    const f32x4 bf = __builtin_convertvector(bj, f32x4);
    f16x4 o0 = __builtin_convertvector(c0 + bf, f16x4);
    f16x4 o1 = __builtin_convertvector(c1 + bf, f16x4);
    if (GELU) {
        o0 = gelu4(o0);
        o1 = gelu4(o1);
    }
    *reinterpret_cast<f16x4 *>(dst) = o0;
    *reinterpret_cast<f16x4 *>(dst + 16 * lds) = o1;
}

template <int NB, bool GELU, int NW, bool LN, int BM = TL_BM>
__global__ void __launch_bounds__(NW * 64) tile_linear_resident_kernel(TL_HOT_PARAMS, const TlArgs args) {
    TL_HOT_TAKE(a, args, N[0])
    a.KC = a.K;
    // BM = 64: 64-row panels and items (four MFMAs per streamed W
    // pair), one workgroup per CU - the panel and the 64-row staging tiles fill
    // the LDS.  Chosen by the launcher where enough 64-row items exist.
    static_assert(BM == TL_BM || (BM == 2 * TL_BM && !LN), "64-row panels: without the LayerNorm epilogue");
    extern __shared__ __attribute__((aligned(16))) unsigned char tl_smem[];
    f16 *xs = reinterpret_cast<f16 *>(tl_smem);
    int rp, lin0, cg0;
    if (!tl_place(a, rp, lin0, cg0))
        return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int c16 = lane & 15, g4 = lane >> 4, khalf8 = (g4 & 1) * 8, hi = lane >> 5;
    const int ldx = a.KC + ((a.KC & 31) ? 0 : TL_PAD);
    const char *xlane = reinterpret_cast<const char *>(xs + c16 * ldx + khalf8);
    const int xrow16 = 16 * ldx * 2; // bytes between the two 16-row subtiles
    constexpr int lds = 16 * NB + 8; // halves per staged row
    f16 *const stage0 = xs + BM * ldx;
    f16 *const stage = stage0 + wave * (BM * (16 * NB + 8));
    f16 *const stage_lane = stage + c16 * lds + g4 * 4;
    const int lane_w = hi * 256 + c16 * 16 + khalf8; // lane's halves inside a 1 KB tile pair

    // pair-index boundaries of a wave's block-rows: lane j holds the start of
    // block-row j, lane NB the end of the last one (read back with v_readlane)
#define TL_BVEC(t_) ((t_).cptr[min((t_).bn0 + min(lane, NB), (t_).nbr)] >> 1)
    // (block-rows beyond the matrix read the last block-row's bias; their
    // output is never stored)
#define TL_BIAS(dst_, t_)                                                                         \
    _Pragma("unroll") for (int k = 0; k < NB; k++)                                                \
        dst_[k] = *reinterpret_cast<const f16x4 *>(                                               \
            (t_).bias + min((t_).bn0 + k, (t_).nbr - 1) * 16 + g4 * 4);
    // wave w fills panel rows (BM/NW)w ... (see tile_linear_plan_kernel)
#define TL_PANEL(rp_)                                                                             \
    {                                                                                             \
        const int pcpr = a.K >> 3;                                                                \
        constexpr int RPW = (BM + NW - 1) / NW; /* panel rows per wave */                         \
        _Pragma("unroll") for (int rr = 0; rr < RPW; rr++) {                                      \
            const int prow = wave * RPW + rr;                                                     \
            const int row = (rp_) * BM + prow;                                                    \
            if (row < a.M && (BM % NW == 0 || prow < BM)) {                                       \
                const f16 *src = a.X + (size_t)row * a.K;                                         \
                f16 *dstrow = xs + prow * ldx;                                                    \
                if (lane < pcpr)                                                                  \
                    load_lds16(src + lane * 8, dstrow);                                           \
                if (64 + lane < pcpr)                                                             \
                    load_lds16(src + (64 + lane) * 8, dstrow + 512);                              \
            }                                                                                     \
        }                                                                                         \
    }
    // behind the panel's requests and those of the first pairs
#define TL_PANEL_WAIT()                                                                           \
    {                                                                                             \
        __builtin_amdgcn_s_waitcnt(0x0F70); /* vmcnt(0): this wave's part has landed */           \
        __syncthreads();                    /* ... and everyone else's */                         \
    }
    // the first pairs of an item's stream
#define TL_PRELOAD(t_)                                                                            \
    {                                                                                             \
        q0 = (t_).q0;                                                                             \
        qend = (t_).qend;                                                                         \
        qlast = max(qend - 1, q0);                                                                \
        wdata = (t_).data;                                                                        \
        wpoff = (t_).poff;                                                                        \
        tl_preload(wdata, wpoff, lane_w, hi, q0, qlast, w, o);                                    \
    }

    // Per-linear arguments are read from the kernel-argument segment with a
    // run-time index (scalar loads).  Indexing the by-value struct itself would
    // make the compiler copy it to scratch memory, and chains of selects over
    // its constant-indexed elements compile to long branch ladders.
    typedef const __attribute__((address_space(4))) char *KArg;
    const KArg ka = (KArg)__builtin_amdgcn_kernarg_segment_ptr() + TL_HOT_BYTES;
#define TL_KARG(type_, field_, lin_)                                                              \
    (*(const __attribute__((address_space(4))) type_ *)(ka + offsetof(TlArgs, field_) +           \
                                                         (lin_) * sizeof(type_)))
    typedef const int *ListPtr;
    auto tl_item = [&](int lin, int cg, ListPtr cptr, int N) {
        TlItem t;
        t.lin = lin;
        t.cg = cg;
        t.bn0 = (cg * NW + wave) * NB;
        typedef f16 *YPtr;
        typedef const int *IPtr;
        typedef const f16 *HPtr;
        t.cptr = cptr;
        t.N = N;
        t.nbr = N >> 4;
        typedef const __attribute__((address_space(4))) int *IConst;
        const IConst cp = (IConst)t.cptr;
        // (all of them requested before the first is waited for)
        const int t0 = cp[min(t.bn0, t.nbr)], t1 = cp[min(t.bn0 + NB, t.nbr)];
        t.data = TL_KARG(HPtr, data, lin);
        t.poff = TL_KARG(IPtr, row_offset, lin);
        t.bias = TL_KARG(HPtr, bias, lin);
        t.Y = TL_KARG(YPtr, Y, lin);
        __builtin_amdgcn_sched_barrier(0);
        t.q0 = t0 >> 1;
        t.qend = t1 >> 1;
        return t;
    };
    // the panel's next item
    auto tl_next = [&](const TlItem &t) {
        const bool cw = t.cg + 1 == a.ncg;
        const int lin = cw ? (t.lin + 1 == a.nlin ? 0 : t.lin + 1) : t.lin;
        return tl_item(lin, cw ? 0 : t.cg + 1, TL_KARG(ListPtr, cptr, lin), TL_KARG(int, N, lin));
    };
    TL_PANEL(rp) // (requested with what came with the wave; the rest of the arguments is on its way)
    ListPtr cptr0 = hot_cptr;
    int n0 = hot_n;
    if (lin0 > 0) { // (wave-uniform)
        cptr0 = TL_KARG(ListPtr, cptr, lin0);
        n0 = TL_KARG(int, N, lin0);
    }
    TlItem cur = tl_item(lin0, cg0, cptr0, n0);

    int bvec = TL_BVEC(cur);
    f16x4 b4[NB];
    TL_BIAS(b4, cur)
    int q0, qend, qlast;
    const f16 *wdata;
    const int *wpoff;
    f16x8 w[TL_DEPTH];
    int o[TL_DEPTH];
    TL_PRELOAD(cur) // (in flight together with the panel)
    TL_PANEL_WAIT()

    for (int it = 0;; it++) {
        const bool has_next = it + 1 < a.ipw;
        const TlItem nxt = tl_next(cur); // (past the last item: a valid linear, never run)
        const int bvec_n = TL_BVEC(nxt);
        f16x4 b4n[NB];
        TL_BIAS(b4n, nxt)

        // a finished block-row goes straight to the wave's staging tile
        // bias of block-row j as a 0/1-masked sum (exact); a chain of selects
        // over b4[] would be turned into an indexed load and put the array into
        // scratch memory
        auto bias_of = [&](int j) {
            f16x4 bj = f16x4{0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < NB; k++)
                bj += b4[k] * ((j == k) ? (f16)1 : (f16)0);
            return bj;
        };
        const TlBounds<NB> bounds = tl_bounds<NB>(bvec);
        tl_stream<NB, BM / 16>(xlane, xrow16, wdata, wpoff, lane_w, hi, bounds, w, o, [&](int j, const f32x4 (&c)[BM / 16]) {
            const f16x4 bj = bias_of(j);
#pragma unroll
            for (int h = 0; h < BM / TL_BM; h++)
                tl_stage_tile<GELU>(stage_lane + h * 32 * lds + j * 16, lds, c[2 * h], c[2 * h + 1], bj);
        });
        // block-rows without any tile: bias only
#pragma unroll
        for (int k = 0; k < NB; k++)
            if (bounds.at[k] == bounds.at[k + 1]) {
#pragma unroll
                for (int h = 0; h < BM / TL_BM; h++)
                    tl_stage_tile<GELU>(stage_lane + h * 32 * lds + k * 16, lds, f32x4{0.f, 0.f, 0.f, 0.f},
                                        f32x4{0.f, 0.f, 0.f, 0.f}, b4[k]);
            }

        if (has_next)
            TL_PRELOAD(nxt)

        if constexpr (LN) {
            // the workgroup holds whole rows: skip connection + LayerNorm here
            TlLnOperands<NB, NW, NW> lnop;
            tl_ln_fetch(lnop, a, wave, lane, rp * BM, cur.N);
            __syncthreads(); // every wave's part of the rows is staged
            tl_ln_rows(lnop, a, stage0, wave, lane, rp * BM, cur.Y, cur.N);
            if (has_next)
                __syncthreads(); // the staging tiles are free again
        } else {
            // staging tile -> Y: 16-byte stores of 32*NB contiguous bytes per row
            const int nvalid = min(NB, cur.nbr - cur.bn0); // the last column group may be partial
            const int cpr = 2 * nvalid;                    // 16-byte chunks per row
            const int m0 = rp * BM;
            f16 *ybase = cur.Y + (size_t)m0 * cur.N + cur.bn0 * 16;
#pragma unroll
            for (int t = 0; t < NB * (BM / TL_BM); t++) {
                const int i = lane + 64 * t;
                const int r = i / (2 * NB), c = i - r * (2 * NB);
                if (c < cpr && m0 + r < a.M) {
                    const u32x4 v = *reinterpret_cast<const u32x4 *>(stage + r * lds + c * 8);
                    *reinterpret_cast<u32x4 *>(ybase + (size_t)r * cur.N + c * 8) = v;
                }
            }
        }
        if (!has_next)
            break;
        cur = nxt;
        bvec = bvec_n;
#pragma unroll
        for (int k = 0; k < NB; k++)
            b4[k] = b4n[k];
    }
#undef TL_PRELOAD
#undef TL_PANEL
#undef TL_PANEL_WAIT
#undef TL_BIAS
#undef TL_BVEC
#undef TL_KARG
}

// ---------------------------------------------------------------------------
// Chunked kernel with fetching waves: K beyond one LDS panel (second
// feed-forward linear, K = 3072, N = 768).  Twelve computing waves of NB
// block-rows each and four waves that do nothing but fetch (one alone takes
// 2.5 us a chunk); LN: the workgroup holds whole rows (one per row panel), and
// skip connection and LayerNorm follow.  K is walked in chunks through two LDS
// panel buffers; the fetching waves request chunk c+1 (global -> LDS DMA) as
// soon as the computing waves have left chunk c-1, so the fetch runs under
// chunk c's MFMAs.  They have to be waves of their own: loads return in order
// within a wave, so a panel request in a computing wave's queue would hold
// back every weight pair requested after it.  One LDS-only barrier per chunk
// hands over both "chunk c has landed" and "buffer (c+1)&1 is free".  The
// computing waves run the pair stream and 4-stage pipeline of the plan kernel,
// restarted per chunk with the first pairs requested before the barrier.
// ---------------------------------------------------------------------------
constexpr int TL_CWAVES = 12;
constexpr int TL_FWAVES = 4; // fetching waves, eight panel rows each
constexpr int TL_CTHREADS = (TL_CWAVES + TL_FWAVES) * 64;

template <int NB, bool GELU, bool LN>
__global__ void __launch_bounds__(TL_CTHREADS) tile_linear_chunked_kernel(TL_HOT_PARAMS, const TlArgs args) {
    TL_HOT_TAKE(a, args, KC)
    extern __shared__ __attribute__((aligned(16))) unsigned char tl_smem[];
    f16 *xs = reinterpret_cast<f16 *>(tl_smem);
    TlCtx x;
    int rp;
    if (!tl_place(a, rp, x.lin, x.cg))
        return;
    x.m0 = rp * TL_BM;
    x.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    x.lane = threadIdx.x & 63;
    x.c16 = x.lane & 15;
    x.g4 = x.lane >> 4;
    x.khalf8 = (x.g4 & 1) * 8;
    x.hi = x.lane >> 5;
    x.ldx = a.KC + ((a.KC & 31) ? 0 : TL_PAD);
    const int lin = x.lin;
    x.bn_wg = x.cg * (TL_CWAVES * NB);
    x.bn0 = x.bn_wg + x.wave * NB;
    x.ld_r = x.ld_c = 0;
    const int lane = x.lane;
    const int pbuf = TL_BM * x.ldx; // halves per panel buffer
    f16 *const stage0 = xs + 2 * pbuf;
    f16 *const Yp = TL_SEL(Y);
    const int N = TL_SEL(N);
    const int nbr = N >> 4;

    if (x.wave >= TL_CWAVES) {
        // ---- the fetching waves ----
        const int row0 = (x.wave - TL_CWAVES) * (TL_BM / TL_FWAVES);
#define TL_FETCH(c_)                                                                              \
    {                                                                                             \
        const int pk0 = (c_) * a.KC;                                                              \
        const int pcpr = min(a.KC, a.K - pk0) >> 3; /* 16-byte pieces per row, <= 96 */           \
        f16 *dst = xs + ((c_) & 1) * pbuf;                                                        \
        const int row1 = min(row0 + TL_BM / TL_FWAVES, a.M - x.m0);                               \
        for (int row = row0; row < row1; row++) {                                                 \
            const f16 *src = a.X + (size_t)(x.m0 + row) * a.K + pk0;                              \
            if (lane < pcpr)                                                                      \
                load_lds16(src + lane * 8, dst + row * x.ldx);                                    \
            if (64 + lane < pcpr)                                                                 \
                load_lds16(src + (64 + lane) * 8, dst + row * x.ldx + 512);                       \
        }                                                                                         \
    }
        TL_FETCH(0)
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
        if (a.nchunk > 1)
            TL_FETCH(1)
        tl_barrier_lds(); // chunk 0 is in LDS
        for (int c = 1; c < a.nchunk; c++) {
            __builtin_amdgcn_s_waitcnt(0x0F70); // chunk c has landed
            tl_barrier_lds();                   // ... and every wave has left chunk c-1
            if (c + 1 < a.nchunk)
                TL_FETCH(c + 1)
        }
#undef TL_FETCH
    } else {
        // ---- the computing waves ----
        const int *const cptr = TL_SEL(cptr);
        const int hi = x.hi;
        const f16 *const bias = TL_SEL(bias);
        f32x4 acc[NB][2];
        f16x4 b4[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) {
            acc[j][0] = f32x4{0.f, 0.f, 0.f, 0.f};
            acc[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            b4[j] = f16x4{0, 0, 0, 0};
            if (x.bn0 + j < nbr)
                b4[j] = *reinterpret_cast<const f16x4 *>(bias + (x.bn0 + j) * 16 + x.g4 * 4);
        }
        const int xrow16 = 16 * x.ldx * 2; // bytes between the two 16-row subtiles
        const f16 *const data = TL_SEL(data);
        const int *const poff = TL_SEL(row_offset);
        const unsigned lane_w = hi * 256 + x.c16 * 16 + x.khalf8; // lane's halves inside a 1 KB tile pair
        // pair-index boundaries of the wave's block-rows in the current chunk
        // (see tile_linear_plan_kernel); the next chunk's are requested a chunk ahead
        int bvec = cptr[min(x.bn0 + min(lane, NB), nbr)] >> 1;

        for (int c = 0; c < a.nchunk; c++) {
            const char *xlane =
                reinterpret_cast<const char *>(xs + (c & 1) * pbuf + x.c16 * x.ldx + x.khalf8);
            const int q0 = __builtin_amdgcn_readfirstlane(bvec);
            const int qend = __builtin_amdgcn_readlane(bvec, NB);
            const int qlast = max(qend - 1, q0);
            f16x8 w[TL_DEPTH];
            int o[TL_DEPTH];
            tl_preload(data, poff, lane_w, hi, q0, qlast, w, o);
            const int cn = min(c + 1, a.nchunk - 1);
            const int bvec_n = cptr[cn * nbr + min(x.bn0 + min(lane, NB), nbr)] >> 1;
            const int bcur = bvec;
            tl_barrier_lds();

            tl_stream<NB, 2>(xlane, xrow16, data, poff, lane_w, hi, tl_bounds<NB>(bcur), w, o,
                             [&](int j, const f32x4 (&c)[2]) { tl_flush_acc(acc, j, c); });
            bvec = bvec_n;
        }
        f16 *stage = stage0 + x.wave * tl_wave_stage_halves<NB>();
        tl_epilogue_wave<NB, GELU, !LN>(a, x, stage, Yp, N, nbr, acc, b4);
    }
    if constexpr (LN) {
        TlLnOperands<NB, TL_CWAVES, TL_CWAVES + TL_FWAVES> lnop;
        tl_ln_fetch(lnop, a, x.wave, lane, x.m0, N);
        __syncthreads(); // every computing wave's part of the rows is staged
        tl_ln_rows(lnop, a, stage0, x.wave, lane, x.m0, Yp, N);
    }
}

// ---------------------------------------------------------------------------
// The chunked kernel on 48-row panels: a computing wave has one block-row, or
// (SPLIT) two waves share one, each with half of the pairs of every chunk.
//
// What bounds these kernels is what a CU takes in - X by DMA, W past the vector
// memory path, 100 to 120 GB/s together - so the best workgroup is the one whose
// panel and lists are equally large.  1536 rows 3072 -> 768 at 50 %: 32 rows x 192
// columns are 197 KB of X and 590 of W on 192 CUs, 48 x 96 are 295 and 295 on 256;
// 2000 rows 4096 -> 1024 at 80 %: 32 x 384 are 262 and 627 on 189, 48 x 192 393 and
// 313 on 252.  us, the other kernels / this: 3072 -> 768 50 % 2791 rows 20.1 / 16.1, 4523 32.4
// / 22.6, 10111 57.2 / 44.8; 80 % 4523 19.1 / 15.2, 10111 35.3 / 29.8; 4096 -> 1024 50 % 770 17.4 / 15.3, 2000
// 23.4 / 20.3, 5134 48.7 / 40.1; 80 % 5134 29.7 / 24.6; 2048 -> 512 80 % 8345 21.7 / 15.6.  With two block-rows
// a wave and more (NB) the panels of all rows fit fewer rounds.
// The panel buffer of the chunk before the last, which everyone has left, stages
// the result (and, SPLIT, the second waves' sums): whole rows of the column
// group, stored line-wise by all sixteen waves.
// ---------------------------------------------------------------------------
constexpr int TL_TALL = 3; // subtiles of a panel

template <int NB, bool SPLIT, bool GELU>
__global__ void __launch_bounds__(TL_CTHREADS) tile_linear_tall_kernel(TL_HOT_PARAMS, const TlArgs args) {
    static_assert(!SPLIT || NB == 1, "two waves share one block-row");
    TL_HOT_TAKE(a, args, KC)
    constexpr int MS = TL_TALL, BM = 16 * MS, BRS = SPLIT ? TL_CWAVES / 2 : TL_CWAVES * NB; // block-rows of a workgroup
    extern __shared__ __attribute__((aligned(16))) unsigned char tl_smem[];
    f16 *xs = reinterpret_cast<f16 *>(tl_smem);
    int rp, lin, cg;
    if (!tl_place(a, rp, lin, cg))
        return;
    const int m0 = rp * BM;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c16 = lane & 15, g4 = lane >> 4, khalf8 = (g4 & 1) * 8, hi = lane >> 5;
    const int ldx = a.KC + ((a.KC & 31) ? 0 : TL_PAD);
    const int pbuf = BM * ldx; // halves per panel buffer
    f16 *const Y = TL_SEL(Y);
    const int N = TL_SEL(N), nbr = N >> 4;
    constexpr int LDS = 16 * BRS + 8; // halves per staged row
    f16 *const stage = xs + (a.nchunk & 1) * pbuf;
    f32x4 *const red = reinterpret_cast<f32x4 *>(stage + BM * LDS);
    static_assert(BM * LDS * 2 % 16 == 0, "aligned sums");
    static_assert(BM * LDS * 2 + (SPLIT ? BRS * MS * 64 * 16 : 0) <= BM * TL_CHUNK * 2, "the staged rows and sums fit a panel buffer");
    if (wave >= TL_CWAVES) {
        // ---- the fetching waves ----
        const int row0 = (wave - TL_CWAVES) * (BM / TL_FWAVES);
        auto fetch = [&](int c) {
            const int pk0 = c * a.KC, pcpr = min(a.KC, a.K - pk0) >> 3; // 16-byte pieces per row, <= 96
            f16 *dst = xs + (c & 1) * pbuf;
            const int row1 = min(row0 + BM / TL_FWAVES, a.M - m0);
            for (int row = row0; row < row1; row++) {
                const f16 *src = a.X + (size_t)(m0 + row) * a.K + pk0;
                if (lane < pcpr)
                    load_lds16(src + lane * 8, dst + row * ldx);
                if (64 + lane < pcpr)
                    load_lds16(src + (64 + lane) * 8, dst + row * ldx + 512);
            }
        };
        fetch(0);
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
        if (a.nchunk > 1)
            fetch(1);
        tl_barrier_lds(); // chunk 0 is in LDS
        for (int c = 1; c < a.nchunk; c++) {
            __builtin_amdgcn_s_waitcnt(0x0F70); // chunk c has landed
            tl_barrier_lds();                   // ... and every wave has left chunk c-1
            if (c + 1 < a.nchunk)
                fetch(c + 1);
        }
        if (SPLIT)
            tl_barrier_lds();
    } else {
        // ---- the computing waves ----
        const int br = SPLIT ? wave >> 1 : wave * NB, half = SPLIT ? wave & 1 : 0, bn = cg * BRS + br;
        const int *const cptr = TL_SEL(cptr);
        const f16 *const data = TL_SEL(data);
        const int *const poff = TL_SEL(row_offset);
        const f16 *const bias = TL_SEL(bias);
        f32x4 acc[NB][MS];
        f16x4 b4[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) {
#pragma unroll
            for (int m = 0; m < MS; m++)
                acc[j][m] = f32x4{0.f, 0.f, 0.f, 0.f};
            b4[j] = *reinterpret_cast<const f16x4 *>(bias + min(bn + j, nbr - 1) * 16 + g4 * 4);
        }
        const unsigned lane_w = hi * 256 + c16 * 16 + khalf8;
        // lane k: first pair of block-row k in a chunk, then the end of the last one; the next chunk's are requested a chunk ahead
        auto ends = [&](int c) { return cptr[min(c, a.nchunk - 1) * nbr + min(bn + min(lane, NB), nbr)] >> 1; };
        int bvec = ends(0);
        for (int c = 0; c < a.nchunk; c++) {
            const char *const xlane = reinterpret_cast<const char *>(xs + (c & 1) * pbuf + c16 * ldx + khalf8);
            TlBounds<NB> b = tl_bounds<NB>(bvec);
            if (SPLIT) {
                const int st = b.at[0], len = b.at[1] - st;
                b.at[0] = st + ((len * half) >> 1);
                b.at[1] = st + ((len * (half + 1)) >> 1);
            }
            f16x8 w[TL_DEPTH];
            int o[TL_DEPTH];
            tl_preload(data, poff, lane_w, hi, b.at[0], max(b.at[NB] - 1, b.at[0]), w, o);
            bvec = ends(c + 1);
            tl_barrier_lds();
            tl_stream<NB, MS>(xlane, 16 * ldx * 2, data, poff, lane_w, hi, b, w, o,
                              [&](int j, const f32x4 (&s)[MS]) { tl_flush_acc(acc, j, s); });
        }
        if (SPLIT) {
            if (half)
#pragma unroll
                for (int m = 0; m < MS; m++)
                    red[(br * MS + m) * 64 + lane] = acc[0][m];
            tl_barrier_lds();
            if (!half)
#pragma unroll
                for (int m = 0; m < MS; m++)
                    acc[0][m] += red[(br * MS + m) * 64 + lane];
        }
        if (!half)
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int m = 0; m < MS; m++) {
                    f16x4 v;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        v[r] = (f16)(acc[j][m][r] + (float)b4[j][r]);
                        if (GELU)
                            v[r] = gelu_h(v[r]);
                    }
                    *reinterpret_cast<f16x4 *>(stage + (m * 16 + c16) * LDS + (br + j) * 16 + g4 * 4) = v;
                }
    }
    tl_barrier_lds(); // the rows are staged
    const int col0 = cg * BRS * 16, cpr = 2 * BRS; // 16-byte pieces per row
    for (int i = threadIdx.x; i < BM * cpr; i += TL_CTHREADS) {
        const int r = i / cpr, c = i - r * cpr;
        if (m0 + r < a.M && col0 + c * 8 < N)
            *reinterpret_cast<u32x4 *>(Y + (size_t)(m0 + r) * N + col0 + c * 8) = *reinterpret_cast<const u32x4 *>(stage + r * LDS + c * 8);
    }
}

// ---------------------------------------------------------------------------
// Fused feed-forward block: Y = LayerNorm(skip + W2 * gelu(W1 * X + b1) + b2)
// in ONE launch (encoder/encoder.cu:36-44 runs it as MLP1, MLP2 and
// skip_layernorm with the [rows x ffn] intermediate written to and read back
// from memory).  One workgroup of 16 waves per 32-row panel keeps the panel of
// X in LDS and walks the hidden dimension in chunks of the second plan's
// chunk width: phase p computes hidden columns [p*KC, (p+1)*KC) with the first
// linear (bias, GELU, rounded to half exactly like the stored intermediate)
// into one of two LDS buffers, then multiplies that buffer with chunk p of the
// second linear into register accumulators that live across all phases.  The
// hidden activations never leave the CU.  Each wave owns NB block-rows of
// either linear per phase.  The first linear runs one phase ahead of the
// second, and the hand-overs ("hidden buffer p is complete", "everyone has
// finished reading it") are event counters in LDS rather than barriers, so a
// wave only ever waits when it is a whole stream ahead of the slowest wave.
// WITH_O: the attention output projection with its skip connection and
// LayerNorm (encoder/encoder.cu:33-35) runs first on the same panel, and its
// normalised rows replace the panel in LDS - steps 6-10 of a layer in one
// launch.
// arguments: [linear 0 = projection (WITH_O),] then the first feed-forward
// linear (N = hidden width) and the second (N = output width, Y = output);
// K = input width, KC / nchunk = the second plan's chunking; skip / gamma /
// beta belong to the first LayerNorm that runs, gamma2 / beta2 to the second.
// ---------------------------------------------------------------------------
constexpr int TL_FFN_WAVES = 16;
constexpr int TL_FFN_MAX_PHASES = 16;

// Workgroup-local event counters in LDS: every wave adds one when it has
// finished a step, and a wave that needs everyone's result waits for the
// count.  Unlike s_barrier this lets a wave run ahead with other work and
// wait only when it is a whole step ahead of the slowest wave.
__device__ __forceinline__ void tl_signal(unsigned *ctr, int lane) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local"); // this wave's LDS writes first
    if (lane == 0)
        __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// The wait is bounded (about 4 million polls by default, tens of milliseconds):
// should a wave ever fail to signal, the waiting wave sets the process's
// wait-status word and goes on - the kernel ends with a wrong result instead of
// hanging the GPU, and the next launch of a fused kernel reports ET_ERR_HIP.
// Every launch site checks on the host that the phase count fits the counters
// (tile_launch_ffn).
__device__ __forceinline__ void tl_wait_count(unsigned *ctr, unsigned target, int spin, int *status, int lane) {
    for (int s = 0;; s++) {
        if ((unsigned)__builtin_amdgcn_readfirstlane(
                (int)__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) >= target)
            break;
        if (s >= spin) {
            if (lane == 0)
                __hip_atomic_store(status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int NB, bool WITH_O>
__global__ void __launch_bounds__(TL_FFN_WAVES * 64) tile_ffn_fused_kernel(const TlArgs a) {
    constexpr int L1 = WITH_O ? 1 : 0, L2 = L1 + 1; // the two feed-forward linears
    extern __shared__ __attribute__((aligned(16))) unsigned char tl_smem[];
    f16 *xs = reinterpret_cast<f16 *>(tl_smem);
    const int rp = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    if (rp >= a.nwg)
        return;
    constexpr int NW = TL_FFN_WAVES;
    TlCtx x;
    x.lin = 1;
    x.cg = 0;
    x.m0 = rp * TL_BM;
    x.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    x.lane = threadIdx.x & 63;
    x.c16 = x.lane & 15;
    x.g4 = x.lane >> 4;
    x.khalf8 = (x.g4 & 1) * 8;
    x.hi = x.lane >> 5;
    x.ldx = a.K + ((a.K & 31) ? 0 : TL_PAD);
    x.bn_wg = 0;
    x.bn0 = x.wave * NB;
    x.ld_r = x.ld_c = 0;
    const int wave = x.wave, lane = x.lane, c16 = x.c16, g4 = x.g4, hi = x.hi;
    const int ldx = x.ldx;
    const int ldh = a.KC + ((a.KC & 31) ? 0 : TL_PAD);
    f16 *const hs = xs + TL_BM * ldx; // two hidden buffers behind the X panel
    const int hbuf = TL_BM * ldh;
    // event counters behind the hidden buffers: [p] first linear of phase p
    // done, [TL_FFN_MAX_PHASES + p] second linear of phase p done
    unsigned *const ctr = reinterpret_cast<unsigned *>(hs + 2 * hbuf);
    const int N1 = a.N[L1], N2 = a.N[L2], nbr1 = N1 >> 4, nbr2 = N2 >> 4;
    const int hbr = a.KC >> 4; // hidden block-rows per phase
    const unsigned lane_w = hi * 256 + c16 * 16 + x.khalf8;

    // the X panel: wave w fetches rows 2w and 2w+1
    {
        const int pcpr = a.K >> 3;
#pragma unroll
        for (int rr = 0; rr < TL_BM / NW; rr++) {
            const int r = wave * (TL_BM / NW) + rr;
            if (x.m0 + r < a.M) {
                const f16 *src = a.X + (size_t)(x.m0 + r) * a.K;
                if (lane < pcpr)
                    load_lds16(src + lane * 8, xs + r * ldx);
                if (64 + lane < pcpr)
                    load_lds16(src + (64 + lane) * 8, xs + r * ldx + 512);
            }
        }
    }
    if (threadIdx.x < 2 * TL_FFN_MAX_PHASES)
        ctr[threadIdx.x] = 0;
    const int *const cptr1 = a.cptr[L1], *const cptr2 = a.cptr[L2];
    const f16 *const data1 = a.data[L1], *const data2 = a.data[L2];
    const int *const poff1 = a.row_offset[L1], *const poff2 = a.row_offset[L2];
    // pair-index boundaries of the wave's block-rows; block-rows past the
    // phase's range or the matrix are empty
    // (read with scalar loads: they do not queue behind the weight pairs in
    // flight, and no wait for them drains those)
    typedef const __attribute__((address_space(4))) int *ScalarInts;
    auto bounds_of = [&](ScalarInts base, int i0, int lim) {
        TlBounds<NB> b;
#pragma unroll
        for (int k = 0; k <= NB; k++)
            b.at[k] = base[min(i0 + k, lim)] >> 1;
        return b;
    };
#define TL_FFN_BOUNDS1(p_) bounds_of((ScalarInts)cptr1, (p_) * hbr + wave * NB, min(((p_) + 1) * hbr, nbr1))
#define TL_FFN_BOUNDS2(p_) bounds_of((ScalarInts)cptr2 + (p_) * nbr2, wave * NB, nbr2)
#define TL_FFN_BIAS1(dst_, p_)                                                                    \
    _Pragma("unroll") for (int k = 0; k < NB; k++)                                                \
        dst_[k] = *reinterpret_cast<const f16x4 *>(                                               \
            a.bias[L1] + min((p_) * hbr + wave * NB + k, nbr1 - 1) * 16 + g4 * 4);
    f32x4 acc[NB][2];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        acc[j][0] = f32x4{0.f, 0.f, 0.f, 0.f};
        acc[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const char *const xlane1 = reinterpret_cast<const char *>(xs + c16 * ldx + x.khalf8);
    const int xrow1 = 16 * ldx * 2, xrow2 = 16 * ldh * 2;

    // One stream of the first linear: hidden columns of phase p_ (bias, GELU,
    // half) into hidden buffer p_ & 1.  w_/o_ hold its first pairs already.
#define TL_FFN_FIRST(p_, bounds_, b1_, w_, o_)                                                      \
    {                                                                                             \
        f16 *const hlane = hs + ((p_) & 1) * hbuf + c16 * ldh + wave * NB * 16 + g4 * 4;          \
        tl_stream<NB, 2>(xlane1, xrow1, data1, poff1, lane_w, hi, bounds_, w_, o_,                \
                      [&](int j, const f32x4 (&c)[2]) {                                           \
                          f16x4 bj = f16x4{0, 0, 0, 0};                                           \
                          _Pragma("unroll") for (int k = 0; k < NB; k++)                          \
                              bj += b1_[k] * ((j == k) ? (f16)1 : (f16)0);                        \
                          tl_stage_tile<true>(hlane + j * 16, ldh, c[0], c[1], bj);               \
                      });                                                              \
        /* block-rows of this phase without any tile: bias only */                                \
        const int lim1 = min(((p_) + 1) * hbr, nbr1);                                             \
        _Pragma("unroll") for (int k = 0; k < NB; k++)                                            \
            if ((p_) * hbr + wave * NB + k < lim1 &&                                              \
                bounds_.at[k] == bounds_.at[k + 1])                                               \
                tl_stage_tile<true>(hlane + k * 16, ldh, f32x4{0.f, 0.f, 0.f, 0.f},               \
                                    f32x4{0.f, 0.f, 0.f, 0.f}, b1_[k]);                           \
        tl_signal(ctr + (p_), lane);                                                              \
    }
#define TL_FFN_PRELOAD(data_, poff_, bounds_, w_, o_)                                               \
    {                                                                                             \
        const int q0_ = bounds_.at[0], qe_ = bounds_.at[NB];                                      \
        tl_preload(data_, poff_, lane_w, hi, q0_, max(qe_ - 1, q0_), w_, o_);                     \
    }

    // Stream order (F = first linear, S = second).  Half of the waves run
    // F(0) F(1) S(0) F(2) S(1) ... S(last), the first linear one phase ahead;
    // the other half F(0) S(0) F(1) S(1) ...  Both orders respect "S(p) after
    // every wave's F(p)" and "F(p+2) after every wave's S(p)" (the hidden buffer
    // it overwrites), what a wave waits for was usually finished a stream ago,
    // and at most times the two halves of a SIMD's waves are in different kinds
    // of stream: F streams load the vector ALU (GELU), S streams hardly do.
    // Register set A serves F(0) and every S, set B every later F.
    f16x8 wA[TL_DEPTH], wB[TL_DEPTH];
    int oA[TL_DEPTH], oB[TL_DEPTH];
    TlBounds<NB> boundsF = TL_FFN_BOUNDS1(0);
    f16x4 b1[NB];
    TL_FFN_BIAS1(b1, 0)
    TlBounds<NB> boundsFn = TL_FFN_BOUNDS1(min(1, a.nchunk - 1));
    f16x4 b1n[NB];
    TL_FFN_BIAS1(b1n, min(1, a.nchunk - 1))
    TlBounds<NB> boundsS = TL_FFN_BOUNDS2(0);
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): this wave's part of the panel has landed
    if constexpr (WITH_O) {
        // Linear 0 (the attention output projection) with its skip connection
        // and LayerNorm comes first: the panel just fetched holds the attention
        // output, and the normalised rows (rounded to half, as the reference
        // stores them) replace it in LDS as the feed-forward block's input and
        // as the skip operand of the final LayerNorm.
        const int NO = a.N[0], nbrO = NO >> 4; // == K
        const TlBounds<NB> boundsO = bounds_of((ScalarInts)a.cptr[0], wave * NB, nbrO);
        f16x4 bO[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) {
            bO[j] = f16x4{0, 0, 0, 0};
            if (x.bn0 + j < nbrO)
                bO[j] = *reinterpret_cast<const f16x4 *>(a.bias[0] + (x.bn0 + j) * 16 + g4 * 4);
        }
        TL_FFN_PRELOAD(a.data[0], a.row_offset[0], boundsO, wB, oB)
        tl_barrier_lds(); // the whole panel has landed; the counters are zero
        {
            tl_stream<NB, 2>(xlane1, xrow1, a.data[0], a.row_offset[0], lane_w, hi, boundsO, wB, oB,
                             [&](int j, const f32x4 (&c)[2]) { tl_flush_acc(acc, j, c); });
        }
        TL_FFN_PRELOAD(data1, poff1, boundsF, wA, oA)
        TlLnOperands<NB, NW, NW> lnop1; // (requested here: their latency runs under the wait for the other waves)
        tl_ln_fetch_skip(lnop1, a.M, wave, lane, x.m0, NO, a.skip + (long)x.m0 * NO, (long)NO);
        // staging tiles in the hidden buffers, which nobody uses yet
        tl_epilogue_wave<NB, false, false>(a, x, hs + wave * tl_wave_stage_halves<NB>(), nullptr, NO, nbrO, acc,
                                           bO);
#pragma unroll
        for (int j = 0; j < NB; j++) {
            acc[j][0] = f32x4{0.f, 0.f, 0.f, 0.f};
            acc[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        tl_ln_fetch_scale(lnop1, lane, NO, a.gamma, a.beta);
        tl_barrier_lds(); // every wave's part is staged, and everyone has left the attention panel
        tl_ln_rows_at(lnop1, a.M, hs, wave, lane, x.m0, NO, xs, (long)ldx);
    } else {
        TL_FFN_PRELOAD(data1, poff1, boundsF, wA, oA)
    }
    tl_barrier_lds(); // the feed-forward input panel is complete (and the counters are zero)
    if (a.nchunk > 1)
        TL_FFN_PRELOAD(data1, poff1, boundsFn, wB, oB)
    TL_FFN_FIRST(0, boundsF, b1, wA, oA)

    const int behind = (wave >> 2) & 1; // (a SIMD's waves are w, w+4, w+8, w+12)
    for (int p = 0; p < a.nchunk; p++) {
        const TlBounds<NB> boundsSn = TL_FFN_BOUNDS2(min(p + 1, a.nchunk - 1));
        TL_FFN_PRELOAD(data2, poff2, boundsS, wA, oA) // S(p), a stream ahead (unless no F runs in between)
        const int fq = p + 1 - behind; // the first-linear phase this wave runs before S(p)
        if (fq >= 1 && fq < a.nchunk) {
            const TlBounds<NB> boundsF2 = TL_FFN_BOUNDS1(min(fq + 1, a.nchunk - 1)); // (scalar loads, used after the stream)
            if (fq >= 2) // F(fq) overwrites the buffer that S(fq-2) read
                tl_wait_count(ctr + TL_FFN_MAX_PHASES + fq - 2, NW, a.spin, a.status, lane);
            TL_FFN_FIRST(fq, boundsFn, b1n, wB, oB)
            boundsFn = boundsF2;
            if (fq + 1 < a.nchunk) { // F(fq+1), a stream (or two) ahead
                TL_FFN_PRELOAD(data1, poff1, boundsFn, wB, oB)
                TL_FFN_BIAS1(b1n, fq + 1)
            }
        }
        tl_wait_count(ctr + p, NW, a.spin, a.status, lane); // hidden buffer p & 1 is complete
        {
            const char *const xlane2 =
                reinterpret_cast<const char *>(hs + (p & 1) * hbuf + c16 * ldh + x.khalf8);
            tl_stream<NB, 2>(xlane2, xrow2, data2, poff2, lane_w, hi, boundsS, wA, oA,
                             [&](int j, const f32x4 (&c)[2]) { tl_flush_acc(acc, j, c); });
            tl_signal(ctr + TL_FFN_MAX_PHASES + p, lane);
        }
        boundsS = boundsSn;
    }
#undef TL_FFN_BOUNDS1
#undef TL_FFN_BOUNDS2
#undef TL_FFN_BIAS1
#undef TL_FFN_FIRST
#undef TL_FFN_PRELOAD

    // output rows -> staging tiles over the (now unused) panel and hidden
    // buffers, then skip connection + LayerNorm over whole rows
    TlLnOperands<NB, NW, NW> lnop;
    if constexpr (WITH_O) { // the skip operand is the panel in LDS
        tl_ln_fetch_skip(lnop, a.M, wave, lane, x.m0, N2, xs, (long)ldx);
        tl_ln_fetch_scale(lnop, lane, N2, a.gamma2, a.beta2);
    } else {
        tl_ln_fetch(lnop, a, wave, lane, x.m0, N2);
    }
    f16x4 b2[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        b2[j] = f16x4{0, 0, 0, 0};
        if (x.bn0 + j < nbr2)
            b2[j] = *reinterpret_cast<const f16x4 *>(a.bias[L2] + (x.bn0 + j) * 16 + g4 * 4);
    }
    tl_barrier_lds(); // every wave has left the hidden buffers
    f16 *const stage0 = WITH_O ? hs : xs;
    tl_epilogue_wave<NB, false, false>(a, x, stage0 + wave * tl_wave_stage_halves<NB>(), a.Y[L2], N2, nbr2,
                                       acc, b2);
    __syncthreads(); // every wave's part of the rows is staged
    tl_ln_rows(lnop, a, stage0, wave, lane, x.m0, a.Y[L2], N2);
}

// ---------------------------------------------------------------------------
// Generic kernel: the caller's own tile_mat (TL_RAW / TL_FILTER) or a dense
// row-major weight (TL_DENSE).  Same mapping, plain per-block-row loops with
// per-lane predicates.
// ---------------------------------------------------------------------------
template <int NB, bool GELU, int MODE>
__global__ void __launch_bounds__(TL_THREADS) tile_linear_generic_kernel(const TlArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char tl_smem[];
    f16 *xs = reinterpret_cast<f16 *>(tl_smem);
    TlCtx x;
    if (!tl_context(a, NB, x))
        return;
    const int lin = x.lin;
    f16 *const Yp = TL_SEL(Y);
    const int *const cptr = TL_SEL(cptr);
    const int *const roff = TL_SEL(row_offset);
    const f16 *const data = TL_SEL(data);
    const f16 *const bias = TL_SEL(bias);
    const int N = TL_SEL(N);
    const int nbr = N >> 4;
    const int hi = x.hi;

    f32x4 acc[NB][2];
    f16x4 b4[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        acc[j][0] = f32x4{0.f, 0.f, 0.f, 0.f};
        acc[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        b4[j] = f16x4{0, 0, 0, 0};
        if (x.bn0 + j < nbr)
            b4[j] = *reinterpret_cast<const f16x4 *>(bias + (x.bn0 + j) * 16 + x.g4 * 4);
    }
    const f16 *xlane = xs + x.c16 * x.ldx + x.khalf8;
    const int xrow16 = 16 * x.ldx;
    const bool rowok = (x.m0 + x.ld_r) < a.M;
    const u32x4 *xsrc = reinterpret_cast<const u32x4 *>(a.X + (size_t)(x.m0 + x.ld_r) * a.K);
    u32x4 *xdst = reinterpret_cast<u32x4 *>(xs + x.ld_r * x.ldx);
    const f16x8 zero8 = f16x8{0, 0, 0, 0, 0, 0, 0, 0};

    for (int c = 0; c < a.nchunk; c++) {
        const int k0 = c * a.KC;
        const int kc = min(a.KC, a.K - k0);
        if (c > 0)
            __syncthreads();
        {
            const int cpr = kc >> 3;
            u32x4 pv[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int cc = x.ld_c + 16 * u;
                pv[u] = u32x4{0u, 0u, 0u, 0u};
                if (rowok && cc < cpr)
                    pv[u] = xsrc[(k0 >> 3) + cc];
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int cc = x.ld_c + 16 * u;
                if (cc < cpr)
                    xdst[cc] = pv[u];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const int bn = x.bn0 + j;
            if (bn >= nbr)
                continue;
            if (MODE == TL_DENSE) {
                const f16 *wrow = data + (size_t)(bn * 16 + x.c16) * a.K + k0 + x.khalf8;
                const int nt = kc >> 4;
                for (int i = 0; i < nt; i += 2) {
                    const bool ok = i + hi < nt;
                    const int off = (ok ? i + hi : i) * 16;
                    f16x8 w = zero8;
                    if (ok)
                        w = *reinterpret_cast<const f16x8 *>(wrow + off);
                    const f16x8 x0 = *reinterpret_cast<const f16x8 *>(xlane + off);
                    const f16x8 x1 = *reinterpret_cast<const f16x8 *>(xlane + off + xrow16);
                    acc[j][0] = mfma16x16x32(w, x0, acc[j][0]);
                    acc[j][1] = mfma16x16x32(w, x1, acc[j][1]);
                }
            } else {
                const int fs = cptr[bn];
                const int fe = cptr[bn + 1];
                const f16 *wlane = data + x.c16 * 16 + x.khalf8;
                for (int i = fs; i < fe; i += 2) {
                    const int ti = min(i + hi, fe - 1);
                    const int off = roff[ti] - k0;
                    const bool ok = (i + hi < fe) && off >= 0 && off < kc;
                    if (MODE == TL_FILTER && __builtin_amdgcn_ballot_w64(ok) == 0)
                        continue;
                    f16x8 w = zero8, x0 = zero8, x1 = zero8;
                    if (ok) {
                        w = *reinterpret_cast<const f16x8 *>(wlane + (size_t)ti * 256);
                        x0 = *reinterpret_cast<const f16x8 *>(xlane + off);
                        x1 = *reinterpret_cast<const f16x8 *>(xlane + off + xrow16);
                    }
                    acc[j][0] = mfma16x16x32(w, x0, acc[j][0]);
                    acc[j][1] = mfma16x16x32(w, x1, acc[j][1]);
                }
            }
        }
    }
    tl_epilogue<NB, GELU>(a, x, xs, Yp, N, nbr, acc, b4);
}

#undef TL_SEL

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
template <int NB, bool GELU, int MODE>
static int launch_inst(const TlArgs &a, size_t lds, hipStream_t st) {
    const dim3 grid(a.per_xcd * 8), block(TL_THREADS);
    if constexpr (MODE == TL_PLAN) {
        // (block-rows per wave beyond 3 never paid off for the plan kernels)
        constexpr int PNB = NB > 3 ? 3 : NB;
        if (a.nchunk == 1) {
            constexpr auto k = &tile_linear_resident_kernel<PNB, GELU, TL_WAVES, false>;
            launch_kernel<k>(grid, block, lds, st, TL_HOT(a, N[0]), a);
        } else {
            constexpr auto k = &tile_linear_plan_kernel<PNB, GELU, TL_WAVES, false>;
            launch_kernel<k>(grid, block, lds, st, TL_HOT(a, KC), a);
        }
    } else {
        launch_kernel<&tile_linear_generic_kernel<NB, GELU, MODE>>(grid, block, lds, st, a);
    }
    return launch_status("tile_linear launch");
}

template <bool GELU, int MODE>
static int launch_nb(int nb, const TlArgs &a, size_t lds, hipStream_t st) {
    switch (nb) {
    case 1: return launch_inst<1, GELU, MODE>(a, lds, st);
    case 2: return launch_inst<2, GELU, MODE>(a, lds, st);
    case 3: return launch_inst<3, GELU, MODE>(a, lds, st);
    case 4: return launch_inst<4, GELU, MODE>(a, lds, st);
    default: return launch_inst<6, GELU, MODE>(a, lds, st);
    }
}

// Fused linear + skip + LayerNorm: one workgroup of 16 waves covers whole rows.
constexpr int TL_LN_WAVES = 16;

template <int NB>
static int launch_ln_inst(const TlArgs &a, size_t lds, hipStream_t st) {
    const dim3 grid(a.per_xcd * 8), block(TL_LN_WAVES * 64);
    if (a.nchunk == 1) {
        constexpr auto k = &tile_linear_resident_kernel<NB, false, TL_LN_WAVES, true>;
        launch_kernel<k>(grid, block, lds, st, TL_HOT(a, N[0]), a);
    } else {
        constexpr auto k = &tile_linear_plan_kernel<NB, false, TL_LN_WAVES, true>;
        launch_kernel<k>(grid, block, lds, st, TL_HOT(a, KC), a);
    }
    return launch_status("tile_linear+LayerNorm launch");
}

// block-rows per wave of the fused kernel for a matrix of nbr block-rows; 0 if
// the rows do not fit one workgroup (then the caller runs the two kernels)
static int ln_block_rows(int nbr) {
    const int need = (nbr + TL_LN_WAVES - 1) / TL_LN_WAVES;
    return need <= 3 ? need : need == 4 ? 4 : need <= 6 ? 6 : 0;
}

template <int NB>
static int launch_chunked_ln_inst(const TlArgs &a, size_t lds, hipStream_t st) {
    constexpr auto k = &tile_linear_chunked_kernel<NB, false, true>;
    launch_kernel<k>(dim3(a.per_xcd * 8), dim3(TL_CTHREADS), lds, st, TL_HOT(a, KC), a);
    return launch_status("tile_linear+LayerNorm (chunked) launch");
}

template <int NB, bool SPLIT, bool GELU>
static int launch_tall(const TlArgs &a, hipStream_t st) {
    ET_REQUIRE(a.KC == TL_CHUNK, ET_ERR_UNSUPPORTED, "48-row panels of %d columns instead of %d", a.KC, TL_CHUNK); // (what the kernel stages over)
    constexpr auto k = &tile_linear_tall_kernel<NB, SPLIT, GELU>;
    const size_t lds = 2 * (size_t)16 * TL_TALL * (a.KC + ((a.KC & 31) ? 0 : TL_PAD)) * sizeof(f16);
    launch_kernel<k>(dim3(a.per_xcd * 8), dim3(TL_CTHREADS), lds, st, TL_HOT(a, KC), a);
    return launch_status("tile_linear (48-row panels) launch");
}

template <int NB, bool GELU>
static int launch_chunked_inst(const TlArgs &a, size_t lds, hipStream_t st) {
    constexpr auto k = &tile_linear_chunked_kernel<NB, GELU, false>;
    launch_kernel<k>(dim3(a.per_xcd * 8), dim3(TL_CTHREADS), lds, st, TL_HOT(a, KC), a);
    return launch_status("tile_linear (chunked) launch");
}

static int g_tile_ln_chunked = 1;
static std::atomic<int> g_tile_chunked{-1}; // et_tuning_set("tile_chunked")
static int g_tile_fuse_ffn = 2; // et_tuning_set("tile_fuse_ffn"): 1 feed-forward block, 2 whole layer tail

// LDS bytes of the fused feed-forward kernel: X panel, two hidden buffers (the
// output staging tiles reuse their storage)
static size_t ffn_lds_bytes(int K1, int KC2) {
    const size_t ldx = K1 + ((K1 & 31) ? 0 : TL_PAD), ldh = KC2 + ((KC2 & 31) ? 0 : TL_PAD);
    size_t panels = (size_t)TL_BM * (ldx + 2 * ldh) * sizeof(f16) + 2 * TL_FFN_MAX_PHASES * sizeof(unsigned);
    const size_t staging = (size_t)TL_FFN_WAVES * TL_BM * (16 * 3 + 8) * sizeof(f16);
    return std::max(panels, staging);
}

// pO: the attention output projection in front of the block (the whole layer
// tail in one launch), or null
static int tile_launch_ffn(const TlProblem *pO, const TlProblem &p1, const TlProblem &p2, const f16 *X,
                           int M, int K1, int KC2, int nchunk2, const f16 *skip, const f16 *gamma,
                           const f16 *beta, const f16 *gamma2, const f16 *beta2, hipStream_t st) {
    // the kernel's LDS event counters cover TL_FFN_MAX_PHASES phases: every launch passes through here
    ET_REQUIRE(nchunk2 >= 1 && nchunk2 <= TL_FFN_MAX_PHASES, ET_ERR_UNSUPPORTED,
               "fused feed-forward: %d phases, the kernel covers %d", nchunk2, TL_FFN_MAX_PHASES);
    // a wave of an earlier launch that gave up an LDS wait left a wrong result behind: say so once
    int *const status = wait_status_device();
    ET_REQUIRE(status, ET_ERR_HIP, "fused feed-forward: no wait-status word");
    {
        const int rc = check_wait_status("fused feed-forward");
        if (rc != ET_OK)
            return rc;
    }
    TlArgs a;
    memset(&a, 0, sizeof(a));
    a.status = status;
    a.spin = tail_spin();
    const TlProblem *ps[3] = {pO ? pO : &p1, pO ? &p1 : &p2, &p2};
    for (int i = 0; i < TL_MAX_LIN; i++) {
        const TlProblem &p = *ps[std::min(i, 2)];
        a.Y[i] = p.Y;
        a.cptr[i] = p.cptr;
        a.row_offset[i] = p.row_offset;
        a.data[i] = p.data;
        a.bias[i] = p.bias;
        a.N[i] = p.N;
    }
    a.X = X;
    a.nlin = pO ? 3 : 2;
    a.gamma2 = gamma2;
    a.beta2 = beta2;
    a.M = M;
    a.K = K1;
    a.KC = KC2;
    a.nchunk = nchunk2;
    a.ncg = 1;
    a.nwg = (M + TL_BM - 1) / TL_BM; // (one workgroup per panel: div and ncg are 1)
    a.ipw = a.div = 1;
    a.per_xcd = (a.nwg + 7) / 8;
    a.skip = skip;
    a.gamma = gamma;
    a.beta = beta;
    const size_t lds = ffn_lds_bytes(K1, KC2);
    if (pO) {
        constexpr auto k = &tile_ffn_fused_kernel<3, true>;
        launch_kernel<k>(dim3(a.per_xcd * 8), dim3(TL_FFN_WAVES * 64), lds, st, a);
    } else {
        constexpr auto k = &tile_ffn_fused_kernel<3, false>;
        launch_kernel<k>(dim3(a.per_xcd * 8), dim3(TL_FFN_WAVES * 64), lds, st, a);
    }
    return launch_status("fused feed-forward launch");
}

static int tile_launch_ln(const TlProblem &p, const f16 *X, int M, int K, int KC, int nchunk,
                          const f16 *skip, const f16 *gamma, const f16 *beta, hipStream_t st) {
    TlArgs a;
    memset(&a, 0, sizeof(a));
    for (int i = 0; i < TL_MAX_LIN; i++) {
        a.Y[i] = p.Y;
        a.cptr[i] = p.cptr;
        a.row_offset[i] = p.row_offset;
        a.data[i] = p.data;
        a.bias[i] = p.bias;
        a.N[i] = p.N;
    }
    a.X = X;
    a.nlin = 1;
    a.M = M;
    a.K = K;
    a.KC = KC;
    a.nchunk = nchunk;
    a.ncg = 1;
    a.nwg = (M + TL_BM - 1) / TL_BM; // (one workgroup per panel: div and ncg are 1)
    a.ipw = a.div = 1;
    a.per_xcd = (a.nwg + 7) / 8;
    a.skip = skip;
    a.gamma = gamma;
    a.beta = beta;
    const size_t lds_x = (size_t)TL_BM * (KC + ((KC & 31) ? 0 : TL_PAD)) * sizeof(f16);
    // K in chunks and rows narrow enough for twelve waves of <= 4 block-rows:
    // the double-buffered kernel with fetching waves
    const int cnb = (p.nbr + TL_CWAVES - 1) / TL_CWAVES;
    if (nchunk > 1 && cnb <= 4 && g_tile_ln_chunked) {
        const size_t lds = 2 * lds_x + (size_t)TL_CWAVES * TL_BM * (16 * cnb + 8) * sizeof(f16);
        switch (cnb) {
        case 1: return launch_chunked_ln_inst<1>(a, lds, st);
        case 2: return launch_chunked_ln_inst<2>(a, lds, st);
        case 3: return launch_chunked_ln_inst<3>(a, lds, st);
        default: return launch_chunked_ln_inst<4>(a, lds, st);
        }
    }
    const int nb = ln_block_rows(p.nbr);
    const size_t lds = lds_x + (size_t)TL_LN_WAVES * TL_BM * (16 * nb + 8) * sizeof(f16);
    switch (nb) {
    case 1: return launch_ln_inst<1>(a, lds, st);
    case 2: return launch_ln_inst<2>(a, lds, st);
    case 3: return launch_ln_inst<3>(a, lds, st);
    case 4: return launch_ln_inst<4>(a, lds, st);
    default: return launch_ln_inst<6>(a, lds, st);
    }
}

// Tuning knobs (et_tuning_set): 0 = automatic.  Those that the choice of a form reads may be set while another thread
// launches: that launch takes the old or the new value, later ones the new.
static std::atomic<int> g_tile_nb{0};
static std::atomic<int> g_tile_min_wgs{512};
static std::atomic<int> g_tile_ipw{0};
static std::atomic<int> g_tile_form{-1}; // et_tuning_set("tile_form"): index in tl_forms
static int g_tile_fuse_ln = 1;
static int g_tile_min_panels = 0; // fewest panels of the fused linear + LayerNorm and layer tail kernels, 0 = automatic
// the layer tail's choice is forced (a layer then runs its steps as separate launches)
bool tail_tuned() { return g_tile_min_panels != 0 || g_tile_fuse_ffn != 2; }

// Block-rows per wave.  Measured on the BERT-base shapes (rows 4096..8192):
// three block-rows per wave is the best trade between panel re-reads (fewer
// with larger NB) and register pressure / workgroup count (better with
// smaller NB); small problems fall back to smaller NB to get enough
// workgroups for 256 CUs.
static int choose_nb(int nrp, int nbr_max, int nlin) {
    const int forced = g_tile_nb;
    if (forced == 1 || forced == 2 || forced == 3 || forced == 4 || forced == 6)
        return forced;
    const int cand[3] = {3, 2, 1};
    for (int i = 0; i < 3; i++) {
        const int nb = cand[i];
        const int ncg = (nbr_max + TL_WAVES * nb - 1) / (TL_WAVES * nb);
        if ((long)nrp * ncg * nlin >= g_tile_min_wgs)
            return nb;
    }
    return 1;
}

constexpr int TL_BM64 = 2 * TL_BM;
static std::atomic<int> g_tile_bm64{1}; // et_tuning_set("tile_bm64")
// rows from which the row-pruned linear runs the register-blocked GEMM (et_tuning_set("row_gemm_min_rows");
// below, 128 x 128 blocks leave most CUs without work and the tile kernels win)
static int g_row_gemm_min_rows = 1024;
// fully populated plans as dense products: 1 by size, 0 never, 2 always (et_tuning_set("plan_dense"))
static int g_plan_dense = 1;

static std::atomic<int> g_tile_rows_most{-1}; // et_tuning_set("tile_splitk_rows"): most rows for which a plan runs on whole rows, -1 automatic
static int g_tile_splitk_k1 = 0;  // et_tuning_set("tile_splitk_k1"): 1: also plans of one chunk, up to tile_splitk_rows rows (-1: 128)

static std::atomic<int> g_tile_order{1}; // et_tuning_set("tile_order"): 0 panels slowest, 2 column groups slowest, 1 fewer bytes
// Whether consecutive workgroups walk the panels of a column group (tl_place): X and W in bytes, numbers of panels
// and of workgroups per panel.  Every L2 that has part of the work takes what all of the work shares, so W times eight
// is what bounds a launch of few rows: 256 rows, 1024 -> 4096: dense 14.2 -> 6.6 us, 50 % 10.0 -> 5.6; 768 -> 3072
// dense 9.7 -> 5.9; 128 rows 3072 -> 768 dense 9.8 -> 6.8.  Only up to x_most bytes of X: beyond, the L2s have time
// enough for W and the launch is up to 10 % slower in this order (1536 rows, 1024 -> 4096, 50 %: 18.7 and 20.9).
bool tl_order(double x_bytes, double w_bytes, long panels, long groups, double x_most) {
    const int order = g_tile_order;
    if (order != 1)
        return order == 2;
    return x_bytes <= x_most && std::min(groups, 8L) * x_bytes + w_bytes < x_bytes + std::min(panels, 8L) * w_bytes;
}
double tl_traffic_mb(double x_mb, double w_mb, long panels, long groups, double x_most) {
    return tl_order(x_mb, w_mb, panels, groups, x_most) ? std::min(groups, 8L) * x_mb + w_mb
                                                        : x_mb + std::min(panels, 8L) * w_mb;
}

// The forms of the single-panel kernel and the choice among them.  An item is a panel of 32 or 64 rows by waves x nb
// block-rows; a workgroup keeps its panel in LDS and does d consecutive items of it.  Small items put more CUs to work
// and end a round sooner, large ones fetch a panel less often and stream each kilobyte of W past more rows.  The choice
// is the least estimated time: per launch, per byte that the L2s take in, per round of workgroups on the busiest CU (a
// start and the stream's latency for each item), per panel, output, GELU and MFMA of the busiest CU, per byte of the
// result and per workgroup.  The figures (us) start from non-negative least squares over 12000 launches (512 / 768 / 1024
// inputs, 512 .. 4096 outputs, one or three linears, 0 .. 90 % pruned, 37 .. 32768 rows; 5 to 6 % off in the mean) and
// are then moved by up to a factor of two where that brings the choice closer to the fastest form: 0.5 % from it in the
// mean, 13 % at most (0.6 % where half of the row counts was left out); the rule before, a number of workgroups to aim
// for, was 6.3 %.  bench/linear_forms.py times the forms and fits the terms anew: on its 320 linears (launches of a graph)
// the estimates are 6 to 8 % off and all choices of this file together 1.4 % behind the fastest form, 19 % at most (2048
// -> 512 dense, 1343 rows: 12.4 against 10.4 us).  1536 rows 768 -> 3072, 50 %: 13.8 -> 11.7 us; 3500 rows 768 -> 768, 90 %:
// 7.3 -> 5.8; 2700 rows 768 -> 3072, 80 %: 16.1 -> 12.4.
struct TlForm {
    int rows, waves, nb;
};
static const TlForm tl_forms[] = {{TL_BM, 8, 1}, {TL_BM, 8, 2}, {TL_BM, 8, 3}, {TL_BM64, 12, 2}, {TL_BM64, 8, 3},
                                  {TL_BM64, 8, 2}, {TL_BM64, 8, 1}};
struct TlCost {
    double launch, traffic, traffic_over, round, item, item_nb, item_stream, panel, out, gelu, mfma, result, wg;
};
static const TlCost tl_cost32 = {2.48, 0.0586, 0.0614, 0.0, 0.458, 0.236, 0.0221, 0.173e-4, 0.403e-3, 0.382e-3, 0.171e-3, 0.192e-6, 0.668e-3},
                    tl_cost64 = {1.92, 0.0693, 0.0209, 0.696, 0.609, 0.381, 0.0884, 0.111e-4, 0.0, 0.534e-3, 0.0, 0.226e-6, 0.681e-3},
                    tl_cost64x12 = {2.80, 0.0152, 0.0728, 0.379, 0.0, 0.322, 0.113, 0.266e-4, 0.0, 0.841e-3, 0.0, 0.293e-6, 0.0};
struct TlChoice {
    const TlForm *form;
    int d, ncg, by_group;
    size_t lds;
    double us;
};
static TlChoice weigh_resident(const TlProblem *probs, int nlin, int M, int K, int nbr_max, bool gelu, int cus) {
    double pairs = 0.0, w_mb = 0.0, result = 0.0; // tile pairs per block-row; W and the result of all linears
    for (int i = 0; i < nlin; i++) {
        const double p = 0.5 * probs[i].ntile / probs[i].nbr;
        pairs += p / nlin;
        w_mb += p * probs[i].nbr * 1024e-6;
        result += (double)M * probs[i].N;
    }
    const double x_mb = 2e-6 * M * K;
    const int nb_set = g_tile_nb, form_set = g_tile_form, ipw_set = g_tile_ipw, bm64 = g_tile_bm64;
    const int fnb = nb_set >= 1 && nb_set <= 3 ? nb_set : 0;
    TlChoice best = {};
    auto lds_of = [&](const TlForm &f) {
        return (size_t)f.rows * (K + ((K & 31) ? 0 : TL_PAD)) * sizeof(f16) +
               (size_t)f.waves * f.rows * (16 * f.nb + 8) * sizeof(f16);
    };
    const TlForm *only = nullptr; // (tuning)
    if (form_set >= 0 && form_set < (int)(sizeof(tl_forms) / sizeof(tl_forms[0])) && lds_of(tl_forms[form_set]) <= 160 * 1024)
        only = &tl_forms[form_set];
    for (const TlForm &f : tl_forms) {
        if (only ? &f != only
                 : (f.rows == TL_BM ? (fnb ? f.nb != fnb : bm64 == 2) : fnb || bm64 == 0) ||
                       (f.waves == 12 && bm64 == 4))
            continue; // (tuning; a form of either height fits every K of one chunk)
        const size_t lds = lds_of(f);
        if (lds > 160 * 1024)
            continue;
        const TlCost &c = f.rows == TL_BM ? tl_cost32 : f.waves == 8 ? tl_cost64 : tl_cost64x12;
        const int ncg = (nbr_max + f.waves * f.nb - 1) / (f.waves * f.nb), per_panel = ncg * nlin;
        const long panels = (M + f.rows - 1) / f.rows;
        const long slots = f.rows == TL_BM && 2 * lds <= 160 * 1024 ? 2 : 1; // workgroups per CU
        const double G = std::min(f.waves * f.nb, nbr_max);
        const double per_item = c.item + f.nb * (c.item_nb + c.item_stream * pairs);
        const double cu_item = G * f.rows * (c.out + (gelu ? c.gelu : 0.0) + c.mfma * pairs);
        const double fixed = c.launch + c.result * result;
        // (beyond 16 items a workgroup the tail of the launch shows; a tuning value counts down to a whole number of
        // workgroups per panel)
        int first = 1, last = std::min(per_panel, 16);
        if (ipw_set > 0) {
            first = std::min(ipw_set, per_panel);
            while (per_panel % first)
                first--;
            last = first;
        }
        for (int d = first; d <= last; d++) {
            if (per_panel % d)
                continue;
            const long groups = per_panel / d, nwg = panels * groups;
            const long on_cu = (nwg + cus - 1) / cus, rounds = (on_cu + slots - 1) / slots;
            const double mb = tl_traffic_mb(x_mb, w_mb, panels, groups, 1.75);
            const bool by_group = tl_order(x_mb, w_mb, panels, groups, 1.75);
            const double us = fixed + c.traffic * mb + c.traffic_over * std::max(0.0, mb - 12.0) +
                              (double)rounds * (c.round + d * per_item) +
                              (double)on_cu * (c.panel * f.rows * K + d * cu_item) + c.wg * (double)nwg;
            if (!best.form || us < best.us)
                best = TlChoice{&f, d, ncg, by_group, lds, us};
        }
    }
    return best;
}

// Plans with K in several chunks: the kernel with the least estimated time (us).  Whole rows (tile_rows.hip) stream W
// once per 16 rows and have no chain of chunks: few rows.  The plan kernel fetches, waits and multiplies chunk by
// chunk, two workgroups of 8 nb block-rows per CU.  The kernel with fetching waves takes in the next chunk meanwhile, one
// workgroup of 12 nb block-rows per CU: where its workgroups just fit one round it is up to a third shorter (3300 rows
// 3072 -> 768, 80 %: 18.9 -> 13.4 us; 1536 rows, 50 %: 16.7 -> 14.1; 2300 rows 4096 -> 1024, 50 %: 48.8 -> 26.6).
// Terms: launch, rounds of workgroups and their chunks, the stream of a wave's pairs, the work of the busiest CU, and
// the megabytes that the L2s take in; fitted like the single-panel forms to 1600 launches (2048 -> 512, 3072 -> 768,
// 4096 -> 1024, 0 to 90 % pruned, 48 to 16384 rows): 5 to 6 % off in the mean, the choice 0.2 % behind the fastest
// kernel, 9 % at most (the rule before: 10.9 %).  The 576 launches that bench/linear_forms.py times in graphs (plan kernel,
// fetching waves, whole rows): 15, 8 and 13 % off.
enum { TL_BY_ROWS = -1, TL_BY_PLAN = 0, TL_BY_TALL = 5, TL_BY_TALL_SPLIT, TL_BY_TALL_2, TL_BY_TALL_3, TL_BY_LAST = TL_BY_TALL_3 }; // or 1 .. 4: fetching waves, that many block-rows per computing wave
static int tall_block_rows(int which) { // of a workgroup
    return which == TL_BY_TALL_SPLIT ? TL_CWAVES / 2 : TL_CWAVES * (which == TL_BY_TALL ? 1 : which - TL_BY_TALL);
}
static double estimate_plan_kernel(int M, double pairs, double x_mb, double w_mb, int nchunk, int nbr_max, int nlin, long cus) {
    const long panels = (M + TL_BM - 1) / TL_BM;
    const int nb = choose_nb((int)panels, nbr_max, nlin), ncg = (nbr_max + TL_WAVES * nb - 1) / (TL_WAVES * nb) * nlin;
    const long wgs = panels * ncg, rounds = (wgs + 2 * cus - 1) / (2 * cus), on_cu = (wgs + cus - 1) / cus;
    return 1.367 + rounds * (0.9615 * nchunk + 0.0867 * nb * pairs) +
           on_cu * (0.4349 * nchunk + 0.01745 * nb * pairs + 0.6037 * nb) + 0.0673 * tl_traffic_mb(x_mb, w_mb, panels, ncg, 1.75);
}
static double estimate_chunked(int M, double pairs, double x_mb, double w_mb, int nchunk, int nbr_max, int nlin, int nb, long cus) {
    const long panels = (M + TL_BM - 1) / TL_BM;
    const int ncg = (nbr_max + TL_CWAVES * nb - 1) / (TL_CWAVES * nb) * nlin;
    const long wgs = panels * ncg;
    const double rounds = (double)((wgs + cus - 1) / cus), fill = std::min(1.0, (double)wgs / cus);
    return 1.775 + rounds * (1.997 + (0.378 + 0.233 * nb) * nchunk + (0.0397 + 0.0140 * fill) * nb * pairs +
                             0.00429 * std::min(TL_CWAVES * nb, nbr_max) * pairs) +
           0.0980 * tl_traffic_mb(x_mb, w_mb, panels, ncg, 1.75);
}
// 48-row panels.  The fit (775 launches of 1536 -> 768, 2048 -> 512 and 1536, 3072 -> 768, 4096 -> 1024, 50 to 90 % pruned,
// 250 to 16384 rows: 2 to 5 % off) times 1.15: the figures above are 6 to 12 % high on the same launches, and with less the
// choice is up to 24 % behind what it was without these forms, with this 1.6 %.  It is 3.6 % faster in the mean over all of
// these launches, and 1 % behind the fastest kernel.
static double estimate_tall(int which, int M, double pairs, double x_mb, double w_mb, int nchunk, int nbr_max, int nlin, long cus) {
    const long panels = (M + 16 * TL_TALL - 1) / (16 * TL_TALL);
    const int brs = tall_block_rows(which), ncg = (nbr_max + brs - 1) / brs * nlin;
    const double nb = (double)brs / TL_CWAVES;
    const long wgs = panels * ncg;
    const double rounds = (double)((wgs + cus - 1) / cus), fill = std::min(1.0, (double)wgs / cus);
    const double traffic = tl_traffic_mb(x_mb, w_mb, panels, ncg, 1.75);
    if (which == TL_BY_TALL_SPLIT)
        return 1.15 * (1.468 + rounds * (2.068 + 1.277 * nchunk + 0.0512 * fill * nb * pairs + 0.00231 * std::min(brs, nbr_max) * pairs) +
                       0.0332 * traffic);
    return 1.15 * (1.094 + rounds * (2.931 + (0.4926 + 0.2443 * nb) * nchunk + (0.0840 + 0.0414 * fill) * nb * pairs) + 0.0736 * traffic);
}
static int weigh_chunked(const TlProblem *probs, int nlin, int M, int K, int nchunk, int nbr_max, long cus, double *us) {
    double pairs = 0.0, w_mb = 0.0;
    for (int i = 0; i < nlin; i++) {
        const double p = 0.5 * probs[i].ntile / probs[i].nbr;
        pairs += p / nlin;
        w_mb += p * probs[i].nbr * 1024e-6;
    }
    const double x_mb = 2e-6 * M * K;
    auto estimate = [&](int which) {
        return which == TL_BY_ROWS   ? tile_rows_estimate(M, K, nbr_max, nlin, pairs, w_mb)
               : which == TL_BY_PLAN ? estimate_plan_kernel(M, pairs, x_mb, w_mb, nchunk, nbr_max, nlin, cus)
               : which >= TL_BY_TALL ? estimate_tall(which, M, pairs, x_mb, w_mb, nchunk, nbr_max, nlin, cus)
                                     : estimate_chunked(M, pairs, x_mb, w_mb, nchunk, nbr_max, nlin, which, cus);
    };
    const bool rows_fit = tile_rows_fits(K);
    const int rows_most = g_tile_rows_most, chunked = g_tile_chunked;
    int best = TL_BY_PLAN;
    if (rows_fit && rows_most >= 0 && M <= rows_most)
        best = TL_BY_ROWS; // (tuning)
    else if (chunked > 0)
        best = std::min(chunked, (int)TL_BY_LAST);
    *us = estimate(best);
    if (best != TL_BY_PLAN)
        return best;
    auto take = [&](int which) {
        const double t = estimate(which);
        if (t < *us) {
            *us = t;
            best = which;
        }
    };
    if (chunked < 0)
        for (int which = 1; which <= TL_BY_LAST; which++)
            take(which);
    if (rows_fit && rows_most < 0)
        take(TL_BY_ROWS);
    return best;
}

// The two choices, kept for sizes that come again (100 rows 768 -> 768, bound by the host: 5.4 -> 4.9 us a call).
static std::atomic<int> g_tunings{0}; // et_tuning_set has returned so many times
typedef KeptChoices<TlChoice, 6 + 3 * TL_MAX_LIN> ResidentChoices;
struct ChunkedChoice {
    int which;
    double us;
};
typedef KeptChoices<ChunkedChoice, 6 + 3 * TL_MAX_LIN> ChunkedChoices;
template <class Key> static Key choice_key(const TlProblem *probs, int nlin, int M, int K, int more, int cus) {
    Key k = {{nlin, M, K, more, cus, g_tunings.load(std::memory_order_acquire)}};
    for (int i = 0; i < nlin; i++) {
        k.v[6 + 3 * i] = probs[i].N;
        k.v[7 + 3 * i] = probs[i].nbr;
        k.v[8 + 3 * i] = probs[i].ntile;
    }
    return k;
}
static TlChoice choose_resident(const TlProblem *probs, int nlin, int M, int K, int nbr_max, bool gelu) {
    static thread_local ResidentChoices kept;
    const int cus = std::max(et_device_cu_count(), 1);
    return kept.get(choice_key<ResidentChoices::Key>(probs, nlin, M, K, gelu, cus),
                    [&] { return weigh_resident(probs, nlin, M, K, nbr_max, gelu, cus); });
}
static int choose_chunked(const TlProblem *probs, int nlin, int M, int K, int nchunk, int nbr_max, double *us) {
    static thread_local ChunkedChoices kept;
    const int cus = std::max(et_device_cu_count(), 1);
    const ChunkedChoice c = kept.get(choice_key<ChunkedChoices::Key>(probs, nlin, M, K, nchunk, cus), [&] {
        ChunkedChoice v;
        v.which = weigh_chunked(probs, nlin, M, K, nchunk, nbr_max, cus, &v.us);
        return v;
    });
    *us = c.us;
    return c.which;
}

// the tile kernels' estimated time for planned linears over one input, launches of their own added up (join_launches)
static double tiles_estimate(const int *out_feat, const int *ntile, const int *nchunk, const int *launch, int launches, int n,
                             int M, int K, bool gelu) {
    double sum = 0.0;
    for (int l = 0; l < launches; l++) {
        TlProblem probs[TL_MAX_LIN];
        int m = 0, chunks = 0, nbr_max = 0;
        for (int i = 0; i < n; i++)
            if (launch[i] == l) {
                probs[m].N = out_feat[i];
                probs[m].nbr = out_feat[i] / 16;
                probs[m].ntile = ntile[i];
                chunks = nchunk[i];
                nbr_max = std::max(nbr_max, probs[m++].nbr);
            }
        double us;
        if (chunks > 1)
            (void)choose_chunked(probs, m, M, K, chunks, nbr_max, &us);
        else
            us = choose_resident(probs, m, M, K, nbr_max, gelu).us;
        sum += us;
    }
    return sum;
}

template <int NB, bool GELU, int NW = TL_WAVES>
static int launch_resident64(const TlArgs &a, size_t lds, hipStream_t st) {
    constexpr auto k = &tile_linear_resident_kernel<NB, GELU, NW, false, TL_BM64>;
    launch_kernel<k>(dim3(a.per_xcd * 8), dim3(NW * 64), lds, st, TL_HOT(a, N[0]), a);
    return launch_status("tile_linear (64-row panels) launch");
}

static int tile_launch_rows(const TlProblem *probs, int nlin, const f16 *X, int M, int K,
                            int KC, int nchunk, bool gelu, int mode, hipStream_t st) {
    TlArgs a;
    memset(&a, 0, sizeof(a));
    int nbr_max = 0;
    for (int i = 0; i < TL_MAX_LIN; i++) {
        const TlProblem &p = probs[i < nlin ? i : 0];
        a.Y[i] = p.Y;
        a.cptr[i] = p.cptr;
        a.row_offset[i] = p.row_offset;
        a.data[i] = p.data;
        a.bias[i] = p.bias;
        a.N[i] = p.N;
        if (i < nlin)
            nbr_max = std::max(nbr_max, p.nbr);
    }
    a.X = X;
    a.nlin = nlin;
    a.M = M;
    a.K = K;
    a.KC = KC;
    a.nchunk = nchunk;
    // Whole rows in LDS (tile_rows.hip).  Plans: see choose_chunked.  Raw lists: always where K is beyond the generic
    // kernel's panel (it filters every list once per chunk: three to eight times slower), else while there is no more
    // than one workgroup per CU (16 rows x 16 block-rows each).
    const int rows_most = g_tile_rows_most;
    int which = TL_BY_PLAN;
    if (mode == TL_PLAN && nchunk > 1) {
        double us;
        which = g_tile_nb == 0 ? choose_chunked(probs, nlin, M, K, nchunk, nbr_max, &us) : TL_BY_PLAN;
    } else if (mode == TL_PLAN && g_tile_splitk_k1 && tile_rows_fits(K) && M <= (rows_most < 0 ? 128 : rows_most)) {
        which = TL_BY_ROWS;
    } else if (g_tile_nb == 0 && tile_rows_fits(K) && (mode == TL_RAW || mode == TL_FILTER)) {
        const long panels = (M + 15) / 16;
        if (nchunk > 1 || panels * ((nbr_max + 15) / 16) <= std::max(et_device_cu_count(), 1))
            which = TL_BY_ROWS;
    }
    if (which == TL_BY_ROWS) {
        const bool raw = mode != TL_PLAN;
        double pairs = 0.0; // per block-row
        LfLinear l[TL_MAX_LIN];
        f16 *Ys[TL_MAX_LIN];
        for (int i = 0; i < nlin; i++) {
            // (a raw list's length is on the device: 80 % pruned is assumed.  That only decides the split; with the true
            // density the launch takes the same time within 2 % from 16 to 4096 rows and 0 to 90 %, but for dense lists
            // over 3072 columns at 200 rows, 11.6 against 8.7 us, and 2000 rows, 48.5 against 44.1)
            const double p = raw ? 0.1 * K / 16 : 0.5 * probs[i].ntile / probs[i].nbr;
            l[i] = LfLinear{probs[i].data, probs[i].cptr, probs[i].row_offset, probs[i].bias, probs[i].nbr,
                            raw ? 1 : nchunk, raw ? 0 : KC * 2, probs[i].npair};
            Ys[i] = probs[i].Y;
            pairs += p / nlin;
        }
        return tile_rows_launch(l, Ys, nlin, X, M, K, pairs, gelu, raw, st);
    }
    auto place = [&](int bm, int order) { // order: by_group, or -1 to be worked out; false: too many workgroups
        const int panels = (M + bm - 1) / bm, per_rp = a.ncg * nlin;
        while (per_rp % a.ipw)
            a.ipw--; // (a tuning value: the items of a workgroup are one panel's)
        a.nwg = panels * (per_rp / a.ipw);
        a.per_xcd = (a.nwg + 7) / 8;
        if (order < 0) {
            double w_bytes = 0.0;
            for (int i = 0; i < nlin; i++)
                w_bytes += mode == TL_DENSE ? 2.0 * probs[i].N * K : 512.0 * (probs[i].ntile ? probs[i].ntile : 0.2 * probs[i].nbr * K / 16);
            order = tl_order(2.0 * M * K, w_bytes, panels, per_rp / a.ipw, 1.75e6);
        }
        a.by_group = order;
        a.div = a.by_group ? panels : per_rp / a.ipw;
        a.div_magic = magic_of(a.div);
        a.ncg_magic = magic_of(a.ncg);
        return quotients_fit((int64_t)panels * (per_rp / a.ipw), a.div) && quotients_fit(per_rp, a.ncg);
    };
    int nb = 0, order = -1;
    if (mode == TL_PLAN && nchunk == 1) { // (on whole rows: returned above)
        const TlChoice c = choose_resident(probs, nlin, M, K, nbr_max, gelu);
        a.ncg = c.ncg;
        a.ipw = c.d;
        if (c.form->rows == TL_BM64) {
            if (!place(TL_BM64, c.by_group))
                return ROWS_TOO_MANY;
            if (c.form->waves == 12)
                return gelu ? launch_resident64<2, true, 12>(a, c.lds, st) : launch_resident64<2, false, 12>(a, c.lds, st);
            if (c.form->nb == 3)
                return gelu ? launch_resident64<3, true>(a, c.lds, st) : launch_resident64<3, false>(a, c.lds, st);
            if (c.form->nb == 2)
                return gelu ? launch_resident64<2, true>(a, c.lds, st) : launch_resident64<2, false>(a, c.lds, st);
            return gelu ? launch_resident64<1, true>(a, c.lds, st) : launch_resident64<1, false>(a, c.lds, st);
        }
        nb = c.form->nb;
        order = c.by_group;
    } else {
        const int nrp = (M + TL_BM - 1) / TL_BM;
        if (which >= TL_BY_TALL) {
            const int brs = tall_block_rows(which);
            a.ncg = (nbr_max + brs - 1) / brs;
            a.ipw = 1;
            if (!place(16 * TL_TALL, -1))
                return ROWS_TOO_MANY;
            switch (which) {
            case TL_BY_TALL: return gelu ? launch_tall<1, false, true>(a, st) : launch_tall<1, false, false>(a, st);
            case TL_BY_TALL_2: return gelu ? launch_tall<2, false, true>(a, st) : launch_tall<2, false, false>(a, st);
            case TL_BY_TALL_3: return gelu ? launch_tall<3, false, true>(a, st) : launch_tall<3, false, false>(a, st);
            default: return gelu ? launch_tall<1, true, true>(a, st) : launch_tall<1, true, false>(a, st);
            }
        }
        if (which > 0) {
            const int cnb = which;
            a.ncg = (nbr_max + TL_CWAVES * cnb - 1) / (TL_CWAVES * cnb);
            a.ipw = 1;
            if (!place(TL_BM, -1))
                return ROWS_TOO_MANY;
            const size_t lds = 2 * (size_t)TL_BM * (KC + ((KC & 31) ? 0 : TL_PAD)) * sizeof(f16) +
                               (size_t)TL_CWAVES * TL_BM * (16 * cnb + 8) * sizeof(f16);
            switch (cnb) {
            case 1: return gelu ? launch_chunked_inst<1, true>(a, lds, st) : launch_chunked_inst<1, false>(a, lds, st);
            case 2: return gelu ? launch_chunked_inst<2, true>(a, lds, st) : launch_chunked_inst<2, false>(a, lds, st);
            case 3: return gelu ? launch_chunked_inst<3, true>(a, lds, st) : launch_chunked_inst<3, false>(a, lds, st);
            default: return gelu ? launch_chunked_inst<4, true>(a, lds, st) : launch_chunked_inst<4, false>(a, lds, st);
            }
        }
        nb = choose_nb(nrp, nbr_max, nlin);
        a.ncg = (nbr_max + TL_WAVES * nb - 1) / (TL_WAVES * nb);
        a.ipw = 1;
    }
    if (!place(TL_BM, order))
        return ROWS_TOO_MANY;
    const size_t lds_x = (size_t)TL_BM * (KC + ((KC & 31) ? 0 : TL_PAD)) * sizeof(f16);
    const size_t lds_y = (size_t)TL_BM * (TL_WAVES * nb * 16 + TL_PAD) * sizeof(f16);
    // plan kernel: panel + one private staging tile per wave; generic kernel:
    // the output tile reuses the panel's storage
    const size_t lds = mode == TL_PLAN
                           ? lds_x + (size_t)TL_WAVES * TL_BM * (16 * nb + 8) * sizeof(f16)
                           : std::max(lds_x, lds_y);
    if (mode == TL_PLAN)
        return gelu ? launch_nb<true, TL_PLAN>(nb, a, lds, st) : launch_nb<false, TL_PLAN>(nb, a, lds, st);
    if (mode == TL_RAW)
        return gelu ? launch_nb<true, TL_RAW>(nb, a, lds, st) : launch_nb<false, TL_RAW>(nb, a, lds, st);
    if (mode == TL_FILTER)
        return gelu ? launch_nb<true, TL_FILTER>(nb, a, lds, st) : launch_nb<false, TL_FILTER>(nb, a, lds, st);
    return gelu ? launch_nb<true, TL_DENSE>(nb, a, lds, st) : launch_nb<false, TL_DENSE>(nb, a, lds, st);
}

static int tile_launch(const TlProblem *probs, int nlin, const f16 *X, int M, int K, int KC, int nchunk, bool gelu, int mode,
                       hipStream_t st) {
    int rc = tile_launch_rows(probs, nlin, X, M, K, KC, nchunk, gelu, mode, st);
    if (rc != ROWS_TOO_MANY)
        return rc;
    const int first = M / 2 / 64 * 64; // (rows are independent)
    ET_REQUIRE(first > 0, ET_ERR_UNSUPPORTED, "tile_linear: %d rows and so many outputs are too many workgroups", M);
    TlProblem rest[TL_MAX_LIN];
    for (int i = 0; i < nlin; i++) {
        rest[i] = probs[i];
        rest[i].Y += (size_t)first * probs[i].N;
    }
    rc = tile_launch(probs, nlin, X, first, K, KC, nchunk, gelu, mode, st);
    return rc != ET_OK ? rc : tile_launch(rest, nlin, X + (size_t)first * K, M - first, K, KC, nchunk, gelu, mode, st);
}

static void chunking(int K, int *KC, int *nchunk, int panel = TL_MAX_PANEL) {
    if (K <= panel) {
        *KC = K;
        *nchunk = 1;
    } else {
        *KC = TL_CHUNK;
        *nchunk = (K + TL_CHUNK - 1) / TL_CHUNK;
    }
}

// Columns of a plan's chunks.  A linear that narrows its input is a feed-forward block's second one: chunks of 768 hidden
// columns are what the fused kernel walks, so only linears that do not get a single panel beyond 992 columns.
static void plan_chunking(int in_feat, int out_feat, int *KC, int *nchunk) {
    chunking(in_feat, KC, nchunk, out_feat < in_feat ? TL_MAX_RAW_PANEL : TL_MAX_PANEL);
}
// Which launch each of n plans over one input goes into.  The kernels of this file walk all linears of a launch in the
// same column chunks, and from 993 to 1024 columns a plan's chunks depend on its width: plans of another geometry get a
// launch of their own.  Returns the number of launches.
static int join_launches(const int *KC, const int *nchunk, int n, int *launch) {
    int launches = 0;
    for (int i = 0; i < n; i++) {
        launch[i] = -1;
        for (int j = 0; j < i && launch[i] < 0; j++)
            if (KC[j] == KC[i] && nchunk[j] == nchunk[i])
                launch[i] = launch[j];
        if (launch[i] < 0)
            launch[i] = launches++;
    }
    return launches;
}

static int raw_tile_linear(void *Y, const void *X, const int *row_ptr, const int *row_offset,
                           const void *data, int M, int N, int K, const void *bias,
                           bool gelu, void *stream, const char *who) {
    ET_REQUIRE(Y && X && row_ptr && bias, ET_ERR_INVALID_ARG, "%s: null pointer", who);
    ET_REQUIRE(M >= 0 && N > 0 && K > 0, ET_ERR_INVALID_ARG, "%s: M=%d N=%d K=%d", who, M, N, K);
    ET_REQUIRE(N % 16 == 0 && K % 16 == 0, ET_ERR_UNSUPPORTED,
               "%s: N=%d and K=%d must be multiples of 16", who, N, K);
    ET_REQUIRE(aligned16(Y) && aligned16(X) && aligned16(bias) && aligned16(data),
               ET_ERR_ALIGNMENT, "%s: Y, X, W_data and bias must be 16-byte aligned", who);
    if (M == 0)
        return ET_OK;
    TlProblem p;
    p.Y = static_cast<f16 *>(Y);
    p.cptr = row_ptr;
    p.row_offset = row_offset;
    p.data = static_cast<const f16 *>(data);
    p.bias = static_cast<const f16 *>(bias);
    p.N = N;
    p.nbr = N / 16;
    int KC, nchunk;
    chunking(K, &KC, &nchunk, TL_MAX_RAW_PANEL);
    return tile_launch(&p, 1, static_cast<const f16 *>(X), M, K, KC, nchunk, gelu,
                       nchunk == 1 ? TL_RAW : TL_FILTER, static_cast<hipStream_t>(stream));
}

} // namespace et

static int g_tail_pair_min_wgs = 0; // et_tuning_set("tile_tail_pair_min_wgs"): 0 = three quarters of the CUs

static int set_knob(const char *key, int value) {
    if (key && !strcmp(key, "tile_splitk_rows")) {
        et::g_tile_rows_most = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_splitk_k1")) {
        et::g_tile_splitk_k1 = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_form")) {
        et::g_tile_form = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "dense_form")) {
        et::set_dense_form(value);
        return ET_OK;
    }
    if (key && !strcmp(key, "plan_dense")) {
        et::g_plan_dense = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "row_gemm_min_rows")) {
        et::g_row_gemm_min_rows = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_nb")) {
        et::g_tile_nb = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_ipw")) {
        et::g_tile_ipw = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_chunked")) {
        et::g_tile_chunked = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_order")) {
        et::g_tile_order = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_bm64")) {
        et::g_tile_bm64 = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_tail_pair_min_wgs")) {
        g_tail_pair_min_wgs = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_tail_pair")) {
        et::set_tail_pair(value);
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_wait_spin")) {
        et::set_tail_spin(value);
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_fuse_ffn")) {
        et::g_tile_fuse_ffn = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_ln_chunked")) {
        et::g_tile_ln_chunked = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_ln_min_panels")) {
        et::g_tile_min_panels = value > 0 ? value : 0;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_fuse_ln")) {
        et::g_tile_fuse_ln = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "tile_min_wgs")) {
        et::g_tile_min_wgs = value;
        return ET_OK;
    }
    if (key && !strcmp(key, "layer_flow_rows")) {
        et::set_flow_rows(value);
        return ET_OK;
    }
    if (key && !strcmp(key, "qkv_attention")) {
        et::set_qkv_attention(value);
        return ET_OK;
    }
    if (key && !strcmp(key, "row_layernorm")) {
        et::set_row_layernorm(value);
        return ET_OK;
    }
    if (key && !strcmp(key, "ln_rows")) {
        et::set_ln_rows(value);
        return ET_OK;
    }
    if (key && !strcmp(key, "attn_packed")) {
        et::set_attn_packed(value);
        return ET_OK;
    }
    if (key && !strcmp(key, "attn_vwin")) {
        et::set_attn_vwin(value);
        return ET_OK;
    }
    if (key && !strcmp(key, "attn_variant")) {
        et::set_attn_variant(value);
        return ET_OK;
    }
    et::set_error("et_tuning_set: unknown key");
    return ET_ERR_INVALID_ARG;
}
extern "C" int et_tuning_set(const char *key, int value) {
    const int rc = set_knob(key, value);
    // Kept choices are weighed again.  Counted behind the write: a choice kept under the new number has read the new value.
    et::g_tunings.fetch_add(1, std::memory_order_release);
    return rc;
}

extern "C" int et_tile_spmm_add_bias(void *Y, const void *X, const int *W_row_ptr,
                                     const int *W_row_offset, const void *W_data, int M,
                                     int N, int K, const void *bias, void *stream) {
    return et::raw_tile_linear(Y, X, W_row_ptr, W_row_offset, W_data, M, N, K, bias, false,
                               stream, "et_tile_spmm_add_bias");
}

extern "C" int et_tile_spmm_add_bias_gelu(void *Y, const void *X, const int *W_row_ptr,
                                          const int *W_row_offset, const void *W_data,
                                          int M, int N, int K, const void *bias,
                                          void *stream) {
    return et::raw_tile_linear(Y, X, W_row_ptr, W_row_offset, W_data, M, N, K, bias, true,
                               stream, "et_tile_spmm_add_bias_gelu");
}

namespace et {
// dense_gemm.hip
int dense_gemm_launch(void *const *Ys, const void *X, const void *const *Ws, const void *const *biases,
                      const int *Ns, int nlin, int M, int K, bool gelu, hipStream_t st);
double dense_gemm_estimate(const int *Ns, int nlin, int M, int K, bool gelu);
int dense_from_plan(f16 *W, const f16 *data, const int *cptr, int K, int KC, int nchunk, int nbr); // null stream

// Plans of fully populated matrices: the dense product where it is estimated to be the shorter launch, from some hundred
// rows on (many outputs) or some thousand (few).  The tile kernels stream W once per 32 or 64 rows and walk it tile by
// tile.  3.0 of the 3.5 us stand for the launch, which dense_gemm_estimate leaves out.  On 252 full plans (16 to 16384 rows,
// random weights, launches of a graph) the choice is then 0.1 % behind the faster side in the mean and 8 % at most, on the
// 80 of bench/linear_forms.py 0.1 to 0.2 % (four runs; 2 to 12 % at most), with 0.3 us less 0.3 to 0.4 %, with 0.3 more 1.1
// to 1.3 %.  Those launches find their operands in the caches; where input and result do not stay there the tile kernels, which read W more often, take
// longer than estimated: from 48 MB on they count a tenth more.  99 plans of 256 to 1024 inputs for which that tenth decides,
// or would with a lower line, by stream, how much longer than the product the tile kernels take on the same operands / on
// operands that change: 10 to 16 MB +1 / -4 %, 16 to 24 +2 / +1, 40 to 48 +4 / +4 (from -3 to +15), 48 to 64 +8 / +6, 64 to 110 +1
// / +14, 110 to 200 +6 / +12.
constexpr double DENSE_LAUNCH_US = 3.5, TILES_BEYOND_MB = 48.0, TILES_BEYOND = 1.1;
struct FullPlansTime {
    double tiles, dense; // us, with what the line adds
};
static FullPlansTime full_plans_time(const int *Ns, const int *ntile, const int *nchunk, const int *launch, int launches, int n,
                                     int M, int K, bool gelu) {
    double mb = K * 2e-6 * M;
    for (int i = 0; i < n; i++)
        mb += Ns[i] * 2e-6 * M;
    return {tiles_estimate(Ns, ntile, nchunk, launch, launches, n, M, K, gelu) * (mb > TILES_BEYOND_MB ? TILES_BEYOND : 1.0),
            DENSE_LAUNCH_US + dense_gemm_estimate(Ns, n, M, K, gelu)};
}
static bool plans_run_dense(const et_tile_plan *const *plans, int n, int M, bool gelu) {
    if (!g_plan_dense || n > 3)
        return false;
    int Ns[3], ntile[3], KC[3], nchunk[3], launch[3];
    for (int i = 0; i < n; i++) {
        if (!plans[i]->d_dense)
            return false;
        Ns[i] = plans[i]->out_feat;
        ntile[i] = plans[i]->ntile;
        KC[i] = plans[i]->KC;
        nchunk[i] = plans[i]->nchunk;
    }
    if (g_plan_dense == 2)
        return true;
    const int launches = join_launches(KC, nchunk, n, launch);
    const FullPlansTime t = full_plans_time(Ns, ntile, nchunk, launch, launches, n, M, plans[0]->in_feat, gelu);
    return t.dense < t.tiles;
}
static int run_plans_dense(const et_tile_plan *const *plans, void *const *Ys, int n, const void *X, int M, bool gelu,
                           hipStream_t st) {
    const void *Ws[3], *biases[3];
    int Ns[3];
    for (int i = 0; i < n; i++) {
        Ws[i] = plans[i]->d_dense;
        biases[i] = plans[i]->d_bias;
        Ns[i] = plans[i]->out_feat;
    }
    return dense_gemm_launch(Ys, X, Ws, biases, Ns, n, M, plans[0]->in_feat, gelu, st);
}
static int row_linear(void *out, const void *in, const void *weight, const void *bias, int M, int N,
                      int K, bool gelu, void *stream) {
    ET_REQUIRE(out && in && weight && bias, ET_ERR_INVALID_ARG, "et_row_spmm_add_bias: null pointer");
    ET_REQUIRE(M >= 0 && N > 0 && K > 0, ET_ERR_INVALID_ARG,
               "et_row_spmm_add_bias: M=%d N=%d K=%d", M, N, K);
    ET_REQUIRE(N % 16 == 0 && K % 16 == 0, ET_ERR_UNSUPPORTED,
               "et_row_spmm_add_bias: N=%d and K=%d must be multiples of 16", N, K);
    ET_REQUIRE(aligned16(out) && aligned16(in) && aligned16(weight) && aligned16(bias),
               ET_ERR_ALIGNMENT, "et_row_spmm_add_bias: pointers must be 16-byte aligned");
    if (M == 0)
        return ET_OK;
    if (g_row_gemm_min_rows > 0 && M >= g_row_gemm_min_rows) {
        const int rc = dense_gemm_launch(&out, in, &weight, &bias, &N, 1, M, K, gelu, static_cast<hipStream_t>(stream));
        if (rc != ET_ERR_UNSUPPORTED)
            return rc;
    }
    TlProblem p;
    p.Y = static_cast<f16 *>(out);
    p.cptr = nullptr;
    p.row_offset = nullptr;
    p.data = static_cast<const f16 *>(weight);
    p.bias = static_cast<const f16 *>(bias);
    p.N = N;
    p.nbr = N / 16;
    int KC, nchunk;
    chunking(K, &KC, &nchunk, TL_MAX_RAW_PANEL);
    return tile_launch(&p, 1, static_cast<const f16 *>(in), M, K, KC, nchunk, gelu, TL_DENSE,
                       static_cast<hipStream_t>(stream));
}
} // namespace et

extern "C" int et_row_spmm_prefers_gemm(int M, int N, int K) {
    return et::g_row_gemm_min_rows > 0 && M >= et::g_row_gemm_min_rows && N > 0 && N % 16 == 0 && K >= 32 &&
                   K % 32 == 0
               ? 1
               : 0;
}

extern "C" int et_row_spmm_add_bias_multi(void *const *outs, const void *in, const void *const *weights,
                                          const void *const *biases, const int *Ns, int n, int M, int K,
                                          void *stream) {
    using namespace et;
    ET_REQUIRE(outs && in && weights && biases && Ns, ET_ERR_INVALID_ARG, "et_row_spmm_add_bias_multi: null pointer");
    ET_REQUIRE(n >= 1 && n <= 3 && M >= 0 && K > 0, ET_ERR_INVALID_ARG, "et_row_spmm_add_bias_multi: n=%d M=%d K=%d",
               n, M, K);
    if (M == 0)
        return ET_OK;
    if (et_row_spmm_prefers_gemm(M, Ns[0], K)) {
        const int rc = dense_gemm_launch(outs, in, weights, biases, Ns, n, M, K, false, static_cast<hipStream_t>(stream));
        if (rc != ET_ERR_UNSUPPORTED)
            return rc;
    }
    for (int i = 0; i < n; i++) { // one after the other
        const int rc = row_linear(outs[i], in, weights[i], biases[i], M, Ns[i], K, false, stream);
        if (rc != ET_OK)
            return rc;
    }
    return ET_OK;
}

extern "C" int et_row_spmm_add_bias(void *out, const void *in, const void *weight,
                                    const void *bias, int M, int N, int K, void *stream) {
    return et::row_linear(out, in, weight, bias, M, N, K, false, stream);
}

extern "C" int et_row_spmm_add_bias_gelu(void *out, const void *in, const void *weight,
                                         const void *bias, int M, int N, int K, void *stream) {
    return et::row_linear(out, in, weight, bias, M, N, K, true, stream);
}

// ---------------------------------------------------------------------------
// plans
// ---------------------------------------------------------------------------
extern "C" int et_tile_plan_create(et_tile_plan **plan, int in_feat, int out_feat, int ntile,
                                   const void *data, const int *row_ptr,
                                   const int *row_offset, const void *bias) {
    using namespace et;
    ET_REQUIRE(plan && row_ptr && bias && (ntile == 0 || (data && row_offset)),
               ET_ERR_INVALID_ARG, "et_tile_plan_create: null pointer");
    *plan = nullptr;
    const int v = et_tile_mat_validate(out_feat, in_feat, ntile, row_ptr, row_offset);
    ET_REQUIRE(v == 0, ET_ERR_FORMAT, "et_tile_plan_create: malformed tile_mat (check %d)", v);
    const int nbr = out_feat / 16;
    int KC, nchunk;
    plan_chunking(in_feat, out_feat, &KC, &nchunk);
    // Plan layout: tiles ordered by (chunk, block-row, column); every
    // (chunk, block-row) segment padded to an even count with an all-zero
    // tile that reuses the segment's last column (so a pair never straddles
    // two block-rows and the kernel needs no odd-tail handling).
    std::vector<int> order(ntile);
    std::iota(order.begin(), order.end(), 0);
    for (int bn = 0; bn < nbr; bn++)
        std::stable_sort(order.begin() + row_ptr[bn], order.begin() + row_ptr[bn + 1],
                         [&](int x, int y) { return row_offset[x] < row_offset[y]; });
    std::vector<int> cptr((size_t)nbr * nchunk + 1, 0);
    for (int bn = 0; bn < nbr; bn++)
        for (int i = row_ptr[bn]; i < row_ptr[bn + 1]; i++)
            cptr[(size_t)(row_offset[i] / KC) * nbr + bn + 1]++;
    for (size_t i = 0; i < (size_t)nbr * nchunk; i++)
        cptr[i + 1] = cptr[i] + (cptr[i + 1] + 1) / 2 * 2;
    // spare all-zero pairs behind the last one: the kernels request the first
    // pairs of a wave's stream before they know whether it is empty, and a
    // stream's last stages request up to 2*TL_DEPTH pairs past its end
    const size_t total = (size_t)cptr.back() + 2 * (2 * TL_DEPTH + 1);
    const int bcols = in_feat / 16;
    bool full = ntile == nbr * bcols && in_feat % 32 == 0; // (the dense product walks K by 32)
    for (int i = 0; i < ntile && full; i++)
        full = row_offset[order[i]] == i % bcols * 16;
    // one device allocation and one transfer: data, column offsets, segment starts, bias (and a full matrix row-major)
    auto part = [](size_t bytes) { return (bytes + 255) / 256 * 256; };
    const size_t at_off = part(total * 512), at_cptr = at_off + part(total * 4), at_bias = at_cptr + part(cptr.size() * 4),
                 at_dense = at_bias + part((size_t)out_feat * 2);
    std::unique_ptr<unsigned char[]> image(new unsigned char[at_dense]); // (uninitialised: written once, below)
    int *const off = reinterpret_cast<int *>(image.get() + at_off);
    const uint16_t *src = static_cast<const uint16_t *>(data);
    auto zero_tiles = [&](size_t first, size_t n) { memset(image.get() + first * 512, 0, n * 512); };
    for (int bn = 0; bn < nbr; bn++) {
        int i = row_ptr[bn];
        for (int c = 0; c < nchunk; c++) { // (a block-row's tiles are in column order, hence by chunk)
            const size_t seg = (size_t)c * nbr + bn;
            int q = cptr[seg];
            for (; i < row_ptr[bn + 1] && row_offset[order[i]] / KC == c; i++, q++) {
                off[q] = (row_offset[order[i]] - c * KC) * 2;
                memcpy(image.get() + (size_t)q * 512, src + (size_t)order[i] * 256, 512);
            }
            if (q < cptr[seg + 1]) {
                off[q] = off[q - 1];
                zero_tiles(q, 1);
            }
        }
    }
    zero_tiles(cptr.back(), total - cptr.back());
    memset(off + cptr.back(), 0, (total - cptr.back()) * 4);
    memcpy(image.get() + at_cptr, cptr.data(), cptr.size() * 4);
    memcpy(image.get() + at_bias, bias, (size_t)out_feat * 2);

    et_tile_plan *p = new et_tile_plan();
    {
        static std::atomic<unsigned long long> next_uid{0}; // (plans are created from any thread)
        p->uid = ++next_uid;
    }
    // column-sorted host copy (the layer-tail program is built from it)
    p->h_row_ptr.assign(row_ptr, row_ptr + nbr + 1);
    p->h_col.resize(ntile);
    p->h_data.reserve((size_t)ntile * 256);
    for (int i = 0; i < ntile; i++) {
        p->h_col[i] = row_offset[order[i]];
        p->h_data.insert(p->h_data.end(), src + (size_t)order[i] * 256, src + (size_t)order[i] * 256 + 256);
    }
    p->in_feat = in_feat;
    p->out_feat = out_feat;
    p->ntile = ntile;
    p->KC = KC;
    p->nchunk = nchunk;
    p->npair = cptr.back() / 2;
    for (size_t i = 0; i + 1 < cptr.size(); i++)
        p->most_pairs = std::max(p->most_pairs, (cptr[i + 1] - cptr[i]) / 2);
    unsigned char *dev = nullptr;
    int rc = et_malloc((void **)&dev, at_dense + (full ? (size_t)out_feat * in_feat * 2 : 0));
    p->d_data = reinterpret_cast<f16 *>(dev);
    if (rc == ET_OK)
        rc = et_memcpy_h2d(dev, image.get(), at_dense);
    if (rc == ET_OK) {
        p->d_row_offset = reinterpret_cast<int *>(dev + at_off);
        p->d_cptr = reinterpret_cast<int *>(dev + at_cptr);
        p->d_bias = reinterpret_cast<f16 *>(dev + at_bias);
    }
    if (full && rc == ET_OK) {
        p->d_dense = reinterpret_cast<f16 *>(dev + at_dense);
        rc = dense_from_plan(p->d_dense, p->d_data, p->d_cptr, in_feat, KC, nchunk, nbr);
        if (rc == ET_OK && hipStreamSynchronize(nullptr) != hipSuccess) { // (the plan may run on any stream)
            set_error("et_tile_plan_create: the row-major copy failed");
            rc = ET_ERR_HIP;
        }
    }
    if (rc != ET_OK) {
        et_tile_plan_destroy(p);
        return rc;
    }
    *plan = p;
    return ET_OK;
}

extern "C" void et_tile_plan_destroy(et_tile_plan *p) {
    if (!p)
        return;
    et_free(p->d_data); // (all of the plan's device memory)
    et::tail_program_destroy(p->tail);
    delete p;
}

extern "C" int et_tile_plan_query(const et_tile_plan *p, int *in_feat, int *out_feat,
                                  int *ntile, int *nchunk, int *chunk_cols) {
    ET_REQUIRE(p, ET_ERR_INVALID_ARG, "et_tile_plan_query: null plan");
    if (in_feat) *in_feat = p->in_feat;
    if (out_feat) *out_feat = p->out_feat;
    if (ntile) *ntile = p->ntile;
    if (nchunk) *nchunk = p->nchunk;
    if (chunk_cols) *chunk_cols = p->KC;
    return ET_OK;
}

extern "C" int et_tile_plan_run_multi(const et_tile_plan *const *plans, void *const *Ys, int n,
                                      const void *X, int M, void *stream) {
    using namespace et;
    ET_REQUIRE(plans && Ys && X, ET_ERR_INVALID_ARG, "et_tile_plan_run_multi: null pointer");
    ET_REQUIRE(n >= 1 && n <= TL_MAX_LIN, ET_ERR_INVALID_ARG, "et_tile_plan_run_multi: n=%d", n);
    ET_REQUIRE(M >= 0, ET_ERR_INVALID_ARG, "et_tile_plan_run_multi: M=%d", M);
    TlProblem pr[TL_MAX_LIN];
    int KC[TL_MAX_LIN], nchunk[TL_MAX_LIN], launch[TL_MAX_LIN];
    for (int i = 0; i < n; i++) {
        ET_REQUIRE(plans[i] && Ys[i], ET_ERR_INVALID_ARG, "et_tile_plan_run_multi: null entry %d", i);
        ET_REQUIRE(plans[i]->in_feat == plans[0]->in_feat, ET_ERR_INVALID_ARG,
                   "et_tile_plan_run_multi: in_feat differs");
        ET_REQUIRE(aligned16(Ys[i]), ET_ERR_ALIGNMENT, "et_tile_plan_run_multi: Y not aligned");
        pr[i].Y = static_cast<f16 *>(Ys[i]);
        pr[i].cptr = plans[i]->d_cptr;
        pr[i].row_offset = plans[i]->d_row_offset;
        pr[i].data = plans[i]->d_data;
        pr[i].bias = plans[i]->d_bias;
        pr[i].N = plans[i]->out_feat;
        pr[i].nbr = plans[i]->out_feat / 16;
        pr[i].ntile = plans[i]->ntile;
        pr[i].npair = plans[i]->npair;
        KC[i] = plans[i]->KC;
        nchunk[i] = plans[i]->nchunk;
    }
    ET_REQUIRE(aligned16(X), ET_ERR_ALIGNMENT, "et_tile_plan_run_multi: X not aligned");
    if (M == 0)
        return ET_OK;
    if (plans_run_dense(plans, n, M, false))
        return run_plans_dense(plans, Ys, n, X, M, false, static_cast<hipStream_t>(stream));
    const int launches = join_launches(KC, nchunk, n, launch);
    for (int l = 0; l < launches; l++) {
        TlProblem joined[TL_MAX_LIN];
        int m = 0, last = 0;
        for (int i = 0; i < n; i++)
            if (launch[i] == l) {
                joined[m++] = pr[i];
                last = i;
            }
        const int rc = tile_launch(joined, m, static_cast<const f16 *>(X), M, plans[0]->in_feat, KC[last], nchunk[last],
                                   false, TL_PLAN, static_cast<hipStream_t>(stream));
        if (rc != ET_OK)
            return rc;
    }
    return ET_OK;
}

extern "C" int et_tile_plan_estimate(int in_feat, const int *out_feat, const int *ntile, int n, int M, int gelu,
                                     double *tiles_us, double *dense_us) {
    using namespace et;
    ET_REQUIRE(out_feat && ntile && tiles_us && dense_us, ET_ERR_INVALID_ARG, "et_tile_plan_estimate: null pointer");
    ET_REQUIRE(in_feat > 0 && in_feat % 16 == 0 && M > 0 && n >= 1 && n <= TL_MAX_LIN, ET_ERR_INVALID_ARG,
               "et_tile_plan_estimate: in_feat=%d M=%d n=%d", in_feat, M, n);
    int KC[TL_MAX_LIN], nchunk[TL_MAX_LIN], launch[TL_MAX_LIN];
    for (int i = 0; i < n; i++) {
        ET_REQUIRE(out_feat[i] > 0 && out_feat[i] % 16 == 0 && ntile[i] >= 0, ET_ERR_INVALID_ARG,
                   "et_tile_plan_estimate: out_feat=%d ntile=%d", out_feat[i], ntile[i]);
        plan_chunking(in_feat, out_feat[i], &KC[i], &nchunk[i]);
    }
    const int launches = join_launches(KC, nchunk, n, launch);
    *tiles_us = tiles_estimate(out_feat, ntile, nchunk, launch, launches, n, M, in_feat, gelu != 0);
    *dense_us = dense_gemm_estimate(out_feat, n, M, in_feat, gelu != 0);
    return ET_OK;
}

extern "C" int et_tile_plan_prefers_dense(int in_feat, const int *out_feat, int n, int M, int gelu) {
    using namespace et;
    if (!g_plan_dense || !out_feat || n < 1 || n > 3 || M <= 0 || in_feat <= 0 || in_feat % 32 != 0)
        return 0;
    int ntile[3], KC[3], nchunk[3], launch[3];
    for (int i = 0; i < n; i++) {
        if (out_feat[i] <= 0 || out_feat[i] % 16 != 0)
            return 0;
        ntile[i] = (in_feat / 16) * (out_feat[i] / 16);
        plan_chunking(in_feat, out_feat[i], &KC[i], &nchunk[i]);
    }
    if (g_plan_dense == 2)
        return 1;
    const int launches = join_launches(KC, nchunk, n, launch);
    const FullPlansTime t = full_plans_time(out_feat, ntile, nchunk, launch, launches, n, M, in_feat, gelu != 0);
    return t.dense < t.tiles;
}

extern "C" int et_tile_plan_launches(int in_feat, const int *out_feat, int n, int *launch, int *nchunk, int *chunk_cols) {
    using namespace et;
    ET_REQUIRE(out_feat && launch && nchunk && chunk_cols, ET_ERR_INVALID_ARG, "et_tile_plan_launches: null pointer");
    ET_REQUIRE(in_feat > 0 && n >= 1 && n <= TL_MAX_LIN, ET_ERR_INVALID_ARG, "et_tile_plan_launches: in_feat=%d n=%d",
               in_feat, n);
    for (int i = 0; i < n; i++)
        plan_chunking(in_feat, out_feat[i], &chunk_cols[i], &nchunk[i]);
    join_launches(chunk_cols, nchunk, n, launch);
    return ET_OK;
}

extern "C" int et_tile_plan_ln_fusable(const et_tile_plan *plan) {
    return plan && et::ln_block_rows(plan->out_feat / 16) != 0 && plan->out_feat % 8 == 0 &&
                   et::g_tile_fuse_ln != 0
               ? 1
               : 0;
}

// The fused kernels run one workgroup per 32-row panel and CU, in rounds; with few panels, or few in a second round, most
// CUs idle and the separate launches (more, smaller workgroups) win.  Whole layers 1024 wide, fused / separate, us:
// 50 %: 4096 rows 144 / 124, 5120 173 / 170, 6144 185 / 199, 10240 360 / 319, 12288 392 / 372; 80 %: 4096 100 / 92,
// 6144 129 / 141, 10240 235 / 226, 12288 264 / 262, 16384 327 / 345.
static bool ln_fusion_pays(int M) {
    const int panels = (M + et::TL_BM - 1) / et::TL_BM, cus = std::max(et_device_cu_count(), 1);
    if (et::g_tile_min_panels)
        return panels >= et::g_tile_min_panels;
    const int rounds = (panels + cus - 1) / cus;
    return panels >= (rounds == 1 ? 0.6 : 0.76) * cus * rounds;
}
// Fewest panels for which the layer tail runs as one launch: its round takes the time of streaming the three linears
// past a panel, whatever the number of panels.  Whole layers, one launch / steps, us: 768 wide 50 %: 3072 rows 92 / 78,
// 4096 93 / 85, 5120 98 / 107; 80 %: 2560 rows 59 / 56, 3072 64 / 62, 3584 64 / 65; 90 %: 2560 52 / 52, 3072 56 / 57;
// 512 wide, 50 %: 3072 57 / 55, 3584 57 / 58.
// The same line decides for the panels of a last round behind full ones (et_tile_plan_run_tail), where the steps' launches
// come on top of the fused one.  Tail behind 256 full panels, last round fused / by steps, us: 768 wide 50 % (line 144): 80
// panels 150 / 127, 128 143 / 141, 144 145 / 155; 80 % (99): 52 87 / 79, 80 87 / 85, 96 87 / 88, 112 87 / 92; 90 % (84): 64
// 73 / 70, 80 73 / 74, 96 73 / 77; 512 wide 50 % (103): 96 79 / 78, 112 79 / 80; 80 % (83): 52 54 / 54, 80 54 / 58 - the
// furthest that it is off.  Behind 512 full panels the same.
static int tail_min_panels(const et_tile_plan *pO, const et_tile_plan *p1, const et_tile_plan *p2) {
    if (et::g_tile_min_panels)
        return et::g_tile_min_panels;
    return 70 + (int)(14.0 * 512e-6 * ((double)pO->ntile + p1->ntile + p2->ntile));
}

extern "C" int et_tile_plan_run_ln(const et_tile_plan *plan, void *Y, const void *X,
                                   const void *skip, const void *gamma, const void *beta, int M,
                                   void *stream) {
    using namespace et;
    ET_REQUIRE(plan && Y && X && skip && gamma && beta, ET_ERR_INVALID_ARG,
               "et_tile_plan_run_ln: null pointer");
    ET_REQUIRE(M >= 0, ET_ERR_INVALID_ARG, "et_tile_plan_run_ln: M=%d", M);
    ET_REQUIRE(aligned16(Y) && aligned16(X) && aligned16(skip) && aligned16(gamma) && aligned16(beta),
               ET_ERR_ALIGNMENT, "et_tile_plan_run_ln: pointers must be 16-byte aligned");
    if (M == 0)
        return ET_OK;
    const int nbr = plan->out_feat / 16;
    if (!et_tile_plan_ln_fusable(plan) || ((!ln_fusion_pays(M) || plans_run_dense(&plan, 1, M, false)) && Y != skip)) {
        // rows too wide for one workgroup, too few of them, or a dense product: the two kernels, one after the other
        ET_REQUIRE(Y != skip, ET_ERR_INVALID_ARG,
                   "et_tile_plan_run_ln: Y must not alias skip for out_feat=%d", plan->out_feat);
        const int rc = et_tile_plan_run(plan, Y, X, M, 0, stream);
        if (rc != ET_OK)
            return rc;
        return et_skip_layernorm(Y, skip, gamma, beta, M, plan->out_feat, stream);
    }
    TlProblem pr;
    pr.Y = static_cast<f16 *>(Y);
    pr.cptr = plan->d_cptr;
    pr.row_offset = plan->d_row_offset;
    pr.data = plan->d_data;
    pr.bias = plan->d_bias;
    pr.N = plan->out_feat;
    pr.nbr = nbr;
    return tile_launch_ln(pr, static_cast<const f16 *>(X), M, plan->in_feat, plan->KC, plan->nchunk,
                          static_cast<const f16 *>(skip), static_cast<const f16 *>(gamma),
                          static_cast<const f16 *>(beta), static_cast<hipStream_t>(stream));
}

extern "C" int et_tile_plan_ffn_fusable(const et_tile_plan *p1, const et_tile_plan *p2) {
    using namespace et;
    if (!p1 || !p2 || !g_tile_fuse_ffn)
        return 0;
    return p1->nchunk == 1 && p2->in_feat == p1->out_feat && p2->nchunk <= TL_FFN_MAX_PHASES &&
                   p2->KC / 16 <= TL_FFN_WAVES * 3 &&
                   p2->out_feat / 16 <= TL_FFN_WAVES * 3 && p2->out_feat % 8 == 0 &&
                   ffn_lds_bytes(p1->in_feat, p2->KC) <= 160 * 1024
               ? 1
               : 0;
}

// Full feed-forward plans: whether the steps of the block (pO: of the whole tail), one after the other, take less than the
// fused kernel, whose round streams all of W past its panels; a last round costs as much as a full one, unless the tail's
// rest runs by steps (et_tile_plan_run_tail).
// A fused round of the tail takes 14 us and 10.7 per MB of W, and inside a layer a tenth more: 256 wide 26, 384 38 to 42, 512
// 58 to 65, 640 90 to 100, 768 117 to 130.  Tail fused / by steps, us: 8192 rows 256 wide 27.9 / 33.7, 384 41.8 / 46.9, 512 65.3 / 63.7
// (the layer 105.6 / 99.9), 768 130 / 110; 16384 rows 512 wide 131 / 110, 768 258 / 200.
// Of the block alone: 9.4 us, 10.5 per MB and 2.9 for each further chunk of hidden columns, where the steps' estimates are
// 7 % high.  Fused / by steps, us: 128 -> 512 7200 rows 12.4 / 15.2, 12700 rows (the second round) 23.2 / 17.7; 256 -> 512 8192 14.7 /
// 16.2, 256 -> 1024 23.6 / 21.5, 384 -> 768 21.5 / 23.2, 12700 rows 38.3 / 31.9, 384 -> 1536 8192 rows 36.9 / 33.6, 640 -> 1280 49.3 / 43.7; from
// 512 wide on the steps.  Over these widths and 5000 to 16384 rows every choice is the faster one.
static bool ffn_runs_dense(const et_tile_plan *pO, const et_tile_plan *p1, const et_tile_plan *p2, int M) {
    using namespace et;
    if (!g_plan_dense || !p1->d_dense || !p2->d_dense)
        return false;
    if (g_plan_dense == 2)
        return true;
    auto linear = [](const et_tile_plan *p, int rows, bool gelu) {
        const int launch = 0;
        const FullPlansTime t = full_plans_time(&p->out_feat, &p->ntile, &p->nchunk, &launch, 1, 1, rows, p->in_feat, gelu);
        return p->d_dense ? std::min(t.tiles, t.dense) : t.tiles;
    };
    auto steps = [&](int rows) { // (a LayerNorm: 5.5 TB/s behind its launch)
        const double ln = 3.0 + 1.1e-6 * rows * p2->out_feat;
        return linear(p1, rows, true) + linear(p2, rows, false) + ln + (pO ? linear(pO, rows, false) + ln : 0.0);
    };
    const int cus = std::max(et_device_cu_count(), 1), panels = (M + TL_BM - 1) / TL_BM, full = panels / cus, rest = panels - full * cus;
    const double w_mb = 512e-6 * ((double)p1->ntile + p2->ntile + (pO ? pO->ntile : 0));
    const double round = pO ? 15.5 + 11.7 * w_mb : (9.4 + 10.5 * w_mb + 2.9 * (p2->nchunk - 1)) * 1.07;
    double fused = round * full;
    if (rest > 0)
        fused += pO && full > 0 && rest < tail_min_panels(pO, p1, p2) ? steps(M - full * cus * TL_BM) : round;
    return steps(M) < fused;
}

extern "C" int et_tile_plan_run_ffn_ln(const et_tile_plan *p1, const et_tile_plan *p2, void *Y,
                                       const void *X, void *hidden, const void *skip,
                                       const void *gamma, const void *beta, int M, void *stream) {
    using namespace et;
    ET_REQUIRE(p1 && p2 && Y && X && skip && gamma && beta, ET_ERR_INVALID_ARG,
               "et_tile_plan_run_ffn_ln: null pointer");
    ET_REQUIRE(M >= 0, ET_ERR_INVALID_ARG, "et_tile_plan_run_ffn_ln: M=%d", M);
    ET_REQUIRE(p2->in_feat == p1->out_feat, ET_ERR_INVALID_ARG,
               "et_tile_plan_run_ffn_ln: the second linear takes %d inputs, the first gives %d",
               p2->in_feat, p1->out_feat);
    ET_REQUIRE(aligned16(Y) && aligned16(X) && aligned16(skip) && aligned16(gamma) && aligned16(beta) &&
                   aligned16(hidden),
               ET_ERR_ALIGNMENT, "et_tile_plan_run_ffn_ln: pointers must be 16-byte aligned");
    if (M == 0)
        return ET_OK;
    const bool fusable = et_tile_plan_ffn_fusable(p1, p2) != 0;
    if (!fusable || (hidden && (!ln_fusion_pays(M) || ffn_runs_dense(nullptr, p1, p2, M)))) {
        // the three steps one after the other, through the caller's buffer
        ET_REQUIRE(hidden, ET_ERR_UNSUPPORTED,
                   "et_tile_plan_run_ffn_ln: these shapes need the hidden buffer (%d x %d halves)", M,
                   p1->out_feat);
        const int rc = et_tile_plan_run(p1, hidden, X, M, 1, stream);
        if (rc != ET_OK)
            return rc;
        return et_tile_plan_run_ln(p2, Y, hidden, skip, gamma, beta, M, stream);
    }
    TlProblem a, b;
    a.Y = nullptr;
    a.cptr = p1->d_cptr;
    a.row_offset = p1->d_row_offset;
    a.data = p1->d_data;
    a.bias = p1->d_bias;
    a.N = p1->out_feat;
    a.nbr = p1->out_feat / 16;
    b.Y = static_cast<f16 *>(Y);
    b.cptr = p2->d_cptr;
    b.row_offset = p2->d_row_offset;
    b.data = p2->d_data;
    b.bias = p2->d_bias;
    b.N = p2->out_feat;
    b.nbr = p2->out_feat / 16;
    return tile_launch_ffn(nullptr, a, b, static_cast<const f16 *>(X), M, p1->in_feat, p2->KC, p2->nchunk,
                           static_cast<const f16 *>(skip), static_cast<const f16 *>(gamma),
                           static_cast<const f16 *>(beta), nullptr, nullptr,
                           static_cast<hipStream_t>(stream));
}

extern "C" int et_tile_plan_tail_fusable(const et_tile_plan *pO, const et_tile_plan *p1,
                                         const et_tile_plan *p2) {
    return pO && et_tile_plan_ffn_fusable(p1, p2) && pO->nchunk == 1 && pO->in_feat == pO->out_feat &&
                   pO->out_feat == p1->in_feat && p2->out_feat == p1->in_feat &&
                   pO->out_feat / 16 <= et::TL_FFN_WAVES * 3 && et::g_tile_fuse_ffn >= 2
               ? 1
               : 0;
}

extern "C" int et_tile_plan_run_tail(const et_tile_plan *pO, const et_tile_plan *p1,
                                     const et_tile_plan *p2, void *Y, const void *attn, const void *input,
                                     void *mid, void *hidden, const void *gamma1, const void *beta1,
                                     const void *gamma2, const void *beta2, int M, void *stream) {
    using namespace et;
    ET_REQUIRE(pO && p1 && p2 && Y && attn && input && gamma1 && beta1 && gamma2 && beta2,
               ET_ERR_INVALID_ARG, "et_tile_plan_run_tail: null pointer");
    ET_REQUIRE(M >= 0, ET_ERR_INVALID_ARG, "et_tile_plan_run_tail: M=%d", M);
    ET_REQUIRE(pO->out_feat == p1->in_feat && p2->in_feat == p1->out_feat && p2->out_feat == p1->in_feat,
               ET_ERR_INVALID_ARG, "et_tile_plan_run_tail: the three linears do not chain (%d->%d, %d->%d, %d->%d)",
               pO->in_feat, pO->out_feat, p1->in_feat, p1->out_feat, p2->in_feat, p2->out_feat);
    ET_REQUIRE(aligned16(Y) && aligned16(attn) && aligned16(input) && aligned16(mid) && aligned16(hidden) &&
                   aligned16(gamma1) && aligned16(beta1) && aligned16(gamma2) && aligned16(beta2),
               ET_ERR_ALIGNMENT, "et_tile_plan_run_tail: pointers must be 16-byte aligned");
    if (M == 0)
        return ET_OK;
    if (!et_tile_plan_tail_fusable(pO, p1, p2) || (mid && ((M + TL_BM - 1) / TL_BM < tail_min_panels(pO, p1, p2) || ffn_runs_dense(pO, p1, p2, M)))) {
        // step by step through the caller's buffers
        ET_REQUIRE(mid, ET_ERR_UNSUPPORTED,
                   "et_tile_plan_run_tail: these shapes need the mid buffer (%d x %d halves)", M, pO->out_feat);
        const int rc = et_tile_plan_run_ln(pO, mid, attn, input, gamma1, beta1, M, stream);
        if (rc != ET_OK)
            return rc;
        return et_tile_plan_run_ffn_ln(p1, p2, Y, mid, hidden, mid, gamma2, beta2, M, stream);
    }
    // The fused kernel runs one workgroup per CU and 32-row panel, in rounds of
    // as many panels as there are CUs.  A last round that would leave most CUs
    // idle costs as much as a full one: with the caller's buffers at hand those
    // rows run step by step instead (after the fused launch on the same stream;
    // rows are independent).
    if (mid && hidden) {
        const int cus = std::max(et_device_cu_count(), 1);
        const int panels = (M + TL_BM - 1) / TL_BM, full = panels / cus * cus, rem = panels - full;
        if (full > 0 && rem > 0 && rem < tail_min_panels(pO, p1, p2)) {
            const int M1 = full * TL_BM;
            int rc = et_tile_plan_run_tail(pO, p1, p2, Y, attn, input, nullptr, nullptr, gamma1, beta1, gamma2,
                                           beta2, M1, stream);
            if (rc != ET_OK)
                return rc;
            const size_t off = (size_t)M1 * pO->out_feat; // all of Y, attn, input, mid are [rows x model width]
            f16 *midr = static_cast<f16 *>(mid) + off;
            rc = et_tile_plan_run_ln(pO, midr, static_cast<const f16 *>(attn) + off,
                                     static_cast<const f16 *>(input) + off, gamma1, beta1, M - M1, stream);
            if (rc != ET_OK)
                return rc;
            return et_tile_plan_run_ffn_ln(p1, p2, static_cast<f16 *>(Y) + off, midr, hidden, midr, gamma2, beta2,
                                           M - M1, stream);
        }
    }
    TlProblem o, a, b;
    o.Y = nullptr;
    o.cptr = pO->d_cptr;
    o.row_offset = pO->d_row_offset;
    o.data = pO->d_data;
    o.bias = pO->d_bias;
    o.N = pO->out_feat;
    o.nbr = pO->out_feat / 16;
    a.Y = nullptr;
    a.cptr = p1->d_cptr;
    a.row_offset = p1->d_row_offset;
    a.data = p1->d_data;
    a.bias = p1->d_bias;
    a.N = p1->out_feat;
    a.nbr = p1->out_feat / 16;
    b.Y = static_cast<f16 *>(Y);
    b.cptr = p2->d_cptr;
    b.row_offset = p2->d_row_offset;
    b.data = p2->d_data;
    b.bias = p2->d_bias;
    b.N = p2->out_feat;
    b.nbr = p2->out_feat / 16;
    return tile_launch_ffn(&o, a, b, static_cast<const f16 *>(attn), M, p1->in_feat, p2->KC, p2->nchunk,
                           static_cast<const f16 *>(input), static_cast<const f16 *>(gamma1),
                           static_cast<const f16 *>(beta1), static_cast<const f16 *>(gamma2),
                           static_cast<const f16 *>(beta2), static_cast<hipStream_t>(stream));
}

extern "C" int et_tile_plan_run(const et_tile_plan *plan, void *Y, const void *X, int M, int gelu,
                                void *stream) {
    using namespace et;
    ET_REQUIRE(plan && Y && X, ET_ERR_INVALID_ARG, "et_tile_plan_run: null pointer");
    ET_REQUIRE(M >= 0, ET_ERR_INVALID_ARG, "et_tile_plan_run: M=%d", M);
    ET_REQUIRE(aligned16(Y) && aligned16(X), ET_ERR_ALIGNMENT, "et_tile_plan_run: Y/X not aligned");
    if (M == 0)
        return ET_OK;
    if (plans_run_dense(&plan, 1, M, gelu != 0))
        return run_plans_dense(&plan, &Y, 1, X, M, gelu != 0, static_cast<hipStream_t>(stream));
    TlProblem pr;
    pr.Y = static_cast<f16 *>(Y);
    pr.cptr = plan->d_cptr;
    pr.row_offset = plan->d_row_offset;
    pr.data = plan->d_data;
    pr.bias = plan->d_bias;
    pr.N = plan->out_feat;
    pr.nbr = plan->out_feat / 16;
    pr.ntile = plan->ntile;
    pr.npair = plan->npair;
    return tile_launch(&pr, 1, static_cast<const f16 *>(X), M, plan->in_feat, plan->KC,
                       plan->nchunk, gelu != 0, TL_PLAN, static_cast<hipStream_t>(stream));
}

// ---------------------------------------------------------------------------
// layer tail with caller-provided scratch: pairs of workgroups over 64-row
// panels (tile_tail.hip) where that applies and pays
// ---------------------------------------------------------------------------
extern "C" size_t et_tile_plan_tail_ws_bytes(const et_tile_plan *pO, const et_tile_plan *p1,
                                             const et_tile_plan *p2, int M) {
    return et::tail_pair_ws_bytes(pO, p1, p2, M);
}

extern "C" size_t et_tail_ws_bytes_for(int d_model, int rows) {
    // (nothing while the paired form is switched off: an encoder's workspace is then the reference's)
    return et::tail_pair_enabled() ? et::tail_ws_bytes_for(d_model, rows) : 0;
}

extern "C" int et_tile_plan_tail_prepare(const et_tile_plan *pO, const et_tile_plan *p1,
                                         const et_tile_plan *p2) {
    using namespace et;
    ET_REQUIRE(pO && p1 && p2, ET_ERR_INVALID_ARG, "et_tile_plan_tail_prepare: null plan");
    (void)wait_status_device(); // (allocated here rather than inside a run)
    if (!tail_pair_applies(pO, p1, p2))
        return ET_OK; // nothing to prepare: et_tile_plan_run_tail_ws will run the other kernels
    return tail_pair_prepare(pO, p1, const_cast<et_tile_plan *>(p2));
}

extern "C" int et_tile_plan_run_tail_ws(const et_tile_plan *pO, const et_tile_plan *p1,
                                        const et_tile_plan *p2, void *Y, const void *attn, const void *input,
                                        void *mid, void *hidden, const void *gamma1, const void *beta1,
                                        const void *gamma2, const void *beta2, int M, void *ws, size_t ws_bytes,
                                        void *stream) {
    using namespace et;
    ET_REQUIRE(pO && p1 && p2 && Y && attn && input && gamma1 && beta1 && gamma2 && beta2,
               ET_ERR_INVALID_ARG, "et_tile_plan_run_tail_ws: null pointer");
    if (ws && M > 0 && tail_pair_applies(pO, p1, p2) && !(mid && hidden && ffn_runs_dense(pO, p1, p2, M))) {
        const size_t need = tail_pair_ws_bytes(pO, p1, p2, M);
        const int cus = std::max(et_device_cu_count(), 1);
        const int wgs = 2 * ((M + 63) / 64);
        const int min_wgs = g_tail_pair_min_wgs > 0 ? g_tail_pair_min_wgs : (3 * cus) / 4;
        if (ws_bytes >= need && (wgs >= min_wgs || !mid || tail_pair_forced())) {
            ET_REQUIRE(aligned16(Y) && aligned16(attn) && aligned16(input) && aligned16(gamma1) &&
                           aligned16(beta1) && aligned16(gamma2) && aligned16(beta2) && aligned16(ws),
                       ET_ERR_ALIGNMENT, "et_tile_plan_run_tail_ws: pointers must be 16-byte aligned");
            const int rc = tail_pair_prepare(pO, p1, const_cast<et_tile_plan *>(p2)); // (returns at once when prepared)
            if (rc != ET_OK)
                return rc;
            return tail_pair_launch(pO, p1, p2, static_cast<f16 *>(Y), static_cast<const f16 *>(attn),
                                    static_cast<const f16 *>(input), static_cast<const f16 *>(gamma1),
                                    static_cast<const f16 *>(beta1), static_cast<const f16 *>(gamma2),
                                    static_cast<const f16 *>(beta2), M, ws, static_cast<hipStream_t>(stream));
        }
    }
    return et_tile_plan_run_tail(pO, p1, p2, Y, attn, input, mid, hidden, gamma1, beta1, gamma2, beta2, M, stream);
}

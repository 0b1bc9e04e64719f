// Dense GEMM on gfx950:  Y[M x N] = X[M x K] W^T + b (+ GELU), W [N x K] row-major, fp16 storage, fp32 accumulate: the
// row-pruned linear on its compacted rows (in place of the cublasGemmEx call plus add_bias kernel of
// kernels/linear.cu:5-34) and the plans of fully populated tile matrices from some hundred rows on.
//
// Both operands are contiguous along K, which is the layout the 16x16x32 MFMA wants for A and for B (8 consecutive k
// per lane), so neither is transposed.  The product is issued as W X^T so that a lane ends with four consecutive output
// features of one row.  K is walked in steps of 64 through two to twelve LDS stages filled by DMA
// (global_load_lds_dwordx4, no registers).  A DMA instruction writes 64 x 16 bytes to consecutive LDS, the source
// address is free per lane: the 16-byte pieces of a row are stored XOR-swizzled by (row / 2) % 8, which puts the sixteen
// rows of a fragment read into sixteen different slots of 256 bytes without padding.
//
// What bounds it: in the middle of a large K the way of the operands into LDS and registers - a launch of 8192 x 8192 x 8192
// whose loop fetches nothing takes three quarters of the time, one that reads no fragments either two thirds, which is the
// matrix unit at the clock it gets (1.9 PFLOP/s); at K = 768 the ends: the launch, the first step's latency and the result's
// way out are 6 of 20 us.  A wave issues in order, and a memory instruction holds it until it is out, with both waves of a
// SIMD at the same place: so nothing goes out in one go, requests and LDS reads stand between the products.  Two stages of 64
// columns are requested half a step to a step before they are needed, which is a round trip to memory under load: where the
// LDS has room for more stages, and every CU has one block, they are taken.  (Stages of 32 columns, four to eight of them,
// are slower: a row's 64 bytes are half a cache line, which is fetched twice.)  All figures here are of normally
// distributed operands: with weights that are all alike the same launches are up to a sixth shorter.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "tile_plan.h"

namespace et {

constexpr int DG_BK = 64; // columns per step
constexpr int DG_MAX_LIN = 3;

struct DgArgs {
    f16 *Y[DG_MAX_LIN];
    const f16 *W[DG_MAX_LIN];
    const f16 *bias[DG_MAX_LIN];
    int N[DG_MAX_LIN];
    int tile0[DG_MAX_LIN + 1]; // first column tile of each linear in the launch's tile list
    const f16 *X;
    int nlin, M, K, tiles_m, tiles_n, per_xcd;
    int by_column;
    GroupWalk walk; // row tiles (by_column: column tiles) are the outer ones
};

template <int B, int E, class F> __device__ __forceinline__ void dg_for(F &&f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>());
        dg_for<B + 1, E>(f);
    }
}

// where a row keeps its 16-byte piece kc of a step
__device__ __forceinline__ int dg_swizzle(int r, int kc) { return kc ^ ((r >> 1) & 7); }

// WM x WN waves of TM x TN MFMA tiles: a block of 16 WM TM rows and 16 WN TN features.  ST stages of 64 columns; a
// step's second half of fragments is read while the first half multiplies, then the stage is handed back, the step ST
// later requested into it and the next step's first fragments read while the second half multiplies: fragment reads,
// requests and the barrier run under MFMAs.
// us a launch, with LDS reads in one go, requests in half of a step and blocks of 64 x 128 to 256 x 256 in two or three
// stages / as here, in turn on one machine: 8192 rows 768 -> 768 14.4 / 13.7, 768 -> 928 16.7 / 16.6, 768 -> 1536 23.2 / 23.1,
// 768 -> 3072 42.4 / 41.8, 3072 -> 768 44.3 / 37.0; 2000 rows 768 -> 2304 13.5 / 12.4, 3072 -> 768 18.8 / 17.0; 2003 rows 3072 ->
// 3072 45.9 / 37.2; 1200 rows 4096 -> 1024 23.3 / 20.4; 16384 rows 1024 -> 4096 126.3 / 119.8 (1150 TFLOP/s), 4096 -> 1024 108.6
// / 103.4 (1330); 4096 x 4096 x 4096 108.6 / 103.4 (1330), 8192 x 8192 x 8192 897 / 753 (1460).
// In the same blocks, as the mean over 60 shapes: reads between the products 256 x 256 6 %, else 2 %; requests over the
// whole step, with three stages and more, 4 to 5 %; the barrier in front of a half's last products 1 to 3 % where a CU has
// one workgroup.
template <bool GELU, int WM, int WN, int TM, int TN, int ST>
__global__ void __launch_bounds__(WM *WN * 64) dense_gemm_kernel(
    // (what the first requests need arrives in registers with the wave)
    const f16 *hot_X, const f16 *hot_W, int hot_M, int hot_K, int hot_N, int hot_per_xcd, int hot_total, int hot_div,
    unsigned hot_div_magic, int hot_nlin, const DgArgs args) {
    DgArgs a = args;
    a.X = hot_X;
    a.M = hot_M;
    a.K = hot_K;
    a.per_xcd = hot_per_xcd;
    a.walk.total = hot_total;
    a.walk.div = hot_div;
    a.walk.div_magic = hot_div_magic;
    a.nlin = hot_nlin & 15;
    a.by_column = hot_nlin >> 4 & 1;
    a.walk.group = hot_nlin >> 5;
    constexpr int NW = WM * WN, BM = WM * TM * 16, BN = WN * TN * 16;
    extern __shared__ __attribute__((aligned(16))) unsigned char dg_smem[];
    f16 *smem = reinterpret_cast<f16 *>(dg_smem);
    constexpr int XT = BM * DG_BK, STAGE = XT + BN * DG_BK; // halves
    // consecutive ids on one XCD walk the column tiles of a group of row tiles (dg_group), whose X tiles stay in that
    // XCD's L2 meanwhile, and W is everywhere - or, where X is the smaller one, the other way round
    const int vid = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    if (vid >= a.walk.total)
        return;
    int outer, inner;
    group_walk_at(a.walk, vid, outer, inner); // (one tile a group: only what came in registers, the rest is a round trip to memory)
    const int tm = a.by_column ? inner : outer, tn_all = a.by_column ? outer : inner;
    int lin = 0, tn = tn_all, N = hot_N;
    const f16 *W = hot_W;
    if (a.nlin > 1) { // (wave-uniform)
#pragma unroll
        for (int i = 1; i < DG_MAX_LIN; i++)
            lin += (i < a.nlin && tn_all >= a.tile0[i]) ? 1 : 0;
        tn = tn_all - (lin == 0 ? a.tile0[0] : lin == 1 ? a.tile0[1] : a.tile0[2]);
        W = lin == 0 ? a.W[0] : lin == 1 ? a.W[1] : a.W[2];
        N = lin == 0 ? a.N[0] : lin == 1 ? a.N[1] : a.N[2];
    }
    f16 *const Y = lin == 0 ? a.Y[0] : lin == 1 ? a.Y[1] : a.Y[2];
    const f16 *const bias = lin == 0 ? a.bias[0] : lin == 1 ? a.bias[1] : a.bias[2];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int c16 = lane & 15, g4 = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;
    const int m0 = tm * BM, n0 = tn * BN;
    const int nk = (a.K + DG_BK - 1) / DG_BK;

    // requests of a stage per wave: 1 KB = eight rows each
    constexpr int NXI = BM / 8 / NW, NWI = BN / 8 / NW;
    static_assert(BM / 8 % NW == 0 && BN / 8 % NW == 0, "whole instructions per wave");
    unsigned xoff[NXI], woff[NWI]; // byte offsets of the lane's pieces in step 0 (rows beyond M, N: the last one's)
#pragma unroll
    for (int i = 0; i < NXI; i++) {
        const int r = (wave * NXI + i) * 8 + (lane >> 3);
        const int kc = dg_swizzle(r, lane & 7);
        xoff[i] = (unsigned)((min(m0 + r, a.M - 1) - m0) * a.K + kc * 8) * 2u;
    }
#pragma unroll
    for (int i = 0; i < NWI; i++) {
        const int r = (wave * NWI + i) * 8 + (lane >> 3);
        const int kc = dg_swizzle(r, lane & 7);
        woff[i] = (unsigned)((min(n0 + r, N - 1) - n0) * a.K + kc * 8) * 2u;
    }
    const char *const xbase = reinterpret_cast<const char *>(a.X + (size_t)m0 * a.K);
    const char *const wbase = reinterpret_cast<const char *>(W + (size_t)n0 * a.K);
    const int tail_cols = a.K - (nk - 1) * DG_BK; // 64, or 32: pieces beyond it re-read the step's first ones
    constexpr int PER = NXI + NWI; // requests of a stage per wave
    auto request = [&](int kt, int slot, auto which) { // one of them
        constexpr int Q = decltype(which)::value, I = Q < NXI ? Q : Q - NXI, PIECE = Q < NXI ? NXI : NWI;
        f16 *dst = smem + slot * STAGE + (Q < NXI ? 0 : XT) + (wave * PIECE + I) * 512;
        const char *src = (Q < NXI ? xbase : wbase) + (size_t)kt * (DG_BK * 2);
        // (beyond a short last step: the swizzle flips bit 2 of a piece's number with the parity of its eight rows)
        const bool tail = kt == nk - 1 && tail_cols < DG_BK;
        const unsigned back = tail && ((lane >> 2 ^ (wave * PIECE + I)) & 1) ? 64u : 0u;
        unsigned o = Q < NXI ? xoff[Q < NXI ? I : 0] : woff[Q < NXI ? 0 : I];
        asm volatile("" : "+v"(o)); // (a 32-bit offset off a uniform base, not a 64-bit pointer kept per piece)
        load_lds16(src + (o - back), dst);
    };
    auto fetch = [&](int kt, int slot) { dg_for<0, PER>([&](auto which) { request(kt, slot, which); }); };
    f32x4 acc[TN][TM]; // [feature subtile][row subtile]
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    f16x8 xf[2][TM], wf[2][TN];
    // LDS byte offsets of the lane's fragment pieces (subtile j is 16 rows further)
    const int rx = wm * TM * 16 + c16, rw = wn * TN * 16 + c16;
    const int px[2] = {rx * 128 + dg_swizzle(rx, g4) * 16, rx * 128 + dg_swizzle(rx, 4 + g4) * 16};
    const int pw[2] = {XT * 2 + rw * 128 + dg_swizzle(rw, g4) * 16, XT * 2 + rw * 128 + dg_swizzle(rw, 4 + g4) * 16};
    auto read = [&](int slot, auto half) {
        constexpr int H = decltype(half)::value;
        const char *s = reinterpret_cast<const char *>(smem) + slot * (STAGE * 2);
#pragma unroll
        for (int i = 0; i < TN; i++)
            wf[H][i] = *reinterpret_cast<const f16x8 *>(s + pw[H] + i * 2048);
#pragma unroll
        for (int j = 0; j < TM; j++)
            xf[H][j] = *reinterpret_cast<const f16x8 *>(s + px[H] + j * 2048);
    };
    // (LDS reads in one go keep the wave from its products until the last one is out: a half's fragments are read behind the
    // products of the other half's first OVER row subtiles)
    constexpr int FRAG = TM + TN, OVER = TM >= 4 ? TM / 2 : TM;
    auto read_some = [&](int slot, auto half, auto jc) {
        constexpr int H = decltype(half)::value, j = decltype(jc)::value;
        const char *s = reinterpret_cast<const char *>(smem) + slot * (STAGE * 2);
        if constexpr (j < OVER)
            dg_for<j * FRAG / OVER, (j + 1) * FRAG / OVER>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if constexpr (i < TN)
                    wf[H][i] = *reinterpret_cast<const f16x8 *>(s + pw[H] + i * 2048);
                else
                    xf[H][i - TN] = *reinterpret_cast<const f16x8 *>(s + px[H] + (i - TN) * 2048);
            });
        __builtin_amdgcn_sched_barrier(0);
    };
    // (two workgroups on a CU: the one that multiplies goes first, and it has the other one's work while its waves wait)
    constexpr bool SHARED = ST * STAGE * 2 <= 80 * 1024;
    auto multiply = [&](auto half, auto &&between) { // between(j): what goes out behind the products of row subtile j
        constexpr int H = decltype(half)::value;
        if (SHARED)
            __builtin_amdgcn_s_setprio(1);
        dg_for<0, TM>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
#pragma unroll
            for (int i = 0; i < TN; i++)
                acc[i][j] = mfma16x16x32(wf[H][i], xf[H][j], acc[i][j]);
            between(jc);
        });
        if (SHARED)
            __builtin_amdgcn_s_setprio(0);
    };
    auto nothing = [](auto) {};
    typedef std::integral_constant<int, 0> h0;
    typedef std::integral_constant<int, 1> h1;
    auto barrier = [] { asm volatile("s_barrier" ::: "memory"); };
    auto landed = [&](auto behind) { // all but the youngest `behind` stages have arrived (this wave's part of them)
        constexpr int V = decltype(behind)::value * PER;
        static_assert(V < 64, "what vmcnt counts");
        __builtin_amdgcn_s_waitcnt(0x0070 | (V & 15) | (V >> 4 << 14)); // vmcnt(V) lgkmcnt(0)
    };
#pragma unroll
    for (int t = 0; t < ST - 1; t++)
        if (t < nk)
            fetch(t, t);
    if (nk >= ST - 1)
        landed(std::integral_constant<int, ST - 2>());
    else
        landed(h0());
    barrier();
    // A stage's requests go out between the products as well, while the matrix unit is busy: with more than two stages the
    // first EARLY of them in the step that frees the place, the others in the first half of the next one.
    constexpr int EARLY = ST > 2 ? (PER + 1) / 2 : PER;
    // The barrier that hands a step's stage over stands in front of the first half's last products, so that the matrix unit
    // has work while the waves wait for each other.  (What is requested in this half goes out before it: it is counted.)
    constexpr int BEFORE = TM >= 4 && !SHARED ? TM - 1 : TM; // row subtiles in front of the barrier
    auto request_some = [&](int stage, int slot, auto jc, auto over, auto from, auto to) { // behind the products of row subtile j
        constexpr int j = decltype(jc)::value, OV = decltype(over)::value, F = decltype(from)::value, N = decltype(to)::value - F;
        if constexpr (j < OV)
            dg_for<F + j * N / OV, F + (j + 1) * N / OV>([&](auto which) { request(stage, slot, which); });
        __builtin_amdgcn_sched_barrier(0);
    };
    typedef std::integral_constant<int, TM> every_t;
    typedef std::integral_constant<int, BEFORE> before_t;
    typedef std::integral_constant<int, 0> none_t;
    typedef std::integral_constant<int, EARLY> early_t;
    typedef std::integral_constant<int, PER> all_t;
    if (ST - 1 < nk)
        dg_for<0, EARLY>([&](auto which) { request(ST - 1, ST - 1, which); });
    read(0, h0());
    int slot = 0, freed = ST - 1;
    auto step = [&](int kt, auto late, auto early, auto behind) {
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): the first half's fragments, read a multiplication ago
        multiply(h0(), [&](auto jc) {
            constexpr int j = decltype(jc)::value;
            read_some(slot, h1(), jc);
            if constexpr (decltype(late)::value && EARLY < PER)
                request_some(kt - 1 + ST, freed, jc, before_t(), early_t(), all_t());
            if constexpr (j == BEFORE - 1) { // this wave has the step's fragments and its part of the next stage
                landed(behind);
                barrier();
            }
        });
        freed = slot;
        slot = slot == ST - 1 ? 0 : slot + 1;
        multiply(h1(), [&](auto jc) {
            read_some(slot, h0(), jc);
            if constexpr (decltype(early)::value)
                request_some(kt + ST, freed, jc, every_t(), none_t(), early_t());
        });
    };
    typedef std::integral_constant<int, ST - 2> steady_t;
    int kt = 0;
    for (; kt < nk - ST; kt++)
        step(kt, std::true_type(), std::true_type(), steady_t());
    if (kt == nk - ST)
        step(kt++, std::true_type(), std::false_type(), steady_t());
    dg_for<0, ST - 2>([&](auto ic) { // everything has been requested
        constexpr int BEHIND = ST - 3 - decltype(ic)::value;
        if (nk - 2 - kt == BEHIND)
            step(kt++, std::false_type(), std::false_type(), std::integral_constant<int, BEHIND>());
    });
    // (the last step apart: with a branch around the next stage's reads the compiler cannot tell which are in flight behind
    // it, and waits for them before it multiplies)
    __builtin_amdgcn_s_waitcnt(0xC07F);
    read(slot, h1());
    __builtin_amdgcn_sched_barrier(0);
    multiply(h0(), nothing);
    if (tail_cols == DG_BK)
        multiply(h1(), nothing);
    __builtin_amdgcn_s_waitcnt(0x0070);
    barrier(); // the stages are free: they stage the output block

    // acc[i][j][r] = Y[row = m0 + wm*16*TM + j*16 + c16][col = n0 + wn*16*TN + i*16 + g4*4 + r]
    // -> the wave's rows in LDS, 64 at a time ([row][16 TN halves + 8]), then 16-byte stores
    constexpr int LDO = 16 * TN + 8, CH = 2 * TN; // 16-byte pieces per row
    constexpr int TR = TM < 4 ? TM : TM % 4 == 0 ? 4 : 3; // row subtiles per pass
    static_assert(TM % TR == 0 && (size_t)NW * TR * 16 * LDO <= ST * (size_t)STAGE, "the output staging fits the stages");
    f16 *os = smem + wave * TR * 16 * LDO;
    f32x4 bf[TN];
#pragma unroll
    for (int i = 0; i < TN; i++) {
        const int col = n0 + (wn * TN + i) * 16 + g4 * 4;
        f16x4 b4 = f16x4{0, 0, 0, 0};
        if (col < N)
            b4 = *reinterpret_cast<const f16x4 *>(bias + col);
        bf[i] = __builtin_convertvector(b4, f32x4);
    }
#pragma unroll
    for (int p = 0; p < TM / TR; p++) {
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int j = 0; j < TR; j++) {
                f16x4 ov = __builtin_convertvector(acc[i][p * TR + j] + bf[i], f16x4);
                if (GELU)
                    ov = gelu4(ov);
                *reinterpret_cast<f16x4 *>(os + (j * 16 + c16) * LDO + i * 16 + g4 * 4) = ov;
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // (the staging block is the wave's own: LDS operations of one wave execute in order)
#pragma unroll
        for (int t = 0; t < (TR * 16 * CH + 63) / 64; t++) {
            const int q = t * 64 + lane, r = q / CH, pc = q % CH;
            const int row = m0 + wm * TM * 16 + p * TR * 16 + r, col = n0 + wn * TN * 16 + pc * 8;
            if (TR * 16 * CH % 64 != 0 && r >= TR * 16) // (three subtiles of three: the last pieces are half a wave's)
                continue;
            if (row < a.M && col < N) // N is a multiple of 16: a piece is inside or outside as a whole
                *reinterpret_cast<u32x4 *>(Y + (size_t)row * N + col) = *reinterpret_cast<const u32x4 *>(os + r * LDO + pc * 8);
        }
    }
}

// Row-major copy of a fully populated plan's weights: a workgroup per (chunk, block-row), a thread per 16-byte half row
// of a tile (tiles of a segment are in column order; a segment's padding tile is not read).
__global__ void __launch_bounds__(256) dense_from_plan_kernel(f16 *W, const f16 *data, const int *cptr, int K, int KC, int nbr) {
    const int c = blockIdx.x / nbr, bn = blockIdx.x - c * nbr;
    const int ntile = (min(KC, K - c * KC) + 15) / 16;
    const f16 *const src = data + (size_t)cptr[blockIdx.x] * 256;
    f16 *const dst = W + (size_t)bn * 16 * K + c * KC;
    for (int q = threadIdx.x; q < ntile * 32; q += 256) {
        const int t = q >> 5, r = (q >> 1) & 15, h = q & 1;
        *reinterpret_cast<u32x4 *>(dst + (size_t)r * K + t * 16 + h * 8) =
            *reinterpret_cast<const u32x4 *>(src + t * 256 + r * 16 + h * 8);
    }
}
int dense_from_plan(f16 *W, const f16 *data, const int *cptr, int K, int KC, int nchunk, int nbr) {
    hipLaunchKernelGGL(dense_from_plan_kernel, dim3(nchunk * nbr), dim3(256), 0, nullptr, W, data, cptr, K, KC, nbr);
    return launch_status("dense_from_plan launch");
}

// How many row tiles (or column tiles, whichever the launch has as its outer ones) are walked together.  What an XCD's
// workgroups fetch at the same time should be few tiles: a block of rows x columns of them, not one row.  Best of 1, 2, 4 ..
// 16 by what the blocks at work take in per step; it is the group measured best for the blocks of 64 x 128 to 256 x 256 (1 to 4
// within 2 %).  8192 x 8192 x 8192 931 -> 863 us (64 x 128 blocks 2370 -> 1240, 128 x 192 1190 -> 930), 2003 rows 3072 -> 3072
// 46.4 -> 44.6, 16384 rows 1024 -> 4096 128.8 -> 126.7.  Not where all blocks are at work at once: 2000 rows 768 -> 2304 (192
// blocks) took 12.5 us instead of 12.0.
// Where a group saves few tiles it is a trade: whole unpruned layers 512 wide, whose Q/K/V launch takes in 16 tiles a step
// instead of 17, without groups / with them, us: on operands that change from pass to pass 33 x 337 rows 144.4 / 146.1, 21 x 600
// 174.6 / 169.5, 24 x 512 163.4 / 160.8, 26 x 512 172.8 / 168.2; on the same ones at every pass 137.5 / 139.0, 157.8 / 159.3,
// 143.4 / 143.5, 153.0 / 155.1.
static int dg_group(int outer, int inner, int outer_rows, int inner_rows, int per_cu) {
    const int cus = std::max(et_device_cu_count(), 8), at_once = cus / 8 * per_cu;
    if ((long)outer * inner <= (long)cus * per_cu)
        return 1;
    int best = 1, least = 0;
    for (int g = 1; g <= std::min(outer, 16); g *= 2) {
        const int cols = std::min(inner, std::max(at_once / g, 1)), rows = std::max(at_once / cols, 1);
        const int taken = rows * outer_rows + cols * inner_rows;
        if (g == 1 || taken < least) {
            best = g;
            least = taken;
        }
    }
    return best;
}

template <bool GELU, int WM, int WN, int TM, int TN, int ST> static int dg_launch_inst(DgArgs &a, hipStream_t st) {
    constexpr int BM = WM * TM * 16, BN = WN * TN * 16;
    constexpr int lds = ST * (BM + BN) * DG_BK * (int)sizeof(f16);
    a.tiles_m = (a.M + BM - 1) / BM;
    a.tiles_n = 0;
    double n = 0.0;
    for (int i = 0; i < DG_MAX_LIN; i++) {
        a.tile0[i] = i < a.nlin ? a.tiles_n : 0;
        if (i < a.nlin) {
            a.tiles_n += (a.N[i] + BN - 1) / BN;
            n += a.N[i];
        }
    }
    // (every L2 that has part of the work takes the operand that all of the work shares)
    a.by_column = tl_order(2.0 * a.M * a.K, 2.0 * a.K * n, a.tiles_m, a.tiles_n, 4.5e6);
    const int outer = a.by_column ? a.tiles_n : a.tiles_m, inner = a.by_column ? a.tiles_m : a.tiles_n;
    if (!group_walk(a.walk, outer, inner, dg_group(outer, inner, a.by_column ? BN : BM, a.by_column ? BM : BN, lds <= 80 * 1024 ? 2 : 1)))
        return ROWS_TOO_MANY;
    a.per_xcd = (a.walk.total + 7) / 8;
    constexpr auto kern = &dense_gemm_kernel<GELU, WM, WN, TM, TN, ST>;
    launch_kernel<kern>(dim3(a.per_xcd * 8), dim3(WM * WN * 64), lds, st, a.X, a.W[0], a.M, a.K, a.N[0],
                       a.per_xcd, a.walk.total, a.walk.div, a.walk.div_magic, a.nlin | a.by_column << 4 | a.walk.group << 5, a);
    return launch_status("dense_gemm launch");
}

// The blocks there are and the time of each form in microseconds, without the launch.  A step takes longer with every
// further workgroup of a CU and with the share of the CUs that have one; the figures are fits to 860 shapes (150 to 18000
// rows, 512 to 4096 columns, random weights, a quarter of them with GELU), the forms near the fastest weighing most.  Fitted
// to one half, the block they choose for the other is 0.2 % behind the fastest in the mean, 17 % at most (512 -> 768, 5453
// rows: 10.6 against 9.0 us), and its estimate with 3.0 us for the launch 3 % off.  What decides is how many bytes of X and
// W the busiest CU takes in, at about 100 GB/s by DMA, and that no CU has a block more than the others: small blocks win
// while they let more CUs take part, large ones where every CU has several, and of those near in size the one whose count
// fills its last round.  (Blocks of 192 x 192 were the shorter launch for some hundred of 860 shapes, by 2 %; 6144 rows
// 768 -> 3072 inside a layer took 5 us more.)  The blocks of 32 to 96 rows x 64 or 96 and of 192 x 256 against the others alone, us: 3072
// -> 768 512 rows 14.8 / 11.0, 1024 16.3 / 12.9, 2000 16.3 / 15.3, 3000 20.6 / 18.2; 4096 -> 1024 512 rows 18.9 / 14.2, 1024
// 19.7 / 16.5; 2048 -> 512 1200 rows 10.8 / 8.9; 1024 -> 4096 3000 rows 30.3 / 27.4, 6000 57.0 / 50.9; 512 -> 2048 6000 rows
// 20.2 / 18.0; the 640 shapes without GELU 10.5 % in the geometric mean.
enum {
    DG_64x128 = 0, DG_128x128, DG_128x128_DEEP, DG_128x192, DG_256x256, DG_192x256, DG_128x192_DEEP, DG_64x64, DG_32x64,
    DG_96x64, DG_96x96, DG_FORMS
};
static std::atomic<int> g_dense_form{-1}; // et_tuning_set("dense_form"): one of the above, -1 chooses
static double dg_estimate(int form, const int *Ns, int nlin, int M, int K, bool gelu) {
    static const int bm[DG_FORMS] = {64, 128, 128, 128, 256, 192, 128, 64, 32, 96, 96};
    static const int bn[DG_FORMS] = {128, 128, 128, 192, 256, 256, 192, 64, 64, 64, 96};
    struct Form {
        double ends;        // the first step's latency and the way out
        double one, fill1;  // a step while no CU has two blocks, per share of CUs that have one
        double two, fill2;  // ... while none has three
        double more, fill3; // ... a block, per block that the CUs have in the mean
        double gelu;        // of 128 x 128 results
    };
    static const Form forms[DG_FORMS] = {
        {0.118, 0.226, 0.091, 0.541, 0.072, 0.238, 0.144, 1.165}, // one per CU (144 KB)
        {0.918, 0.279, 0.234, 0.323, 0.338, 0.292, 0.275, 0.827}, // two per CU (64 KB)
        {0.708, 0.269, 0.189, 0.682, 0.186, 0.237, 0.372, 1.096}, // one per CU (128 KB)
        {1.425, 0.303, 0.494, 0.579, 0.441, 0.429, 0.352, 0.745}, // two per CU (80 KB)
        {5.481, 0.677, 0.784, 1.777, 0.821, 1.479, 0.301, 0.890}, // one per CU (128 KB)
        {4.006, 0.535, 0.631, 1.451, 0.617, 0.759, 0.735, 0.859}, // one per CU (112 KB)
        {1.758, 0.294, 0.361, 0.778, 0.344, 0.415, 0.418, 1.088}, // one per CU (120 KB)
        {0.000, 0.166, 0.049, 0.425, 0.037, 0.135, 0.136, 0.619}, // one per CU (128 KB)
        {0.000, 0.133, 0.034, 0.332, 0.035, 0.151, 0.067, 0.037}, // one per CU (144 KB)
        {0.041, 0.211, 0.056, 0.532, 0.012, 0.189, 0.122, 1.351}, // one per CU (140 KB)
        {0.401, 0.250, 0.082, 0.551, 0.082, 0.134, 0.286, 1.423}, // one per CU (144 KB)
    };
    const long cus = std::max(et_device_cu_count(), 1);
    long tiles = 0;
    for (int i = 0; i < nlin; i++)
        tiles += (Ns[i] + bn[form] - 1) / bn[form];
    tiles *= (M + bm[form] - 1) / bm[form];
    const Form &f = forms[form];
    const long n = (tiles + cus - 1) / cus; // blocks of the busiest CU
    const double fill = (double)tiles / (double)cus;
    const double step = n <= 1 ? f.one + f.fill1 * fill : n <= 2 ? f.two + f.fill2 * fill : f.more * (double)n + f.fill3 * fill;
    return f.ends + step * ((K + DG_BK - 1) / DG_BK) + (gelu ? f.gelu * (double)n * bm[form] * bn[form] / 16384.0 : 0.0);
}
// The choice, kept for sizes that come again: a plan's launch asks twice, for the line to the tile kernels and for the
// block (61 rows 768 -> 768 without pruning, bound by the host: 5.0 us a call weighed each time, 4.4 so).
struct DenseChoice {
    int form;
    double us;
};
typedef KeptChoices<DenseChoice, 5 + DG_MAX_LIN> DenseChoices;
static DenseChoice dg_choose(const int *Ns, int nlin, int M, int K, bool gelu) {
    static thread_local DenseChoices kept;
    DenseChoices::Key k = {{nlin, M, K, gelu, std::max(et_device_cu_count(), 1)}};
    for (int i = 0; i < nlin; i++)
        k.v[5 + i] = Ns[i];
    return kept.get(k, [&] {
        DenseChoice best = {0, dg_estimate(0, Ns, nlin, M, K, gelu)};
        for (int f = 1; f < DG_FORMS; f++) {
            const double us = dg_estimate(f, Ns, nlin, M, K, gelu);
            if (us < best.us)
                best = DenseChoice{f, us};
        }
        return best;
    });
}
double dense_gemm_estimate(const int *Ns, int nlin, int M, int K, bool gelu) {
    const int set = g_dense_form;
    return set >= 0 ? dg_estimate(set, Ns, nlin, M, K, gelu) : dg_choose(Ns, nlin, M, K, gelu).us;
}
void set_dense_form(int v) { g_dense_form = v < DG_FORMS ? v : -1; }

// nlin linears over the same X in one launch.  Returns ET_ERR_UNSUPPORTED where
// the shapes do not fit this kernel (the caller then takes the tile path).
static int dense_gemm_rows(void *const *Ys, const void *X, const void *const *Ws, const void *const *biases,
                           const int *Ns, int nlin, int M, int K, bool gelu, hipStream_t st) {
    if (nlin < 1 || nlin > DG_MAX_LIN || K < 32 || K % 32 != 0 || M <= 0)
        return ET_ERR_UNSUPPORTED;
    DgArgs a;
    memset(&a, 0, sizeof(a));
    for (int i = 0; i < DG_MAX_LIN; i++) {
        const int s = i < nlin ? i : 0;
        if (Ns[s] <= 0 || Ns[s] % 16 != 0 || !aligned16(Ys[s]) || !aligned16(Ws[s]) || !aligned16(biases[s]))
            return ET_ERR_UNSUPPORTED;
        a.Y[i] = static_cast<f16 *>(Ys[s]);
        a.W[i] = static_cast<const f16 *>(Ws[s]);
        a.bias[i] = static_cast<const f16 *>(biases[s]);
        a.N[i] = Ns[s];
    }
    if (!aligned16(X))
        return ET_ERR_UNSUPPORTED;
    a.X = static_cast<const f16 *>(X);
    a.nlin = nlin;
    a.M = M;
    a.K = K;
    const int set = g_dense_form, form = set >= 0 ? set : dg_choose(Ns, nlin, M, K, gelu).form;
    switch (form) {
#define DG_CASE(form_, ...)                                                                                            \
    case form_: return gelu ? dg_launch_inst<true, __VA_ARGS__>(a, st) : dg_launch_inst<false, __VA_ARGS__>(a, st);
        DG_CASE(DG_64x128, 2, 4, 2, 2, 6)
        DG_CASE(DG_128x128, 2, 4, 4, 2, 2)
        DG_CASE(DG_128x128_DEEP, 2, 4, 4, 2, 4)
        DG_CASE(DG_128x192, 2, 4, 4, 3, 2)
        DG_CASE(DG_256x256, 2, 4, 8, 4, 2)
        DG_CASE(DG_128x192_DEEP, 2, 4, 4, 3, 3)
        // (four waves: a block of 64 x 64 in eight is 3 % slower, its waves read more fragments for a product)
        DG_CASE(DG_64x64, 2, 2, 2, 2, 8)
        DG_CASE(DG_32x64, 2, 2, 1, 2, 12)
        DG_CASE(DG_96x64, 2, 2, 3, 2, 7)
        DG_CASE(DG_96x96, 2, 2, 3, 3, 6)
        DG_CASE(DG_192x256, 2, 4, 6, 4, 2)
#undef DG_CASE
    }
    return ET_ERR_UNSUPPORTED;
}
int dense_gemm_launch(void *const *Ys, const void *X, const void *const *Ws, const void *const *biases,
                      const int *Ns, int nlin, int M, int K, bool gelu, hipStream_t st) {
    int rc = dense_gemm_rows(Ys, X, Ws, biases, Ns, nlin, M, K, gelu, st);
    if (rc != ROWS_TOO_MANY)
        return rc;
    const int first = M / 2 / 256 * 256; // (rows are independent)
    ET_REQUIRE(first > 0, ET_ERR_UNSUPPORTED, "dense product: %d rows and so many outputs are too many blocks", M);
    void *rest[DG_MAX_LIN];
    for (int i = 0; i < nlin; i++)
        rest[i] = static_cast<f16 *>(Ys[i]) + (size_t)first * Ns[i];
    rc = dense_gemm_launch(Ys, X, Ws, biases, Ns, nlin, first, K, gelu, st);
    return rc != ET_OK ? rc
                       : dense_gemm_launch(rest, static_cast<const f16 *>(X) + (size_t)first * K, Ws, biases, Ns, nlin, M - first, K, gelu, st);
}

} // namespace et

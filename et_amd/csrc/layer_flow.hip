// A whole encoder layer in ONE launch for few rows (Q/K/V, attention, output
// projection, skip + LayerNorm, feed-forward block, skip + LayerNorm;
// encoder/encoder.cu:20-45 of the reference).
//
// Why.  With few rows a layer is a chain of launches that each do a microsecond
// of work: seven launches of 3-10 us for 37 to a few hundred rows, of which
// ~2.4 us each is the boundary between two dependent launches and most of the
// rest is fetching weights that were known all along.  Here every step of the
// layer is cut into units of work, one workgroup per unit, all in one grid; a
// unit requests its weights first and only then waits for the rows it needs.
// A hand-over between workgroups (store, acknowledge, counter, poll, load) was
// measured at 1.5 us, and the weights of the later steps arrive while the
// earlier ones run.
//
// Order and progress.  A workgroup takes a ticket from a counter in memory and
// runs the unit of that number; units are numbered step by step, so a unit only
// ever waits for units with smaller numbers, whose workgroups have taken their
// ticket before and are on the chip.  Whatever else runs on the device, the
// smallest unfinished unit never waits: no deadlock, and no assumption about
// how many workgroups are resident.  (Waits are bounded all the same and report
// through the wait-status word.)
//
// Visibility.  The chip has eight L2 caches that are not coherent with each
// other.  Rows handed over inside the launch are stored with agent scope (past
// the writer's L2), counted in after their acknowledgement, and every such
// buffer is written once per launch and read only after the counter says so -
// no cache can hold an older copy of a line from this launch, and those of
// earlier launches were dropped when this one started.  Plain loads are then
// correct; the buffers must not be reused inside the launch.  Nor may a line
// hold rows of two panels: the line would be pulled into an L2 with one panel's
// rows, before the other's are stored, and read there again later.  So every
// buffer that is handed over lies in the object's own scratch, from whole lines
// on, and rows are whole lines (d and dff multiples of 64); the caller's
// workspace units need only be 16-byte aligned and are not used.
//
// Counters (one 128-byte line each): a workgroup that finishes a unit adds one
// to its row panel's counter of that step.  The workgroup that completes the
// last step of a panel runs its final LayerNorm; the one that does so for the
// last panel ends the launch's books.  There are two sets of counters, taken in
// turn: the launch that uses one leaves the other at zero for its successor.
// Its own set it must leave alone - after a wait that gave up, units of earlier
// steps may still be running and add to it.  The word that the tickets come from
// also says whose turn it is (its top bit); it can be set back at that point,
// since the units that complete the last panel have the highest tickets.
//
// Units.  Linears: 16 rows x (16 / split) block-rows of 16 output features; the
// pairs of surviving tiles of a block-row are split over `split` waves, so that
// a wave has its whole share of W in registers before it waits, and the partial
// sums meet in LDS in a fixed order.  The projections and the first feed-forward
// linear hold the 16-row panel in LDS; the second feed-forward linear (hidden
// width: too wide for a panel) reads its operand from memory, only the surviving
// tiles' columns, two block-rows per workgroup with eight waves each.  The first LayerNorm is
// recomputed by every workgroup of the first feed-forward linear that needs the
// rows (one hand-over less), and by those of the second one for its skip operand
// while they wait, where every unit has a CU of its own (0.2 to 0.7 us less than
// having the first linear's store it; with more units 1.2 us more).  Attention: attention_block, 256 query rows per
// unit and head.  Where the lists are short enough for a wave's registers, heads
// are 64 wide and sequences at most 128 rows, a unit is a head's projections AND
// attention (qkv_block.h): a hand-over less.  80 % pruned, 768 wide: 16 rows
// 24.5 -> 18.9 us, 37 25.1 -> 21.1, 64 25.0 -> 22.8, 96 28.1 -> 24.9.  Where the
// 21 us of 37 rows go: launch and ticket 3, projections and attention 5.8 (a CU
// reads 1 KB of X from LDS per product), then per step 1.2 to 2.5 of work (rows
// from memory 0.9, LayerNorm of 16 rows 0.9), 0.7 for the stores to be
// acknowledged and 0.4 until the counter is seen.
#include "qkv_block.h"
#include "row_ln.h"
#include "tile_walk.h"

#include <algorithm>
#include <cstring>
#include <vector>

namespace et {

int tail_spin();

constexpr int LF_WAVES = 16;
constexpr int LF_BM = 16;      // rows per panel: a wave each in the LayerNorms
constexpr int LF_QB = 256;     // query rows per attention unit
constexpr int LF_SHARE = 12;   // ... that a wave's share of a block-row should not exceed
constexpr int LF_CS = 32;      // counter stride in words: a line each
constexpr int LF_HEAD_PAIRS = 12; // tile pairs of a block-row in a unit of projections and attention (sixteen waves: 128 registers)

struct LfArgs {
    AttnArgs at; // Q, K, V, out: scratch that the steps hand over
    QaArgs qa;   // FUSED: projections and attention of a head
    LfLinear q, k, v, o, m1, m2;
    const f16 *in;
    f16 *out;
    f16 *oraw, *ln1, *hid, *fraw; // output projection, first LayerNorm, hidden activations, second linear
    const f16 *gamma1, *beta1, *gamma2, *beta2;
    unsigned *ctr;  // tickets and the set in turn, then the two sets of nctr counters
    const int *blk; // attention blocks: [2i] sequence, [2i+1] query block; then per panel first and last block
    int M, d, dff, npanel, nblk;
    float inv_d;
    int again; // the second feed-forward linear's units compute the first LayerNorm's rows once more
    int u_at, u_o, u_f1, u_f2;             // first unit of each step (Q/K/V: 0)
    int g_qkv, g_o, g_f1, g_f2;            // units per panel
    int gl_q, gl_k;                        // ... of the query and key linears
    int s_qkv, s_o, s_f1, s_f2;            // log2 of the split
    int nctr;                              // counters in a set
    int misc;                              // LDS byte offset of the broadcast words
    int spin;
    int *status;
};

// ---- hand-over --------------------------------------------------------------
// wave 0: lanes 0..n-1 wait until counter first + lane has reached target
__device__ __forceinline__ void lf_poll(const LfArgs &a, const unsigned *ctr, int first, int n, unsigned target) {
    const int lane = threadIdx.x & 63;
    for (int i0 = 0; i0 < n; i0 += 64) {
        const int i = min(i0 + lane, n - 1);
        for (int s = 0;; s++) {
            const unsigned c = __hip_atomic_load(ctr + (size_t)(first + i) * LF_CS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__builtin_amdgcn_ballot_w64(c < target) == 0)
                break;
            if (s >= a.spin) {
                if (lane == 0)
                    __hip_atomic_store(a.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
    }
}
// barrier that orders LDS traffic and keeps the compiler from moving any memory access across it
__device__ __forceinline__ void lf_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
__device__ __forceinline__ void lf_wait(const LfArgs &a, const unsigned *ctr, int wave, int first, int n, unsigned target) {
    asm volatile("" ::: "memory");
    if (wave == 0)
        lf_poll(a, ctr, first, n, target);
    lf_barrier();
}
// every store of the workgroup is acknowledged, then one is added to the counter; thread 0 gets the old value
__device__ __forceinline__ unsigned lf_signal(unsigned *ctr, int c) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lf_barrier();
    unsigned old = 0;
    if (threadIdx.x == 0)
        old = __hip_atomic_fetch_add(ctr + (size_t)c * LF_CS, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return old;
}

// panel in LDS
__device__ __forceinline__ void lf_multiply(f32x4 &acc, LfPairs<LF_D> &p, int n, const LfLinear &l, LfWalk &w,
                                            const char *xlane, unsigned lane_w2, unsigned hi4) {
    while (n > 0) {
#pragma unroll
        for (int g = 0; g < LF_D; g += 2)
            if (n > g) {
                const f16x8 x0 = *reinterpret_cast<const f16x8 *>(xlane + p.o[g] + p.co[g]);
                const f16x8 x1 = *reinterpret_cast<const f16x8 *>(xlane + p.o[g + 1] + p.co[g + 1]);
                acc = mfma16x16x32(p.w[g], x0, acc);
                acc = mfma16x16x32(p.w[g + 1], x1, acc);
            }
        n = lf_request(p, l, w, lane_w2, hi4);
    }
}
// operand rows in memory
__device__ __forceinline__ void lf_multiply_direct(f32x4 &acc, LfPairs<LF_D> &p, int n, const LfLinear &l,
                                                   LfWalk &w, const char *xr, unsigned lane_w2,
                                                   unsigned hi4) {
    while (n > 0) {
        f16x8 x[LF_D];
#pragma unroll
        for (int g = 0; g < LF_D; g += 2)
            if (n > g) {
#pragma unroll
                for (int i = g; i < g + 2; i++)
                    x[i] = *reinterpret_cast<const f16x8 *>(xr + (p.o[i] + p.co[i]));
            }
#pragma unroll
        for (int g = 0; g < LF_D; g += 2)
            if (n > g) {
#pragma unroll
                for (int i = g; i < g + 2; i++)
                    acc = mfma16x16x32(p.w[i], x[i], acc);
            }
        n = lf_request(p, l, w, lane_w2, hi4);
    }
}

// Sums of the split waves meet in LDS (`red`, free for everyone once the barrier
// in front is passed) and are added in the order of the split; bias, GELU, half,
// 8-byte stores of four consecutive features: by the first of the waves that
// share the block-row.
__device__ __forceinline__ f16x4 lf_bias(const LfLinear &l, int bn, int lane) {
    return *reinterpret_cast<const f16x4 *>(l.bias + min(bn, l.nbr - 1) * 16 + (lane >> 4) * 4);
}
template <bool GELU>
__device__ __forceinline__ void lf_put(const LfArgs &a, f32x4 t, f16x4 bias, f16 *Y, int N, int bn, int row, int g4) {
    f16x4 o = __builtin_convertvector(t + __builtin_convertvector(bias, f32x4), f16x4);
    if (GELU)
        o = gelu4(o);
    if (row < a.M)
        store_agent4(Y + (size_t)row * N + bn * 16 + g4 * 4, o);
}
template <bool GELU>
__device__ __forceinline__ void lf_finish(const LfArgs &a, f32x4 acc, f32x4 *red, const LfLinear &l, f16x4 bias,
                                          f16 *Y, int N, int bn, int j, int sub, int ls, int m0, int lane) {
    const int c16 = lane & 15, g4 = lane >> 4, split = 1 << ls, br = LF_WAVES >> ls;
    if (ls == 0) {
        if (bn < l.nbr)
            lf_put<GELU>(a, acc, bias, Y, N, bn, m0 + c16, g4);
        return;
    }
    lf_barrier(); // every wave has read its operands
    red[(sub * br + j) * 64 + lane] = acc;
    lf_barrier();
    if (sub > 0 || bn >= l.nbr)
        return;
    for (int k = 1; k < split; k++)
        acc += red[(k * br + j) * 64 + lane];
    lf_put<GELU>(a, acc, bias, Y, N, bn, m0 + c16, g4);
}

// rows of model width in a wave's registers (row_ln.h)
typedef RowPieces<2> LfPieces;
__device__ __forceinline__ LfPieces lf_pieces(const LfArgs &a, const f16 *row, int lane) { return row_pieces<2>(row, a.d >> 3, lane); }
__device__ __forceinline__ const f16 *lf_row(const LfArgs &a, const f16 *rows, int row) {
    return rows + (size_t)min(row, a.M - 1) * a.d;
}
__device__ __forceinline__ LfPieces lf_layernorm(const LfArgs &a, const LfPieces &y, const LfPieces &skip, const LfPieces &gamma,
                                                 const LfPieces &beta, int lane) {
    return row_layernorm(y, skip, gamma, beta, a.d >> 3, a.inv_d, lane);
}
__device__ __forceinline__ void lf_put_row(const LfArgs &a, f16 *row, const LfPieces &v, int lane) {
    row_put(row, v, a.d >> 3, lane);
}

// rows of X -> panel, DMA; rows at or beyond M stay unwritten (they only feed rows that are never stored)
__device__ __forceinline__ void lf_panel(const LfArgs &a, const f16 *X, f16 *xs, int ldx, int m0, int wave, int lane) {
    const int npiece = a.d >> 3;
    if (m0 + wave < a.M) {
        const f16 *src = X + (size_t)(m0 + wave) * a.d;
        f16 *dst = xs + wave * ldx;
        if (lane < npiece)
            load_lds16(src + lane * 8, dst);
        if (64 + lane < npiece)
            load_lds16(src + (64 + lane) * 8, dst + 512);
    }
}

template <int HD, bool MASK, bool FUSED>
__global__ void __launch_bounds__(LF_WAVES * 64, 4) layer_flow_kernel(const LfArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lf_smem[];
    unsigned *const bc = reinterpret_cast<unsigned *>(lf_smem + a.misc);
    if (threadIdx.x == 0)
        bc[0] = __hip_atomic_fetch_add(a.ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    lf_barrier();
    const unsigned ticket = __builtin_amdgcn_readfirstlane(bc[0]);
    const int unit = (int)(ticket & 0x7FFFFFFFu), set = (int)(ticket >> 31);
    unsigned *const ctr = a.ctr + (size_t)(1 + set * a.nctr) * LF_CS;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int c16 = lane & 15, khalf8 = ((lane >> 4) & 1) * 8;
    const unsigned lane_w2 = (unsigned)((lane >> 5) * 256 + c16 * 16 + khalf8) * 2, hi4 = (lane >> 5) * 4;
    // counters: finished panels, then per panel Q/K/V, O, first and second feed-forward linear, then per attention block
    const int c_qkv = 1, c_o = c_qkv + a.npanel, c_f1 = c_o + a.npanel, c_f2 = c_f1 + a.npanel, c_at = c_f2 + a.npanel;
    f16 *const xs = reinterpret_cast<f16 *>(lf_smem);
    f32x4 *const red = reinterpret_cast<f32x4 *>(lf_smem);
    const int ldx = a.d + 16;
    const char *const xlane = reinterpret_cast<const char *>(xs + c16 * ldx + khalf8);

    if ((!FUSED && unit < a.u_at) || (unit >= a.u_o && unit < a.u_f2)) {
        // ---- a linear on a panel in LDS: Q/K/V, output projection, first feed-forward linear
        const int step = !FUSED && unit < a.u_at ? 0 : unit < a.u_f1 ? 1 : 2;
        const int rel = unit - (step == 0 ? 0 : step == 1 ? a.u_o : a.u_f1);
        const int per = step == 0 ? a.g_qkv : step == 1 ? a.g_o : a.g_f1;
        const int ls = step == 0 ? a.s_qkv : step == 1 ? a.s_o : a.s_f1;
        const int panel = rel / per;
        int grp = rel - panel * per;
        const int grp0 = grp;
        LfLinear l = a.q;
        f16 *Y = const_cast<f16 *>(a.at.Q);
        if (step == 0) {
            if (grp >= a.gl_q + a.gl_k) {
                l = a.v;
                Y = const_cast<f16 *>(a.at.V);
                grp -= a.gl_q + a.gl_k;
            } else if (grp >= a.gl_q) {
                l = a.k;
                Y = const_cast<f16 *>(a.at.K);
                grp -= a.gl_q;
            }
        } else if (step == 1) {
            l = a.o;
            Y = a.oraw;
        } else {
            l = a.m1;
            Y = a.hid;
        }
        const int m0 = panel * LF_BM;
        const int br = LF_WAVES >> ls, j = wave & (br - 1), sub = wave / br;
        const int bn = grp * br + j;
        if (step == 0)
            lf_panel(a, a.in, xs, ldx, m0, wave, lane);
        LfWalk w = lf_walk(l, bn, sub, ls, lane);
        const f16x4 bias = lf_bias(l, bn, lane);
        LfPairs<LF_D> p;
        const int n = lf_request(p, l, w, lane_w2, hi4);
        if (step == 0) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        } else if (step == 1) {
            // the attention blocks that hold this panel's rows
            const int b0 = a.blk[2 * a.nblk + 2 * panel], b1 = a.blk[2 * a.nblk + 2 * panel + 1];
            lf_wait(a, ctr, wave, c_at + b0, b1 - b0 + 1, (unsigned)a.at.nhead);
            lf_panel(a, a.at.out, xs, ldx, m0, wave, lane);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        } else {
            const LfPieces skip = lf_pieces(a, lf_row(a, a.in, m0 + wave), lane), gamma = lf_pieces(a, a.gamma1, lane),
                           beta = lf_pieces(a, a.beta1, lane);
            lf_wait(a, ctr, wave, c_o + panel, 1, (unsigned)a.g_o);
            const LfPieces v = lf_layernorm(a, lf_pieces(a, lf_row(a, a.oraw, m0 + wave), lane), skip, gamma, beta, lane);
            lf_put_row(a, xs + wave * ldx, v, lane);
            // (the skip operand of the second LayerNorm)
            if (!a.again && grp0 == 0 && m0 + wave < a.M)
#pragma unroll
                for (int i = 0; i < 2; i++)
                    if (lane + 64 * i < a.d >> 3)
                        store_agent8(a.ln1 + (size_t)(m0 + wave) * a.d + (lane + 64 * i) * 8, v.p[i]);
        }
        lf_barrier();
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        lf_multiply(acc, p, n, l, w, xlane, lane_w2, hi4);
        if (step == 2)
            lf_finish<true>(a, acc, red, l, bias, Y, l.nbr * 16, bn, j, sub, ls, m0, lane);
        else
            lf_finish<false>(a, acc, red, l, bias, Y, l.nbr * 16, bn, j, sub, ls, m0, lane);
        (void)lf_signal(ctr, (step == 0 ? c_qkv : step == 1 ? c_o : c_f1) + panel);
    } else if (unit < a.u_o) {
        // ---- attention: block of query rows of one head
        const int rel = unit - a.u_at;
        const int ib = rel / a.at.nhead, h = rel - ib * a.at.nhead;
        const int b = a.blk[2 * ib], qb = a.blk[2 * ib + 1];
        if constexpr (FUSED) { // ... and its projections
            qkv_attention_block<LF_WAVES, LF_HEAD_PAIRS, MASK, true>(a.qa, b, h);
        } else {
            const int row0 = a.at.cu_seqlens ? a.at.cu_seqlens[b] : b * a.at.seq_len;
            const int row1 = a.at.cu_seqlens ? a.at.cu_seqlens[b + 1] : row0 + a.at.seq_len;
            const int p0 = row0 / LF_BM, p1 = (row1 - 1) / LF_BM;
            lf_wait(a, ctr, wave, c_qkv + p0, p1 - p0 + 1, (unsigned)a.g_qkv);
            attention_block<HD, 1, LF_WAVES, false, false, false, HD, false, true, MASK>(a.at, b, h, qb);
        }
        (void)lf_signal(ctr, c_at + ib);
    } else {
        // ---- second feed-forward linear; whoever completes a panel runs its LayerNorm
        const int rel = unit - a.u_f2;
        const int panel = rel / a.g_f2, grp = rel - panel * a.g_f2;
        const int m0 = panel * LF_BM, ls = a.s_f2;
        const int br = LF_WAVES >> ls, j = wave & (br - 1), sub = wave / br;
        const int bn = grp * br + j;
        LfWalk w = lf_walk(a.m2, bn, sub, ls, lane);
        const f16x4 bias = lf_bias(a.m2, bn, lane);
        LfPairs<LF_D> p;
        const int n = lf_request(p, a.m2, w, lane_w2, hi4);
        // The skip operand of the second LayerNorm is the first one's rows, which the linear before stores - and is held up
        // by it.  Where every unit has a CU of its own from the start, this one computes them again while it waits.
        f16 *const midrow = xs + LF_WAVES * 64 * 8 + wave * a.d; // (behind the partial sums)
        if (a.again) {
            const LfPieces skip = lf_pieces(a, lf_row(a, a.in, m0 + wave), lane), gamma = lf_pieces(a, a.gamma1, lane),
                           beta = lf_pieces(a, a.beta1, lane);
            lf_wait(a, ctr, wave, c_o + panel, 1, (unsigned)a.g_o);
            const LfPieces v = lf_layernorm(a, lf_pieces(a, lf_row(a, a.oraw, m0 + wave), lane), skip, gamma, beta, lane);
            lf_put_row(a, midrow, v, lane);
        }
        lf_wait(a, ctr, wave, c_f1 + panel, 1, (unsigned)a.g_f1);
        const char *xr = reinterpret_cast<const char *>(a.hid + (size_t)min(m0 + c16, a.M - 1) * a.dff + khalf8);
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        lf_multiply_direct(acc, p, n, a.m2, w, xr, lane_w2, hi4);
        lf_finish<false>(a, acc, red, a.m2, bias, a.fraw, a.d, bn, j, sub, ls, m0, lane);
        const unsigned old = lf_signal(ctr, c_f2 + panel);
        if (threadIdx.x == 0)
            bc[1] = old;
        lf_barrier();
        if ((int)bc[1] != a.g_f2 - 1)
            return;
        // every unit of every earlier step of this panel is done; if this is the last panel, of the launch
        if (threadIdx.x == 0)
            bc[2] = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        {
            const LfPieces y = lf_pieces(a, lf_row(a, a.fraw, m0 + wave), lane),
                           skip = lf_pieces(a, a.again ? midrow : lf_row(a, a.ln1, m0 + wave), lane),
                           gamma = lf_pieces(a, a.gamma2, lane), beta = lf_pieces(a, a.beta2, lane);
            const LfPieces v = lf_layernorm(a, y, skip, gamma, beta, lane);
            if (m0 + wave < a.M)
                lf_put_row(a, a.out + (size_t)(m0 + wave) * a.d, v, lane);
        }
        lf_barrier();
        if ((int)bc[2] == a.npanel - 1) {
            unsigned *const other = a.ctr + (size_t)(1 + (set ^ 1) * a.nctr) * LF_CS;
            for (int i = threadIdx.x; i < a.nctr; i += LF_WAVES * 64)
                __hip_atomic_store(other + (size_t)i * LF_CS, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (threadIdx.x == 0)
                __hip_atomic_store(a.ctr, (unsigned)(set ^ 1) << 31, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// ---- host side --------------------------------------------------------------
static int g_flow_rows = -1; // et_tuning_set("layer_flow_rows"): rows up to which a layer runs as one launch, -1 automatic
void set_flow_rows(int v) { g_flow_rows = v; }
bool tail_tuned();

// Automatic choice.  With projections and attention as one unit: while there is about one unit per CU - then all of them
// request their weights at once; a second round of units costs what a launch does.  One launch against the separate ones
// (five to seven), us, 80 % pruned, sequences x rows (units): 768 wide 1 x 16 (51) 18.9 / 23.8, 1 x 37 (129) 21.1 / 25.0, 1 x 64
// (168) 22.8 / 26.1, 1 x 96 (246) 24.9 / 28.4, 3 x 32 (270) 24.7 / 24.6, 1 x 112 (285) 30.9 / 29.5, 8 x 16 (408) 24.9 / 24.1; 512
// wide 2 x 64 (224) 20.0 / 24.5, 1 x 128 (216) 23.9 / 29.0, 8 x 16 (272) 21.0 / 24.3; 1024 wide 1 x 64 (224) 24.5 / 27.6, 6 x 10
// (304) 25.9 / 24.9.  Else up to 96 rows, and up to 30 MB of W in all (every 16-row panel streams the layer's tiles once),
// where the separate launches do not have projections and attention in one either: 768 wide, 50 % pruned 1 x 37 27.4 / 29.5,
// 1 x 64 29.9 / 29.4; with them 2 x 32 29.5 / 27.0.
constexpr int LF_MOST_ROWS = 96;
constexpr double LF_MOST_MB = 30.0;
constexpr int LF_MOST_ROOM = 160; // rows of a layer that an object is made for: what fits the units of a narrow one
constexpr int LF_MAX_ROWS = 2048; // (forced by the tuning key)
static int flow_rows_limit() { return g_flow_rows < 0 ? LF_MOST_ROOM : std::min(g_flow_rows, LF_MAX_ROWS); }
} // namespace et

struct et_layer_flow {
    const et_tile_plan *p[6] = {};
    int d = 0, dff = 0, seq_len = 0, nheads = 0, batch = 0;
    et::f16 *scratch = nullptr; // Q, K, V, attention, oraw, ln1, fraw: rows x d; hid: rows x dff
    unsigned *ctr = nullptr;
    int nctr = 0; // counters in a set: enough for the padded batch and for any lengths
    int *d_blk[2] = {nullptr, nullptr}; // padded batch, packed sequences
    double mbytes = 0.0; // of surviving tiles in the six linears
    int nblk[2] = {0, 0}, rows[2] = {0, 0};
    bool packed = false; // et_layer_flow_set_packed has been called
    bool fused = false;  // a head's projections and attention are one unit
    int s_qkv = 0, s_o = 0, s_f1 = 0, s_f2 = 0;                   // log2 of the splits
    int gl_q = 0, gl_k = 0, g_qkv = 0, g_o = 0, g_f1 = 0, g_f2 = 0; // units per panel (fused: none of Q/K/V)
    int units(int which) const { return npanel(which) * (g_qkv + g_o + g_f1 + g_f2) + nblk[which] * nheads; }
    int npanel(int which) const { return (rows[which] + et::LF_BM - 1) / et::LF_BM; }
};

namespace et {
// attention blocks of sequences with these row ranges, and the blocks that hold each panel's rows
static int flow_tables(et_layer_flow *f, int which, const int *cu, int batch) {
    std::vector<int> blk, first_row;
    const int rows = cu[batch];
    for (int b = 0; b < batch; b++)
        for (int q = 0; cu[b] + q * LF_QB < cu[b + 1]; q++) {
            blk.push_back(b);
            blk.push_back(q);
            first_row.push_back(cu[b] + q * LF_QB);
        }
    const int n = (int)first_row.size(), npanel = (rows + LF_BM - 1) / LF_BM;
    for (int p = 0, i = 0; p < npanel; p++) {
        const int m0 = p * LF_BM, m1 = std::min(m0 + LF_BM, rows) - 1;
        while (i + 1 < n && first_row[i + 1] <= m0)
            i++;
        int k = i;
        while (k + 1 < n && first_row[k + 1] <= m1)
            k++;
        blk.push_back(i);
        blk.push_back(k);
    }
    f->nblk[which] = n;
    f->rows[which] = rows;
    if (blk.empty())
        return ET_OK;
    return et_memcpy_h2d(f->d_blk[which], blk.data(), blk.size() * sizeof(int));
}

static int flow_split(const et_tile_plan *p, int most) {
    // pairs per block-row (every chunk's run is padded to a whole pair); a wave's share fits its registers
    const int pairs = (p->ntile / std::max(p->out_feat / 16, 1) + p->nchunk + 1) / 2;
    int ls = 0;
    while (ls < 4 && (pairs >> ls) > most)
        ls++;
    return ls;
}
} // namespace et

extern "C" int et_layer_flow_create(et_layer_flow **flow, const et_tile_plan *q, const et_tile_plan *k,
                                    const et_tile_plan *v, const et_tile_plan *o, const et_tile_plan *m1,
                                    const et_tile_plan *m2, int seq_len, int nheads, int batch) {
    using namespace et;
    ET_REQUIRE(flow && q && k && v && o && m1 && m2, ET_ERR_INVALID_ARG, "et_layer_flow_create: null pointer");
    *flow = nullptr;
    const int d = o->out_feat, dff = m1->out_feat;
    const long rows = (long)seq_len * batch;
    if (seq_len <= 0 || batch <= 0 || nheads <= 0 || rows > flow_rows_limit())
        return ET_OK; // (too many rows: the caller runs the steps one by one)
    const int hd = d / nheads;
    // whole 128-byte lines per row, rows within two 16-byte pieces per lane, a panel within half of the LDS
    const bool shapes = d % 64 == 0 && dff % 64 == 0 && d <= 1024 && d % nheads == 0 && (hd == 32 || hd == 64) &&
                        q->in_feat == d && k->in_feat == d && v->in_feat == d && q->out_feat == d && k->out_feat == d &&
                        v->out_feat == d && o->in_feat == d && m1->in_feat == d && m2->in_feat == dff &&
                        m2->out_feat == d && m2->nchunk <= LF_MAX_CHUNK;
    if (!shapes)
        return ET_OK;
    et_layer_flow *f = new et_layer_flow();
    const et_tile_plan *ps[6] = {q, k, v, o, m1, m2};
    for (int i = 0; i < 6; i++) {
        f->p[i] = ps[i];
        f->mbytes += ps[i]->ntile * 512e-6;
    }
    f->fused = qa_shapes(q, k, v, seq_len, d, nheads, LF_HEAD_PAIRS);
    auto groups = [](const et_tile_plan *p, int s) {
        const int br = LF_WAVES >> s;
        return (p->out_feat / 16 + br - 1) / br;
    };
    if (!f->fused) {
        f->s_qkv = std::max(std::max(flow_split(q, LF_SHARE), flow_split(k, LF_SHARE)), flow_split(v, LF_SHARE));
        f->gl_q = groups(q, f->s_qkv);
        f->gl_k = groups(k, f->s_qkv);
        f->g_qkv = f->gl_q + f->gl_k + groups(v, f->s_qkv);
    }
    f->s_o = flow_split(o, LF_SHARE);
    f->s_f1 = flow_split(m1, LF_SHARE);
    f->s_f2 = 3;
    f->g_o = groups(o, f->s_o);
    f->g_f1 = groups(m1, f->s_f1);
    f->g_f2 = groups(m2, f->s_f2);
    f->d = d;
    f->dff = dff;
    f->seq_len = seq_len;
    f->nheads = nheads;
    f->batch = batch;
    const int npanel = (int)((rows + LF_BM - 1) / LF_BM);
    const int nblk = batch * ((seq_len + LF_QB - 1) / LF_QB);
    f->nctr = 1 + 4 * npanel + nblk;
    const size_t act = (size_t)rows * (7 * (size_t)d + dff) * sizeof(f16);
    const size_t ctr = (size_t)(1 + 2 * f->nctr) * LF_CS * sizeof(unsigned);
    const size_t tab = ((size_t)2 * nblk + 2 * npanel) * sizeof(int);
    // one allocation: activations, counters, the two block tables
    char *base = nullptr;
    auto up = [](size_t n) { return (n + 255) / 256 * 256; };
    int rc = et_malloc(reinterpret_cast<void **>(&base), up(act) + up(ctr) + 2 * up(tab));
    if (rc != ET_OK) {
        delete f;
        return rc;
    }
    f->scratch = reinterpret_cast<f16 *>(base);
    f->ctr = reinterpret_cast<unsigned *>(base + up(act));
    f->d_blk[0] = reinterpret_cast<int *>(base + up(act) + up(ctr));
    f->d_blk[1] = reinterpret_cast<int *>(base + up(act) + up(ctr) + up(tab));
    (void)wait_status_device(); // (allocated here rather than inside a run)
    rc = et_fill_zero(f->ctr, up(ctr), nullptr);
    if (rc == ET_OK)
        rc = et_device_synchronize();
    if (rc == ET_OK) {
        std::vector<int> cu(batch + 1);
        for (int b = 0; b <= batch; b++)
            cu[b] = b * seq_len;
        rc = flow_tables(f, 0, cu.data(), batch);
    }
    if (rc != ET_OK) {
        et_layer_flow_destroy(f);
        return rc;
    }
    *flow = f;
    return ET_OK;
}

extern "C" void et_layer_flow_destroy(et_layer_flow *f) {
    if (!f)
        return;
    et_free(f->scratch);
    delete f;
}

extern "C" int et_layer_flow_set_packed(et_layer_flow *f, const int *cu) {
    using namespace et;
    ET_REQUIRE(f && cu, ET_ERR_INVALID_ARG, "et_layer_flow_set_packed: null pointer");
    // (scratch, counters and tables are sized for the padded batch)
    ET_REQUIRE(cu[0] == 0, ET_ERR_INVALID_ARG, "et_layer_flow_set_packed: the first row is %d", cu[0]);
    for (int b = 0; b < f->batch; b++)
        ET_REQUIRE(cu[b + 1] >= cu[b] && cu[b + 1] - cu[b] <= f->seq_len, ET_ERR_INVALID_ARG,
                   "et_layer_flow_set_packed: sequence %d has %d rows of at most %d", b, cu[b + 1] - cu[b], f->seq_len);
    const int rc = flow_tables(f, 1, cu, f->batch);
    f->packed = rc == ET_OK;
    return rc;
}

extern "C" int et_layer_flow_pays(const et_layer_flow *f, int rows) {
    using namespace et;
    if (!f || rows <= 0 || rows > flow_rows_limit() || tail_pair_enabled() || tail_tuned())
        return 0;
    if (g_flow_rows >= 0)
        return 1;
    const int which = f->packed && rows == f->rows[1] ? 1 : 0, cus = std::max(et_device_cu_count(), 1);
    if (f->fused)
        return rows <= f->rows[which] && f->units(which) <= cus + cus / 16;
    return rows <= LF_MOST_ROWS && (rows + LF_BM - 1) / LF_BM * f->mbytes <= LF_MOST_MB &&
           !et_qkv_attention_pays(f->p[0], f->p[1], f->p[2], f->seq_len, f->d, f->nheads, f->batch);
}

extern "C" int et_layer_flow_run(et_layer_flow *f, void *out, const void *in, void *Q, void *K, void *V, void *attn,
                                 const void *mask, const int *seq_lens, const int *cu_seqlens, const void *gamma1,
                                 const void *beta1, const void *gamma2, const void *beta2, float log2_scale,
                                 void *stream) {
    using namespace et;
    ET_REQUIRE(f && out && in && Q && K && V && attn && gamma1 && beta1 && gamma2 && beta2, ET_ERR_INVALID_ARG,
               "et_layer_flow_run: null pointer");
    ET_REQUIRE(aligned16(out) && aligned16(in) && aligned16(Q) && aligned16(K) && aligned16(V) && aligned16(attn) &&
                   aligned16(gamma1) && aligned16(beta1) && aligned16(gamma2) && aligned16(beta2),
               ET_ERR_ALIGNMENT, "et_layer_flow_run: pointers must be 16-byte aligned");
    const int which = cu_seqlens ? 1 : 0;
    ET_REQUIRE(!which || f->packed, ET_ERR_INVALID_ARG, "et_layer_flow_run: cu_seqlens without et_layer_flow_set_packed");
    LfArgs a;
    memset(&a, 0, sizeof(a));
    a.M = f->rows[which];
    if (a.M == 0)
        return ET_OK;
    {
        const int rc = check_wait_status("layer in one launch");
        if (rc != ET_OK)
            return rc;
    }
    a.status = wait_status_device();
    ET_REQUIRE(a.status, ET_ERR_HIP, "layer in one launch: no wait-status word");
    a.spin = tail_spin();
    const size_t unit = (size_t)f->seq_len * f->batch * f->d;
    a.at.Q = f->scratch;
    a.at.K = f->scratch + unit;
    a.at.V = f->scratch + 2 * unit;
    a.at.out = f->scratch + 3 * unit;
    a.oraw = f->scratch + 4 * unit;
    a.ln1 = f->scratch + 5 * unit;
    a.fraw = f->scratch + 6 * unit;
    a.hid = f->scratch + 7 * unit;
    a.at.mask = static_cast<const f16 *>(mask);
    a.at.seq_lens = cu_seqlens ? nullptr : seq_lens;
    a.at.cu_seqlens = cu_seqlens;
    a.at.ldq = a.at.ldv = f->d;
    a.at.seq_len = f->seq_len;
    a.at.nhead = f->nheads;
    a.at.batch = f->batch;
    a.at.log2_scale = log2_scale;
    if (attention_finish_args(a.at, f->d))
        a.at.mask = nullptr; // (zero everywhere: adds nothing)
    LfLinear *ls[6] = {&a.q, &a.k, &a.v, &a.o, &a.m1, &a.m2};
    for (int i = 0; i < 6; i++) {
        const et_tile_plan *p = f->p[i];
        ls[i]->data = p->d_data;
        ls[i]->cptr = p->d_cptr;
        ls[i]->poff = p->d_row_offset;
        ls[i]->bias = p->d_bias;
        ls[i]->nbr = p->out_feat / 16;
        ls[i]->nchunk = p->nchunk;
        ls[i]->kc2 = p->KC * 2;
        ls[i]->spare = p->npair;
    }
    a.in = static_cast<const f16 *>(in);
    a.out = static_cast<f16 *>(out);
    a.gamma1 = static_cast<const f16 *>(gamma1);
    a.beta1 = static_cast<const f16 *>(beta1);
    a.gamma2 = static_cast<const f16 *>(gamma2);
    a.beta2 = static_cast<const f16 *>(beta2);
    a.ctr = f->ctr;
    a.blk = f->d_blk[which];
    a.d = f->d;
    a.inv_d = 1.0f / (float)f->d;
    a.dff = f->dff;
    a.npanel = f->npanel(which);
    a.nblk = f->nblk[which];
    a.nctr = f->nctr;
    a.s_qkv = f->s_qkv;
    a.s_o = f->s_o;
    a.s_f1 = f->s_f1;
    a.s_f2 = f->s_f2;
    a.gl_q = f->gl_q;
    a.gl_k = f->gl_k;
    a.g_qkv = f->g_qkv;
    a.g_o = f->g_o;
    a.g_f1 = f->g_f1;
    a.g_f2 = f->g_f2;
    const bool fused = f->fused;
    a.u_at = a.npanel * a.g_qkv;
    a.u_o = a.u_at + a.nblk * f->nheads;
    a.u_f1 = a.u_o + a.npanel * a.g_o;
    a.u_f2 = a.u_f1 + a.npanel * a.g_f1;
    const int total = a.u_f2 + a.npanel * a.g_f2;
    a.again = total <= std::max(et_device_cu_count(), 1);
    const bool wide = f->d / f->nheads == 64;
    const size_t lds_at = wide ? attn_lds_bytes<64, 1, LF_WAVES, false>() : attn_lds_bytes<32, 1, LF_WAVES, false>();
    const size_t lds_x = (size_t)LF_BM * (f->d + 16) * sizeof(f16);
    size_t lds_head = 0;
    if (fused) {
        qa_operands(a.qa, f->p[0], f->p[1], f->p[2], f->seq_len, f->d, 160 * 1024 - 64);
        a.qa.X = a.in;
        a.qa.mask = a.at.mask;
        a.qa.out = a.at.out;
        a.qa.seq_lens = a.at.seq_lens;
        a.qa.cu_seqlens = a.at.cu_seqlens;
        a.qa.seq_len = f->seq_len;
        a.qa.nhead = f->nheads;
        a.qa.batch = f->batch;
        a.qa.log2_scale = log2_scale;
        a.qa.scale = a.at.scale;
        lds_head = qa_lds(a.qa.ring, f->d, f->seq_len);
    }
    a.misc = (int)std::max(std::max(fused ? lds_head : lds_at, lds_x), (size_t)LF_WAVES * 64 * sizeof(f32x4) + (size_t)LF_BM * f->d * sizeof(f16));
    const size_t lds = a.misc + 64;
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto launch = [&](auto hd_c, auto mask_c, auto fused_c) -> int {
        constexpr auto kern = &layer_flow_kernel<decltype(hd_c)::value, decltype(mask_c)::value, decltype(fused_c)::value>;
        launch_kernel<kern>(dim3(total), dim3(LF_WAVES * 64), lds, st, a);
        return launch_status("layer in one launch");
    };
    typedef std::integral_constant<int, 64> wide_t;
    typedef std::integral_constant<int, 32> narrow_t;
    if (fused)
        return a.at.mask ? launch(wide_t(), std::true_type(), std::true_type()) : launch(wide_t(), std::false_type(), std::true_type());
    if (wide)
        return a.at.mask ? launch(wide_t(), std::true_type(), std::false_type()) : launch(wide_t(), std::false_type(), std::false_type());
    return a.at.mask ? launch(narrow_t(), std::true_type(), std::false_type()) : launch(narrow_t(), std::false_type(), std::false_type());
}

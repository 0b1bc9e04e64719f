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
// rows (one hand-over less).  Attention: attention_block, 256 query rows per
// unit and head.
#include "attention_block.h"
#include "tile_plan.h"
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

struct LfArgs {
    AttnArgs at; // Q, K, V, out: scratch that the steps hand over
    LfLinear q, k, v, o, m1, m2;
    const f16 *in;
    f16 *out;
    f16 *oraw, *ln1, *hid, *fraw; // output projection, first LayerNorm, hidden activations, second linear
    const f16 *gamma1, *beta1, *gamma2, *beta2;
    unsigned *ctr;  // tickets and the set in turn, then the two sets of nctr counters
    const int *blk; // attention blocks: [2i] sequence, [2i+1] query block; then per panel first and last block
    int M, d, dff, npanel, nblk;
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

// LayerNorm(y + skip) of one row, spread over the wave in 16-byte pieces (the math and the order of summation of
// skip_layernorm.hip).  Every load is requested before the first value is used.  put(piece, values).
template <class Put>
__device__ __forceinline__ void lf_layernorm(const LfArgs &a, const f16 *Y, const f16 *S, const f16 *gamma,
                                             const f16 *beta, int row, int lane, Put &&put) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const int npiece = a.d >> 3;
    const float inv_n = 1.0f / (float)a.d;
    const size_t at = (size_t)min(row, a.M - 1) * a.d;
    f16x8 x[2], s[2], g[2], b[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int pc = min(lane + 64 * i, npiece - 1) * 8;
        x[i] = *reinterpret_cast<const f16x8 *>(Y + at + pc);
        s[i] = *reinterpret_cast<const f16x8 *>(S + at + pc);
        g[i] = *reinterpret_cast<const f16x8 *>(gamma + pc);
        b[i] = *reinterpret_cast<const f16x8 *>(beta + pc);
    }
    __builtin_amdgcn_sched_barrier(0);
    float sum = 0.f, var = 0.f;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        x[i] += s[i]; // half add, one rounding
        if (lane + 64 * i >= npiece)
            x[i] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 8; j += 2)
            sum = __builtin_amdgcn_fdot2(h2{x[i][j], x[i][j + 1]}, h2{(f16)1, (f16)1}, sum, false);
    }
    const float mean = wave_sum(sum) * inv_n;
#pragma unroll
    for (int i = 0; i < 2; i++)
        if (lane + 64 * i < npiece) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float d = (float)x[i][j] - mean;
                var += d * d;
            }
        }
    const float rstd = rsqrtf(wave_sum(var) * inv_n + 1e-6f);
    const float shift = -mean * rstd;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        f16x8 o;
#pragma unroll
        for (int j = 0; j < 8; j++)
            o[j] = (f16)(__builtin_fmaf((float)x[i][j], rstd, shift) * (float)g[i][j] + (float)b[i][j]);
        if (lane + 64 * i < npiece)
            put(lane + 64 * i, o);
    }
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

template <int HD, bool MASK>
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

    if (unit < a.u_at || (unit >= a.u_o && unit < a.u_f2)) {
        // ---- a linear on a panel in LDS: Q/K/V, output projection, first feed-forward linear
        const int step = unit < a.u_at ? 0 : unit < a.u_f1 ? 1 : 2;
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
            lf_wait(a, ctr, wave, c_o + panel, 1, (unsigned)a.g_o);
            lf_layernorm(a, a.oraw, a.in, a.gamma1, a.beta1, m0 + wave, lane, [&](int piece, f16x8 v) {
                *reinterpret_cast<f16x8 *>(xs + wave * ldx + piece * 8) = v;
                if (grp0 == 0 && m0 + wave < a.M) // the skip operand of the second LayerNorm
                    store_agent8(a.ln1 + (size_t)(m0 + wave) * a.d + piece * 8, v);
            });
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
        const int row0 = a.at.cu_seqlens ? a.at.cu_seqlens[b] : b * a.at.seq_len;
        const int row1 = a.at.cu_seqlens ? a.at.cu_seqlens[b + 1] : row0 + a.at.seq_len;
        const int p0 = row0 / LF_BM, p1 = (row1 - 1) / LF_BM;
        lf_wait(a, ctr, wave, c_qkv + p0, p1 - p0 + 1, (unsigned)a.g_qkv);
        attention_block<HD, 1, LF_WAVES, false, false, false, HD, false, true, MASK>(a.at, b, h, qb);
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
        lf_layernorm(a, a.fraw, a.ln1, a.gamma2, a.beta2, m0 + wave, lane, [&](int piece, f16x8 v) {
            if (m0 + wave < a.M)
                *reinterpret_cast<f16x8 *>(a.out + (size_t)(m0 + wave) * a.d + piece * 8) = v;
        });
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

// Automatic choice: up to 96 rows, and up to 30 MB of W in all (every 16-row panel streams the layer's tiles once).
// One launch against seven, us, rows 37 / 64 / 96 / 128: 768 wide, 80 % pruned 25.2 / 25.5 / 29.7 / 33.3 against
// 30.3 / 30.2 / 30.9 / 30.6; 50 % 27.9 / 31.2 / 33.0 against 32.2 / 32.4 / 34.0; dense 34.5 / 38.8 against
// 35.1 / 35.4; 512 wide, 80 % 22.4 / 22.9 / 25.0 / 27.8 against 30.
constexpr int LF_MOST_ROWS = 96;
constexpr double LF_MOST_MB = 30.0;
constexpr int LF_MAX_ROWS = 2048; // (forced by the tuning key)
static int flow_rows_limit() { return g_flow_rows < 0 ? LF_MOST_ROWS : std::min(g_flow_rows, LF_MAX_ROWS); }
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
    return g_flow_rows >= 0 || (rows + LF_BM - 1) / LF_BM * f->mbytes <= LF_MOST_MB ? 1 : 0;
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
    a.dff = f->dff;
    a.npanel = (a.M + LF_BM - 1) / LF_BM;
    a.nblk = f->nblk[which];
    a.nctr = f->nctr;
    a.s_qkv = std::max(std::max(flow_split(f->p[0], LF_SHARE), flow_split(f->p[1], LF_SHARE)), flow_split(f->p[2], LF_SHARE));
    a.s_o = flow_split(f->p[3], LF_SHARE);
    a.s_f1 = flow_split(f->p[4], LF_SHARE);
    a.s_f2 = 3;
    auto groups = [](const et_tile_plan *p, int s) {
        const int br = LF_WAVES >> s;
        return (p->out_feat / 16 + br - 1) / br;
    };
    a.gl_q = groups(f->p[0], a.s_qkv);
    a.gl_k = groups(f->p[1], a.s_qkv);
    a.g_qkv = a.gl_q + a.gl_k + groups(f->p[2], a.s_qkv);
    a.g_o = groups(f->p[3], a.s_o);
    a.g_f1 = groups(f->p[4], a.s_f1);
    a.g_f2 = groups(f->p[5], a.s_f2);
    a.u_at = a.npanel * a.g_qkv;
    a.u_o = a.u_at + a.nblk * f->nheads;
    a.u_f1 = a.u_o + a.npanel * a.g_o;
    a.u_f2 = a.u_f1 + a.npanel * a.g_f1;
    const int total = a.u_f2 + a.npanel * a.g_f2;
    const bool wide = f->d / f->nheads == 64;
    const size_t lds_at = wide ? attn_lds_bytes<64, 1, LF_WAVES, false>() : attn_lds_bytes<32, 1, LF_WAVES, false>();
    const size_t lds_x = (size_t)LF_BM * (f->d + 16) * sizeof(f16);
    a.misc = (int)std::max(std::max(lds_at, lds_x), (size_t)LF_WAVES * 64 * sizeof(f32x4));
    const size_t lds = a.misc + 64;
    hipStream_t st = static_cast<hipStream_t>(stream);
    static_assert(attn_lds_bytes<64, 1, LF_WAVES, false>() + 64 <= 64 * 1024 && LF_BM * (1024 + 16) * 2 + 64 <= 64 * 1024,
                  "no opt-in for dynamic LDS needed");
    const auto kern = wide ? (a.at.mask ? layer_flow_kernel<64, true> : layer_flow_kernel<64, false>)
                           : (a.at.mask ? layer_flow_kernel<32, true> : layer_flow_kernel<32, false>);
    hipLaunchKernelGGL(kern, dim3(total), dim3(LF_WAVES * 64), lds, st, a);
    return launch_status("layer in one launch");
}

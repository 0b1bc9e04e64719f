// Tile-pruned linear on whole rows: a workgroup of 16 waves keeps 16 rows of X
// with ALL of their K columns in LDS (up to 4848 columns) and its waves walk the
// tile lists of their block-rows over them.
//
// Where it is used.  (1) Plans with K in several column chunks, few to a few
// thousand rows: the chunked kernels of tile_linear.hip fetch a chunk, wait,
// multiply, wait, four to six times per work item - a chain of memory round
// trips (BERT-base second feed-forward linear, 80 % pruned: 12-13 us for any
// row count below 1000) - while here the whole panel and the first pairs of
// every wave are requested at once.  (2) The caller's own tile_mat (unsorted,
// odd counts): with the row in LDS the order of the tiles does not matter, and
// the pairs stream through registers instead of one tile after the other
// (1000 rows, 3072 -> 768, 80 %: 34 us before).
// What it costs: W is streamed once per 16 rows (L2 to CU, ~130 GB/s per CU),
// so with many rows and dense lists the 32-row kernels win; the launcher in
// tile_linear.hip chooses by estimated time.
//
// Few rows: the pairs of a block-row are split over 2^ls waves so that a wave's
// share arrives in one or two round trips; the partial sums meet in LDS and are
// added in a fixed order.  More rows than fill the chip: a wave takes several
// block-rows one after the other and the panel is fetched once for all of them.
#include "tile_plan.h"
#include "tile_walk.h"

#include <algorithm>
#include <cstring>

namespace et {

constexpr int TR_WAVES = 16;
constexpr int TR_BM = 16;
constexpr int TR_MAX_LIN = 4;

struct TrArgs {
    LfLinear l[TR_MAX_LIN]; // RAW: cptr = row_ptr, poff = row_offset (element columns), nchunk = 1
    f16 *Y[TR_MAX_LIN];
    const f16 *X;
    int nlin, M, K, ldx, ncg, total, per_xcd, nb, ls;
    int div, by_group; // workgroups of a panel (by_group: of a column group) that consecutive ids take
    unsigned div_magic, ncg_magic;
};

// The caller's list: pair i of a block-row is tiles 2i and 2i + 1, 1 KB of
// consecutive W; `n` of a pair's two tiles exist (the last pair of an odd list
// has one, slots past the end none).
struct TrRawWalk {
    int t, end;
};
typedef LfPairs<LF_D> TrSlots; // co: RAW: tiles in the slot, else byte offset of the column chunk

template <int I>
__device__ __forceinline__ void tr_load_raw(TrSlots &p, const LfLinear &l, TrRawWalk &w, unsigned lane_w2, int hi) {
    const int n = min(max(w.end - w.t, 0), 2);
    const int t = n > 0 ? w.t : w.end - 1; // (an empty slot re-reads the last tile and is multiplied as zero)
    const int h = hi < n ? hi : 0;
    p.co[I] = n;
    p.o[I] = l.poff[t + h] * 2;
    p.w[I] = *reinterpret_cast<const f16x8 *>(reinterpret_cast<const char *>(l.data) + (size_t)t * 512 + lane_w2 -
                                              (hi - h) * 512);
    w.t += n;
}

template <bool GELU, bool RAW>
__global__ void __launch_bounds__(TR_WAVES * 64) tile_rows_kernel(
    // (what comes before the first requests arrives in registers with the wave)
    const f16 *hot_X, const int *hot_cptr, int hot_M, int hot_K, int hot_total, int hot_per_xcd, int hot_div, unsigned hot_div_magic,
    int hot_ncg, unsigned hot_ncg_magic, int hot_form, int hot_nbr, const TrArgs args) {
    TrArgs a = args;
    a.X = hot_X;
    a.M = hot_M;
    a.K = hot_K;
    a.ldx = hot_K + ((hot_K & 31) ? 0 : 16);
    a.total = hot_total;
    a.per_xcd = hot_per_xcd;
    a.div = hot_div;
    a.div_magic = hot_div_magic;
    a.ncg = hot_ncg;
    a.ncg_magic = hot_ncg_magic;
    a.nb = hot_form & 15;
    a.ls = hot_form >> 4 & 15;
    a.by_group = hot_form >> 8;
    extern __shared__ __attribute__((aligned(16))) unsigned char tr_smem[];
    f16 *const xs = reinterpret_cast<f16 *>(tr_smem);
    // (consecutive ids on one XCD: the column groups of a panel, or, by_group, the panels of a column group)
    const int vid = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    if (vid >= a.total)
        return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c16 = lane & 15, g4 = lane >> 4, khalf8 = (g4 & 1) * 8, hi = lane >> 5;
    const unsigned lane_w2 = (unsigned)(hi * 256 + c16 * 16 + khalf8) * 2, hi4 = hi * 4;
    const QuotRem of = quot_rem(vid, a.div, a.div_magic);
    const int panel = a.by_group ? of.r : of.q;
    const QuotRem rest = quot_rem(a.by_group ? of.q : of.r, a.ncg, a.ncg_magic);
    const int lin = rest.q, cg = rest.r;
    const int m0 = panel * TR_BM;
    // the panel: wave w fetches row w, DMA
    if (m0 + wave < a.M) {
        const f16 *src = a.X + (size_t)(m0 + wave) * a.K;
        f16 *dst = xs + wave * a.ldx;
        const int npiece = a.K >> 3;
        for (int c0 = 0; c0 < npiece; c0 += 64)
            if (c0 + lane < npiece)
                load_lds16(src + (c0 + lane) * 8, dst + c0 * 8);
    }
    LfLinear l = a.l[0];
    f16 *Y = a.Y[0];
    l.cptr = hot_cptr;
    l.nbr = hot_nbr;
    if (lin > 0) { // (wave-uniform)
#pragma unroll
        for (int i = 1; i < TR_MAX_LIN; i++)
            if (lin == i) {
                l = a.l[i];
                Y = a.Y[i];
            }
    }
    const int N = l.nbr * 16;
    const int br = TR_WAVES >> a.ls, j = wave & (br - 1), sub = wave / br;

    const char *const xlane = reinterpret_cast<const char *>(xs + c16 * a.ldx + khalf8);
    for (int ib = 0; ib < a.nb; ib++) {
        const int bn = (cg * a.nb + ib) * br + j;
        LfWalk w;
        TrRawWalk rw;
        TrSlots p;
        int n;
        if constexpr (RAW) {
            rw.t = rw.end = 0;
            if (bn < l.nbr) {
                const int t0 = l.cptr[bn], t1 = l.cptr[bn + 1];
                const int pairs = (t1 - t0 + 1) >> 1;
                rw.t = __builtin_amdgcn_readfirstlane(t0 + 2 * ((pairs * sub) >> a.ls));
                rw.end = __builtin_amdgcn_readfirstlane(min(t0 + 2 * ((pairs * (sub + 1)) >> a.ls), t1));
            }
        } else {
            w = lf_walk(l, bn, sub, a.ls, lane);
        }
        auto pairs_left = [&] { return RAW ? (rw.end - rw.t + 1) >> 1 : w.left; };
        auto load = [&](auto ic) {
            constexpr int I = decltype(ic)::value;
            if constexpr (RAW)
                tr_load_raw<I>(p, l, rw, lane_w2, hi);
            else
                lf_load<LF_D, I>(p, l, w, lane_w2, hi4);
        };
        n = min(pairs_left(), LF_D);
        // two pairs at a time; a group is requested as a whole where its first pair exists (wave-uniform)
#define TR_GROUP(i_, cond_)                                                                       \
    if (cond_) {                                                                                  \
        load(std::integral_constant<int, i_>());                                                  \
        load(std::integral_constant<int, i_ + 1>());                                              \
    }
        TR_GROUP(0, n > 0) TR_GROUP(2, n > 2) TR_GROUP(4, n > 4) TR_GROUP(6, n > 6)
        if (ib == 0) {
            __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): pairs and panel
            __syncthreads();
        }
        const f16x4 b4 = *reinterpret_cast<const f16x4 *>(l.bias + min(bn, l.nbr - 1) * 16 + g4 * 4);
        f32x4 acc0 = f32x4{0.f, 0.f, 0.f, 0.f}, acc1 = f32x4{0.f, 0.f, 0.f, 0.f};
        auto multiply = [&](auto ic) {
            constexpr int I = decltype(ic)::value;
            if constexpr (RAW) {
                f16x8 x0 = *reinterpret_cast<const f16x8 *>(xlane + p.o[I]);
                f16x8 x1 = *reinterpret_cast<const f16x8 *>(xlane + p.o[I + 1]);
                f16x8 w0 = p.w[I], w1 = p.w[I + 1];
                const f16x8 zero8 = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
                if (p.co[I] + p.co[I + 1] < 4) { // (wave-uniform: the end of the list)
                    w0 = hi < p.co[I] ? w0 : zero8;
                    x0 = hi < p.co[I] ? x0 : zero8;
                    w1 = hi < p.co[I + 1] ? w1 : zero8;
                    x1 = hi < p.co[I + 1] ? x1 : zero8;
                }
                acc0 = mfma16x16x32(w0, x0, acc0);
                acc1 = mfma16x16x32(w1, x1, acc1);
            } else {
                const f16x8 x0 = *reinterpret_cast<const f16x8 *>(xlane + p.o[I] + p.co[I]);
                const f16x8 x1 = *reinterpret_cast<const f16x8 *>(xlane + p.o[I + 1] + p.co[I + 1]);
                acc0 = mfma16x16x32(p.w[I], x0, acc0);
                acc1 = mfma16x16x32(p.w[I + 1], x1, acc1);
            }
        };
        // Long lists of the caller's own: as long as a round's pairs are all in flight and as many to come, it asks nothing
        // and its waits are counted - a request that may not have gone out makes the compiler wait for all of them, a round
        // trip for every two pairs.  3072 -> 768: 1067 rows 80 % 8.4 -> 7.7 us, 50 % 13.1 -> 12.1, dense 26.8 -> 21.7; 4096
        // rows 20.6 -> 18.6, 43.4 -> 34.8, 74.7 -> 58.9; 4096 -> 1024, 1067 rows, dense 64.5 -> 48.4.  (A plan's lists may
        // step into the next column chunk at every pair, which is a branch again: no faster.)
        if constexpr (RAW) {
            while (n == LF_D && pairs_left() >= LF_D) {
#define TR_ROUND(i_)                                                                              \
    multiply(std::integral_constant<int, i_>());                                                  \
    load(std::integral_constant<int, i_>());                                                      \
    load(std::integral_constant<int, i_ + 1>());
                TR_ROUND(0) TR_ROUND(2) TR_ROUND(4) TR_ROUND(6)
#undef TR_ROUND
            }
        }
        while (n > 0) {
            int m = 0; // pairs in the slots of the next round
#define TR_STEP(i_)                                                                               \
    if (n > i_) {                                                                                 \
        multiply(std::integral_constant<int, i_>());                                              \
        const int more = min(pairs_left(), 2);                                                    \
        m += more;                                                                                \
        TR_GROUP(i_, more > 0)                                                                    \
    }
            TR_STEP(0) TR_STEP(2) TR_STEP(4) TR_STEP(6)
#undef TR_STEP
            n = m;
        }
#undef TR_GROUP
        f32x4 t = acc0 + acc1;
        if (a.ls > 0) { // (one block-row per wave then)
            f32x4 *const red = reinterpret_cast<f32x4 *>(tr_smem);
            __syncthreads(); // every wave has read its operands
            red[(sub * br + j) * 64 + lane] = t;
            __syncthreads();
            if (sub > 0)
                return;
            for (int k = 1; k < (1 << a.ls); k++)
                t += red[(k * br + j) * 64 + lane];
        }
        if (bn < l.nbr) {
            f16x4 o = __builtin_convertvector(t + __builtin_convertvector(b4, f32x4), f16x4);
            if (GELU)
                o = gelu4(o);
            if (m0 + c16 < a.M)
                *reinterpret_cast<f16x4 *>(Y + (size_t)(m0 + c16) * N + bn * 16 + g4 * 4) = o;
        }
    }
}

static size_t tile_rows_lds(int K) {
    const size_t panel = (size_t)TR_BM * (K + ((K & 31) ? 0 : 16)) * sizeof(f16);
    return std::max(panel, (size_t)TR_WAVES * 64 * sizeof(f32x4));
}

// the split and the block-rows per wave with the least estimated time; microseconds.  A round of workgroups costs
// its round trips (about 1.2 us), the panel and its lists at the rate a CU takes them in (130 GB/s); pairs: tile
// pairs per block-row.
static void tile_rows_plan(int M, int K, int nbr_max, int nlin, double pairs, int cus, int *nb, int *ls) {
    const int panels = (M + TR_BM - 1) / TR_BM;
    double best = 1e30;
    for (int s = 0; s <= 4; s++)
        for (int b = 1; b <= (s == 0 ? 4 : 1); b++) {
            const int br = TR_WAVES >> s;
            const int ncg = (nbr_max + br * b - 1) / (br * b);
            const long wgs = (long)panels * ncg * nlin;
            const double share = pairs / (1 << s);
            const double bytes = 32.0 * K + 1024.0 * br * b * pairs / (1 << s) * (1 << s);
            // (a wave walks its pairs eight at a time, at best one round trip of 0.6 us per eight when few waves share
            // the CU)
            const double lat = 1.2 + b * (0.3 + 0.35 * share / LF_D) + (s ? 0.3 : 0.0);
            const double rounds = (double)((wgs + cus - 1) / cus);
            const double t = rounds * (lat + bytes / 130e3);
            if (t < best * 0.999) {
                best = t;
                *nb = b;
                *ls = s;
            }
        }
}

// the launch's time in microseconds; traffic: megabytes that the L2s take in.  Fit to 312 launches (2048 -> 512, 3072 ->
// 768 and 4096 -> 1024, 0 to 90 % pruned, 48 to 16384 rows), 4.5 % off in the mean; 9 % on the 96 launches of a graph that
// bench/linear_forms.py times.
double tile_rows_estimate(int M, int K, int nbr_max, int nlin, double pairs, double w_mb) {
    const int cus = std::max(et_device_cu_count(), 1), panels = (M + TR_BM - 1) / TR_BM;
    int nb = 1, ls = 0;
    tile_rows_plan(M, K, nbr_max, nlin, pairs, cus, &nb, &ls);
    const int group = (TR_WAVES >> ls) * nb, ncg = (nbr_max + group - 1) / group * nlin;
    const long wgs = (long)panels * ncg;
    const double rounds = (double)((wgs + cus - 1) / cus);
    return 1.75 + 0.0514 * tl_traffic_mb(2e-6 * M * K, w_mb, panels, ncg, 2.5) +
           rounds * (0.4525 + 43.3e-5 * K + 1.093e-2 * group * pairs + 1.4 * nb + 0.0825 * std::min(1.0, (double)wgs / cus));
}

bool tile_rows_fits(int K) { return K % 16 == 0 && tile_rows_lds(K) <= 160 * 1024; }

// lins[i].cptr etc.: plan layout, or the caller's row_ptr / row_offset / data for raw
int tile_rows_launch(const LfLinear *lins, f16 *const *Ys, int nlin, const f16 *X, int M, int K, double pairs, bool gelu,
                     bool raw, hipStream_t st) {
    TrArgs a;
    memset(&a, 0, sizeof(a));
    int nbr_max = 0;
    for (int i = 0; i < TR_MAX_LIN; i++) {
        a.l[i] = lins[i < nlin ? i : 0];
        a.Y[i] = Ys[i < nlin ? i : 0];
        nbr_max = std::max(nbr_max, a.l[i].nbr);
    }
    a.X = X;
    a.nlin = nlin;
    a.M = M;
    a.K = K;
    a.ldx = K + ((K & 31) ? 0 : 16); // row stride == 32 (mod 64) bytes: conflict-free
    a.nb = 1;
    tile_rows_plan(M, K, nbr_max, nlin, pairs, std::max(et_device_cu_count(), 1), &a.nb, &a.ls);
    const int per = (TR_WAVES >> a.ls) * a.nb;
    a.ncg = (nbr_max + per - 1) / per;
    const int panels = (M + TR_BM - 1) / TR_BM;
    a.by_group = tl_order(2.0 * M * K, 1024.0 * pairs * nbr_max * nlin, panels, a.ncg * nlin, 2.5e6);
    a.div = a.by_group ? panels : a.ncg * nlin;
    if (!quotients_fit((int64_t)panels * a.ncg * nlin, a.div) || !quotients_fit((int64_t)a.ncg * nlin, a.ncg))
        return ROWS_TOO_MANY;
    a.total = panels * a.ncg * nlin;
    a.per_xcd = (a.total + 7) / 8;
    a.div_magic = magic_of(a.div);
    a.ncg_magic = magic_of(a.ncg);
    const size_t lds = tile_rows_lds(K);
    auto launch = [&](auto gelu_c, auto raw_c) -> int {
        constexpr auto kern = &tile_rows_kernel<decltype(gelu_c)::value, decltype(raw_c)::value>;
        launch_kernel<kern>(dim3(a.per_xcd * 8), dim3(TR_WAVES * 64), lds, st, a.X, a.l[0].cptr, a.M, a.K, a.total, a.per_xcd,
                           a.div, a.div_magic, a.ncg, a.ncg_magic, a.nb | a.ls << 4 | a.by_group << 8, a.l[0].nbr, a);
        return launch_status("tile_linear (whole rows) launch");
    };
    if (raw)
        return gelu ? launch(std::true_type(), std::true_type()) : launch(std::false_type(), std::true_type());
    return gelu ? launch(std::true_type(), std::false_type()) : launch(std::false_type(), std::false_type());
}

} // namespace et

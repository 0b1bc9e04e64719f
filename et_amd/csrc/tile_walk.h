// A wave's share of a block-row's tile pairs, for kernels that hold whole rows of
// the operand (layer_flow.hip, tile_rows.hip): the plan layout keeps the pairs of
// a (column chunk, block-row) in one run, so a block-row is one run per chunk.
#pragma once
#include "common.h"

namespace et {

constexpr int LF_D = 8; // pairs in flight per wave
constexpr int LF_MAX_CHUNK = 16;

struct LfLinear {
    const f16 *data;
    const int *cptr, *poff;
    const f16 *bias;
    int nbr, nchunk, kc2, spare; // kc2: bytes of a column chunk; spare: an all-zero pair
};

// ---- the pairs of a wave ----------------------------------------------------
// A block-row's pairs lie in one run per column chunk; the wave takes part `sub`
// of 2^ls of all of them.  State is wave-uniform.
struct LfWalk {
    int st, en; // lane c: first pair / end of the block-row's run in chunk c
    int c, q, qe, left, coff, kc2, spare;
};
__device__ __forceinline__ LfWalk lf_walk(const LfLinear &l, int bn, int sub, int ls, int lane) {
    LfWalk w;
    w.kc2 = l.kc2;
    w.spare = l.spare;
    w.c = 0;
    w.left = 0;
    w.coff = 0;
    w.q = w.qe = 0;
    w.st = w.en = 0;
    if (bn < l.nbr) {
        const int i = min(lane, l.nchunk - 1) * l.nbr + bn;
        w.st = l.cptr[i] >> 1;
        w.en = l.cptr[i + 1] >> 1;
        int total = 0;
        for (int c = 0; c < l.nchunk; c++)
            total += __builtin_amdgcn_readlane(w.en, c) - __builtin_amdgcn_readlane(w.st, c);
        int skip = (total * sub) >> ls;
        w.left = ((total * (sub + 1)) >> ls) - skip;
        w.q = __builtin_amdgcn_readlane(w.st, 0);
        w.qe = __builtin_amdgcn_readlane(w.en, 0);
        while (w.left > 0 && skip >= w.qe - w.q) {
            skip -= w.qe - w.q;
            w.c++;
            w.q = __builtin_amdgcn_readlane(w.st, w.c);
            w.qe = __builtin_amdgcn_readlane(w.en, w.c);
            w.coff += w.kc2;
        }
        w.q += skip;
    }
    return w;
}
// The next pair, the pair whose columns it is multiplied with and the byte offset of its column chunk.  Where a share is
// odd, the spare pair's zero weights follow, over the columns of the share's last pair: over other columns an infinite
// activation would make NaN of a block-row that has no tile there.  (Leaving the spare pair out of the product instead
// costs a branch per two pairs: 34.3 -> 34.6 us for a dense layer of 128 rows.)  The caller has taken a pair before.
__device__ __forceinline__ void lf_next(LfWalk &w, int &q, int &qcol, int &coff) {
    q = w.spare;
    qcol = w.q - 1;
    coff = w.coff;
    if (w.left > 0) {
        while (w.q >= w.qe) {
            w.c++;
            w.q = __builtin_amdgcn_readlane(w.st, w.c);
            w.qe = __builtin_amdgcn_readlane(w.en, w.c);
            w.coff += w.kc2;
        }
        q = qcol = w.q++;
        coff = w.coff;
        w.left--;
    }
}
template <int D> struct LfPairs {
    f16x8 w[D];
    int o[D], co[D];
};
template <int D, int I>
__device__ __forceinline__ void lf_load(LfPairs<D> &p, const LfLinear &l, LfWalk &w, unsigned lane_w2, unsigned hi4) {
    int q, qcol;
    lf_next(w, q, qcol, p.co[I]);
    p.o[I] = *reinterpret_cast<const int *>(reinterpret_cast<const char *>(l.poff) + (size_t)qcol * 8 + hi4);
    p.w[I] = *reinterpret_cast<const f16x8 *>(reinterpret_cast<const char *>(l.data) + (size_t)q * 1024 + lane_w2);
}
// groups of two pairs, skipped as a whole where the share has ended (wave-uniform)
template <int D>
__device__ __forceinline__ int lf_request(LfPairs<D> &p, const LfLinear &l, LfWalk &w, unsigned lane_w2, unsigned hi4) {
    const int n = min(w.left, D);
#define LF_TWO(i_)                                                                                \
    if (n > i_) {                                                                                 \
        lf_load<D, i_>(p, l, w, lane_w2, hi4);                                                    \
        lf_load<D, i_ + 1>(p, l, w, lane_w2, hi4);                                                \
    }
    LF_TWO(0) LF_TWO(2) LF_TWO(4) LF_TWO(6)
#undef LF_TWO
    static_assert(D == 8, "four groups of two");
    return n;
}

} // namespace et

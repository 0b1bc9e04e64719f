// One workgroup's work in the kernels that project a head's Q, K and V and attend over them without writing any of the
// three (qkv_attention.hip, layer_flow.hip): sequences of up to 128 rows, heads of 64 columns.
//
// Mapping.  A head is four block-rows in each of Q, K and V, a wave each, whose tile pairs stay in registers.  The
// sequence's rows pass in panels of 16 through a ring of up to eight LDS buffers, filled by DMA as far ahead as the ring
// allows; up to 64 rows the whole sequence is requested at once.  The sums (+ bias, rounded to half as the projections store them) go to LDS rows of 80 halves,
// conflict-free for the fragment reads.  Then wave w takes query rows 16w..16w+15: all scores of a row (at most 128) are
// in registers at once, so the softmax is the textbook one - no running maximum.
#pragma once
#include "attention_block.h"
#include "tile_plan.h"

namespace et {

constexpr int QA_LD = 64 + 16; // halves per row of Q, K and V in LDS
constexpr int QA_MOST = 128;   // rows of a sequence
constexpr int QA_RING = 8;     // panels in LDS

struct QaLinear {
    const f16 *data;
    const int *cptr, *poff; // pairs of block-row bn: from cptr[bn] / 2 on; byte offset of a tile's columns
    const f16 *bias;
    int spare; // an all-zero pair
};
struct QaArgs {
    QaLinear l[3];
    const f16 *X, *mask;
    f16 *out;
    const int *seq_lens, *cu_seqlens;
    int d, seq_len, max_len, nhead, batch, ldx;
    int rows32, ring; // LDS rows of Q, K and V each; panels in LDS
    int by_seq; // the heads of a sequence on one XCD
    unsigned nhead_magic;
    float log2_scale, scale;
};

// vmcnt(n) for a number known at run time (wave-uniform)
__device__ __forceinline__ void qa_wait(int n) {
    if (n >= 12)
        __builtin_amdgcn_s_waitcnt(0x0F70 | 12);
    else if (n >= 8)
        __builtin_amdgcn_s_waitcnt(0x0F70 | 8);
    else if (n >= 4)
        __builtin_amdgcn_s_waitcnt(0x0F70 | 4);
    else if (n >= 2)
        __builtin_amdgcn_s_waitcnt(0x0F70 | 2);
    else
        __builtin_amdgcn_s_waitcnt(0x0F70);
}

// NW: 12 waves, of which the first eight also fetch X, or 16, of which the last four fetch.  PAIRS: most tile pairs of a
// block-row.  FLOW: the rows are read by other workgroups of the same launch (store_agent8).
template <int NW, int PAIRS, bool MASK, bool FLOW>
__device__ __forceinline__ void qkv_attention_block(const QaArgs &a, const int b, const int h) {
    static_assert(NW == 12 || NW == 16, "twelve block-rows, a wave each");
    extern __shared__ __attribute__((aligned(16))) unsigned char qa_smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c16 = lane & 15, g4 = lane >> 4, khalf8 = (g4 & 1) * 8, hi = lane >> 5;
    int row0, len, rows_alloc;
    if (a.cu_seqlens) {
        row0 = a.cu_seqlens[b];
        len = rows_alloc = min(max(a.cu_seqlens[b + 1] - row0, 0), a.max_len);
    } else {
        row0 = b * a.seq_len;
        rows_alloc = a.seq_len;
        len = a.seq_lens ? min(max(a.seq_lens[b], 0), a.seq_len) : a.seq_len;
    }
    const int panel = 16 * a.ldx; // halves
    f16 *const xs = reinterpret_cast<f16 *>(qa_smem);
    f16 *const qs = xs + a.ring * panel, *const ks = qs + a.rows32 * QA_LD, *const vs = ks + a.rows32 * QA_LD;
    auto store = [](f16 *p, f16x8 v) {
        if constexpr (FLOW)
            store_agent8(p, v);
        else
            *reinterpret_cast<f16x8 *>(p) = v;
    };
    f16 *const obase = a.out + (size_t)row0 * a.d + h * 64 + g4 * 16;

    if (len > 0) {
        // ---- projections: wave w makes block-row w % 4 of the head in Q, K or V
        const bool makes = NW == 12 || wave < 12;
        const int lin = min(wave >> 2, 2), bn = h * 4 + (wave & 3);
        const QaLinear l = lin == 0 ? a.l[0] : lin == 1 ? a.l[1] : a.l[2];
        typedef const __attribute__((address_space(4))) int *IConst; // (scalar loads)
        const int st = ((IConst)l.cptr)[bn] >> 1, n = makes ? (((IConst)l.cptr)[bn + 1] >> 1) - st : 0;
        const unsigned lane_w2 = (unsigned)(hi * 256 + c16 * 16 + khalf8) * 2;
        const int npiece = a.d >> 3, npanel = (len + 15) >> 4;
        const f16 *const X = a.X + (size_t)row0 * a.d;
        // panel p: the fetching waves take some rows each, one or two requests a row (rows that do not exist re-read the
        // last one: what comes of them is never used)
        constexpr int F0 = NW == 16 ? 12 : 0, FROWS = NW == 16 ? 4 : 2;
        const int per_panel = npiece > 64 ? 2 * FROWS : FROWS;
        auto fetch = [&](int p, int slot) {
            if (wave < F0 || (wave - F0) * FROWS >= 16)
                return;
#pragma unroll
            for (int r = 0; r < FROWS; r++) {
                const int pr = (wave - F0) * FROWS + r;
                const f16 *src = X + (size_t)min(p * 16 + pr, len - 1) * a.d;
                f16 *dst = xs + slot * panel + pr * a.ldx;
                if (lane < npiece)
                    load_lds16_untracked(src, lane * 16, dst);
                if (npiece > 64) // (whole pieces beyond 64 only: the others' lanes are off)
                    if (lane + 64 < npiece)
                        load_lds16_untracked(src, lane * 16 + 1024, dst + 512);
            }
        };
        for (int p = 0; p < min(npanel, a.ring); p++)
            fetch(p, p);
        // the wave's pairs; behind the list's end zero weights over the last pair's columns (other columns may hold an
        // infinity)
        f16x8 w[PAIRS];
        int o[PAIRS];
#pragma unroll
        for (int i = 0; i < PAIRS; i += 2)
            if (n > i) { // (wave-uniform)
#pragma unroll
                for (int j = i; j < i + 2; j++) {
                    const int q = j < n ? st + j : l.spare, qc = st + min(j, n - 1);
                    o[j] = *reinterpret_cast<const int *>(reinterpret_cast<const char *>(l.poff) + (size_t)qc * 8 + hi * 4);
                    w[j] = *reinterpret_cast<const f16x8 *>(reinterpret_cast<const char *>(l.data) + (size_t)q * 1024 + lane_w2);
                }
            }
        const f16x4 bias = *reinterpret_cast<const f16x4 *>(l.bias + bn * 16 + g4 * 4);
        // the wave's mask values (below) come with them
        const int q0 = wave * 16, q = q0 + c16;
        f16x4 mk[QA_MOST / 16];
        if (MASK && q0 < len) {
#pragma unroll
            for (int k = 0; k < QA_MOST / 16; k++)
                if (k * 16 < len) {
                    const int key = k * 16 + g4 * 4;
                    mk[k] = load4_guard(a.mask + (size_t)min(q, a.seq_len - 1) * a.seq_len + key, 0, a.seq_len - key);
                }
        }
        const f32x4 bias4 = __builtin_convertvector(bias, f32x4);
        const char *const xlane = reinterpret_cast<const char *>(xs + c16 * a.ldx + khalf8);
        f16 *const dst = (lin == 0 ? qs : lin == 1 ? ks : vs) + c16 * QA_LD + (wave & 3) * 16 + g4 * 4;
        const bool values = makes && lin == 2; // (they meet probabilities that are zero: rows behind the sequence have to be numbers)

        int slot = 0;
        for (int p = 0; p < npanel; p++) {
            // requests of later panels that may be under way
            qa_wait((min(npanel - 1, max(a.ring - 1, p + a.ring - 2)) - p) * per_panel);
            __syncthreads(); // panel p is there, and everyone is through with panel p-1
            if (p > 0 && p + a.ring - 1 < npanel)
                fetch(p + a.ring - 1, slot == 0 ? a.ring - 1 : slot - 1);
            const char *const xp = xlane + slot * panel * 2;
            f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int i = 0; i < PAIRS; i += 2)
                if (n > i) {
                    const f16x8 x0 = *reinterpret_cast<const f16x8 *>(xp + o[i]);
                    const f16x8 x1 = *reinterpret_cast<const f16x8 *>(xp + o[i + 1]);
                    acc[0] = mfma16x16x32(w[i], x0, acc[0]);
                    acc[1] = mfma16x16x32(w[i + 1], x1, acc[1]);
                }
            f16x4 v = __builtin_convertvector(acc[0] + acc[1] + bias4, f16x4);
            if (values && p * 16 + c16 >= len)
                v = f16x4{0, 0, 0, 0};
            if (makes)
                *reinterpret_cast<f16x4 *>(dst + p * 16 * QA_LD) = v;
            slot = slot + 1 == a.ring ? 0 : slot + 1;
        }
        if (values && (npanel & 1)) // (the second product takes 32 keys at a time)
            *reinterpret_cast<f16x4 *>(dst + npanel * 16 * QA_LD) = f16x4{0, 0, 0, 0};
        __syncthreads();

        // ---- attention of query rows 16 wave .. 16 wave + 15 (the arithmetic of attention_block)
        if (q0 < len) {
            const f16 sc = (f16)a.scale;
            f16x8 qf[2];
#pragma unroll
            for (int s = 0; s < 2; s++)
                qf[s] = *reinterpret_cast<const f16x8 *>(qs + q * QA_LD + s * 32 + g4 * 8) * sc;
            // scores, transposed: s4[k][r] = S[q][key = 16 k + 4 g4 + r]
            f32x4 s4[QA_MOST / 16];
            float mx = -INFINITY;
#pragma unroll
            for (int k = 0; k < QA_MOST / 16; k++)
                if ((k & ~1) * 16 < len) { // (whole 32-key steps)
                    f32x4 t = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < 2; s++) {
                        const f16x8 kf = *reinterpret_cast<const f16x8 *>(ks + (k * 16 + c16) * QA_LD + s * 32 + g4 * 8);
                        t = mfma16x16x32(kf, qf[s], t);
                    }
                    const int key = k * 16 + g4 * 4;
                    if (MASK) {
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            t[r] += (float)mk[k][r];
                    }
                    if (k * 16 + 16 > len) { // (wave-uniform)
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            t[r] = key + r < len ? t[r] : -INFINITY;
                    }
                    mx = fmaxf(fmaxf(mx, t[0]), t[1]);
                    mx = fmaxf(fmaxf(mx, t[2]), t[3]);
                    s4[k] = t;
                }
            mx = xor_max_16_32(mx);
            const float ls = a.log2_scale, m = mx == -INFINITY ? 0.f : mx * ls;
            f32x4 ot[4], la = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int d = 0; d < 4; d++)
                ot[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < QA_MOST / 32; kk++)
                if (kk * 32 < len) {
                    f16x8 pf;
#pragma unroll
                    for (int k = 0; k < 2; k++)
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            pf[k * 4 + r] = (f16)__builtin_amdgcn_exp2f(__builtin_fmaf(s4[2 * kk + k][r], ls, -m));
                    const f16x8 ones8 = f16x8{1, 1, 1, 1, 1, 1, 1, 1};
                    la = mfma16x16x32(ones8, pf, la);
#pragma unroll
                    for (int d = 0; d < 4; d++) {
                        typedef short s16x4 __attribute__((ext_vector_type(4)));
                        typedef __attribute__((address_space(3))) s16x4 *lds4;
                        const f16 *vrow = vs + (kk * 32 + g4 * 4 + (c16 >> 2)) * QA_LD + d * 16 + (c16 & 3) * 4;
                        const f16x4 v0 = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)vrow));
                        const f16x4 v1 = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(vrow + 16 * QA_LD)));
                        ot[d] = mfma16x16x32(f16x8{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]}, pf, ot[d]);
                    }
                }
            const float inv = la[0] > 0.f ? 1.0f / la[0] : 0.f;
            f16x4 o[4];
#pragma unroll
            for (int d = 0; d < 4; d++)
                o[d] = __builtin_convertvector(ot[d] * inv, f16x4);
            transpose_pieces_4x4(o); // the lane's 16 columns are now 16 g4 .. 16 g4 + 15
            if (q < len) {
                f16 *p = obase + (size_t)q * a.d;
                store(p, f16x8{o[0][0], o[0][1], o[0][2], o[0][3], o[1][0], o[1][1], o[1][2], o[1][3]});
                store(p + 8, f16x8{o[2][0], o[2][1], o[2][2], o[2][3], o[3][0], o[3][1], o[3][2], o[3][3]});
            }
        }
    }
    // rows of the padded layout behind the sequence read as zero
    const f16x8 zero8 = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    for (int q = wave * 16 + c16; q < rows_alloc; q += NW * 16)
        if (q >= len) {
            f16 *p = obase + (size_t)q * a.d;
            store(p, zero8);
            store(p + 8, zero8);
        }
}

// LDS bytes with `ring` panels; panels: as many as the sequence has and `most` bytes hold
inline size_t qa_lds(int ring, int d, int max_len) {
    return ((size_t)16 * ring * (d + 16) + (size_t)3 * ((max_len + 31) / 32 * 32) * QA_LD) * sizeof(f16);
}
inline int qa_ring(int d, int max_len, size_t most) {
    int ring = (max_len + 15) / 16 < QA_RING ? (max_len + 15) / 16 : QA_RING;
    while (ring > 1 && qa_lds(ring, d, max_len) > most)
        ring--;
    return ring;
}
// sizes and plans that the block takes
bool qa_shapes(const et_tile_plan *q, const et_tile_plan *k, const et_tile_plan *v, int max_len, int d, int nheads, int pairs);
void qa_operands(QaArgs &a, const et_tile_plan *q, const et_tile_plan *k, const et_tile_plan *v, int max_len, int d, size_t lds);

} // namespace et

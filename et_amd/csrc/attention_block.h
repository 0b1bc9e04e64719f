// One workgroup's attention: the key-tiled online-softmax block that every
// attention kernel (attention.hip) and the one-launch layer for few rows
// (layer_flow.hip) runs; the layout is described in attention.hip.
#pragma once
#include "common.h"

#include <cmath>
#include <type_traits>

namespace et {

constexpr int AT_KT = 64; // keys per tile

struct AttnArgs {
    f16 *out;
    const f16 *Q, *K, *V, *QK, *mask;
    const int *seq_lens, *cu_seqlens;
    const int *qk_head_ptr, *v_col_id, *v_head_ptr;
    // optional: one bit per (16 query rows, 64-key tile) of the mask, set when
    // any of its elements is non-zero (et_attention_mask_summary); msum_words
    // 32-bit words per group of 16 rows
    const unsigned *msum;
    int msum_words;
    int ldq, ldv, ldo, seq_len, nhead, batch, nqb, total, per_xcd;
    // columns per head in Q, K, V and the output where that is not the kernel's
    // HD (any multiple of 16 below it; the register-staged kernel only): 0 = HD
    int head_width;
    // columns per head in Q and K where they are narrower than the head (compact Q / K with the same number of
    // kept columns in every head; register-staged kernel): 0 = the head's width
    int qk_width;
    float log2_scale, scale;
};

// eight (four) halves at p + d0 of which those at or beyond n read as zero.
// Whole groups are one load that needs no more than the 2-byte alignment of a
// half (compact operands start at arbitrary columns; the hardware takes
// unaligned multi-dword accesses to global memory), only a group that straddles
// n is fetched element by element.
typedef f16x8 f16x8_u __attribute__((aligned(2)));
typedef f16x4 f16x4_u __attribute__((aligned(2)));
__device__ __forceinline__ f16x8 load8_guard(const f16 *p, int d0, int n) {
    if (d0 + 8 <= n)
        return *reinterpret_cast<const f16x8_u *>(p + d0);
    f16x8 v;
#pragma unroll
    for (int j = 0; j < 8; j++)
        v[j] = (d0 + j < n) ? p[d0 + j] : (f16)0;
    return v;
}
__device__ __forceinline__ f16x4 load4_guard(const f16 *p, int d0, int n) {
    if (d0 + 4 <= n)
        return *reinterpret_cast<const f16x4_u *>(p + d0);
    f16x4 v;
#pragma unroll
    for (int j = 0; j < 4; j++)
        v[j] = (d0 + j < n) ? p[d0 + j] : (f16)0;
    return v;
}

// Maximum over the four lanes l, l^16, l^32, l^48 (a query's four key groups),
// result in all four.  gfx950's row-swap instructions exchange whole rows of 16
// lanes between two registers in the vector ALU, so no LDS round trip as with
// __shfl_xor.  (The empty asm statements keep the optimiser from reasoning
// about the swapped copies: it otherwise folds max(a, b) of the pair away.)
__device__ __forceinline__ float xor_max_16_32(float v) {
    unsigned a = __builtin_bit_cast(unsigned, v), b = a;
    asm("" : "+v"(b));
    auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false); // a: lanes 0-31 twice, b: lanes 32-63 twice
    unsigned x0 = r[0], x1 = r[1];
    asm("v_max_f32 %0, %0, %1" : "+v"(x0) : "v"(x1));
    unsigned y1 = x0;
    asm("" : "+v"(y1));
    auto q = __builtin_amdgcn_permlane16_swap(x0, y1, false, false); // even rows twice, odd rows twice
    unsigned z0 = q[0], z1 = q[1];
    asm("v_max_f32 %0, %0, %1" : "+v"(z0) : "v"(z1));
    return __builtin_bit_cast(float, z0);
}

// 4 x 4 transpose of 8-byte pieces over the four lanes l, l+16, l+32, l+48: on entry piece j of the lane in
// row g (g = lane / 16) is element (g, j), on return it is element (j, g).  Two row-swap steps per dword.
__device__ __forceinline__ void transpose_pieces_4x4(f16x4 (&p)[4]) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    u32x2 pc[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
        pc[j] = __builtin_bit_cast(u32x2, p[j]);
#pragma unroll
    for (int d = 0; d < 2; d++) {
        auto s01 = __builtin_amdgcn_permlane16_swap(pc[0][d], pc[1][d], false, false);
        auto s23 = __builtin_amdgcn_permlane16_swap(pc[2][d], pc[3][d], false, false);
        auto t02 = __builtin_amdgcn_permlane32_swap(s01[0], s23[0], false, false);
        auto t13 = __builtin_amdgcn_permlane32_swap(s01[1], s23[1], false, false);
        pc[0][d] = t02[0];
        pc[2][d] = t02[1];
        pc[1][d] = t13[0];
        pc[3][d] = t13[1];
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
        p[j] = __builtin_bit_cast(f16x4, pc[j]);
}

// PLAIN: the launcher has established that there is no mask (or an all-zero
// one), every sequence has full length and seq_len is a multiple of the
// workgroup's query rows - no guards, no mask bookkeeping.
// Wave priority in the two MFMA sections of a key tile (0 in the softmax
// between them): a wave that has its scores or its P ready issues its MFMAs
// ahead of the waves that are in the vector-ALU part (-1 %).
#ifndef AT_PRIO
#define AT_PRIO 1
#endif

// HDK: width of a head in Q and K.  HDK < HD is attention-aware pruning with
// the same number of kept columns in every head: Q and K are compact
// [rows x nhead*HDK], head h at columns h*HDK, and the scores contract over
// HDK; V and the output keep HD columns per head.
// VWIN (pruned variant with dense Q/K and compact V whose row pitch is a
// multiple of 8): K and V are staged by DMA like the unpruned kernel.  A head's
// compact value columns [c0, c1) start at an arbitrary column, which DMA cannot
// address (16-byte pieces), so the tile holds the 16-byte-aligned WINDOW of 80
// columns that begins at c0 rounded down to 8; the product runs over the
// window's 16-column subtiles that reach into [c0, c1) (at most five), and the
// columns of the window that belong to neighbouring heads are never written.
// FLOW: the output rows are read by other workgroups of the SAME launch: they
// are stored past the XCD's own L2 (store_agent8).
// One workgroup's work: the NW*16*QS query rows of block qb of (sequence b, head h).
// MASK: there may be a mask.  Without one (and not PLAIN: ragged lengths) nothing of its bookkeeping is compiled in.
// KS: the waves form KS groups over the same query rows; group k takes key tiles k, k + KS, ... through tile buffers of its
// own, and the groups' partial results meet in LDS behind the loop.
template <int HD, int QS, int NW, bool PRUNED, bool SHAREDQK, bool PLAIN = false, int HDK = HD, bool VWIN = false,
          bool FLOW = false, bool MASK = !PLAIN, int KS = 1>
__device__ __forceinline__ void attention_block(const AttnArgs &a, const int b, const int h, const int qb) {
    static_assert(!PLAIN || ((!PRUNED || VWIN) && !SHAREDQK), "the plain form exists for the DMA-staged kernels only");
    static_assert(!PLAIN || !MASK, "the plain form has no mask");
    static_assert(HDK == HD || (!PRUNED && !SHAREDQK && HDK % 32 == 0), "narrow Q/K heads: on-the-fly kernel only");
    static_assert(!VWIN || (PRUNED && HD == 64), "the value-window form exists for the pruned kernel with 64-wide heads");
    static_assert(KS == 1 || (!PRUNED && !SHAREDQK && QS == 1 && NW % KS == 0), "key groups: the DMA-staged form, a subtile a wave");
    constexpr int AT_WAVES = NW / KS;         // of a group, each owning 16*QS query rows
    constexpr int AT_THREADS = AT_WAVES * 64; // of a group
    constexpr int DK = HDK / 32;   // k-steps of Q K^T
    constexpr int DV = VWIN ? 5 : HD / 16; // 16-wide column subtiles of the output (of the 80-column window)
    // LDS row strides.  K rows are read with ds_read_b128 by 16 lanes at a
    // time: a stride of 32 (mod 64) bytes is conflict-free (measured); V^T rows
    // are read with ds_read_b64, for which an odd multiple of 16 bytes is.
    constexpr int LDK = HDK + 16;
    constexpr int LDV = AT_KT + 8;
    constexpr int QB = AT_WAVES * 16 * QS; // queries per workgroup
    constexpr int LDO = HD + 8;
    // Unpruned operands are staged by DMA (global -> LDS, no registers) in their
    // natural [key][d] layout, K and V alike; the transposed V^T fragments the
    // second contraction needs are then produced by the LDS transpose read
    // (ds_read_b64_tr_b16).  The pruned variant gathers ragged column sets and
    // keeps the register path, which transposes V while storing it - except in
    // its value-window form (VWIN), which is DMA-staged as well.
    constexpr bool DMA = !PRUNED || VWIN;
    constexpr int LDVN = HD + 16; // V row stride in the natural layout (as LDK)
    constexpr int KBUF = AT_KT * LDK, VBUF = DMA ? AT_KT * LDVN : HD * LDV;
    constexpr int SM_KV = 2 * (KBUF + VBUF); // double-buffered key/value tiles
    constexpr int SM_O = QB * LDO;
    constexpr int SM = SM_KV > SM_O ? SM_KV : SM_O;
    extern __shared__ __attribute__((aligned(16))) unsigned char at_smem[];
    f16 *smem = reinterpret_cast<f16 *>(at_smem);
    static_assert(KS * SM * 2 <= 160 * 1024, "LDS budget");

    const int bh = b * a.nhead + h;

    int row0, len, rows_alloc; // first row, valid rows, rows that exist for this sequence
    if (a.cu_seqlens) {
        row0 = a.cu_seqlens[b];
        len = a.cu_seqlens[b + 1] - row0;
        rows_alloc = len;
    } else {
        row0 = b * a.seq_len;
        len = a.seq_lens ? a.seq_lens[b] : a.seq_len;
        rows_alloc = a.seq_len;
    }
    len = min(max(len, 0), a.seq_len);
    const int q0 = qb * QB;
    if (q0 >= rows_alloc)
        return;

    int qc0 = h * HDK, nqk = HD, vc0 = h * HD, nv = HD;
    // head width of the data (HD unless the launcher says otherwise: heads of 48,
    // 80, 96 ... columns run as ragged heads of the next built width)
    const int hw = (PRUNED && !VWIN && a.head_width) ? a.head_width : HD;
    if (PRUNED && !VWIN && a.head_width) {
        qc0 = vc0 = h * hw;
        nqk = nv = hw;
    }
    if (PRUNED && !VWIN && a.qk_width) {
        qc0 = h * a.qk_width;
        nqk = a.qk_width;
    }
    if (PRUNED) {
        if (a.qk_head_ptr) {
            qc0 = a.qk_head_ptr[h];
            nqk = min(a.qk_head_ptr[h + 1] - qc0, HD);
        }
        if (a.v_head_ptr) {
            vc0 = a.v_head_ptr[h];
            nv = min(a.v_head_ptr[h + 1] - vc0, HD);
        }
    }
    // value window: vskip columns of a neighbouring head in front of the head's own nv
    int vskip = 0;
    if (VWIN) {
        // The window starts at the head's first column rounded down to 8, and never
        // beyond ldv - 8: a head that keeps no columns and sits at the very end
        // (v_head_ptr[h] == ldv) would otherwise start its window behind the row,
        // and the clamp of the staging offsets below (ldv - 8 - vc0) would go
        // negative.  The launcher guarantees ldv >= 8.
        const int w0 = min(vc0 & ~7, a.ldv - 8);
        vskip = vc0 - w0;
        vc0 = w0;
        nv += vskip; // columns of the window up to the head's last one
    }

    const int group = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / AT_WAVES;
    const int tid = threadIdx.x - group * AT_THREADS;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) - group * AT_WAVES;
    const int lane = threadIdx.x & 63;
    smem += group * SM;
    const int c16 = lane & 15;
    const int g4 = lane >> 4;
    f16 *obase = a.out + (size_t)row0 * a.ldo + h * hw;
    const f16x8 zero8 = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    auto store_out = [](f16 *p, f16x8 v) {
        if constexpr (FLOW)
            store_agent8(p, v);
        else
            *reinterpret_cast<f16x8 *>(p) = v;
    };

    if (q0 < len) {
        // ---- Q fragments (B operand of S^T), scaled in half like the reference
        f16x8 qf[QS][DK];
        auto load_q = [&] {
            const f16 sc = (f16)a.scale;
#pragma unroll
            for (int qs = 0; qs < QS; qs++) {
                const int q = q0 + (wave * QS + qs) * 16 + c16;
#pragma unroll
                for (int s = 0; s < DK; s++) {
                    f16x8 v = zero8;
                    if (!SHAREDQK && q < len) {
                        const f16 *qrow = a.Q + (size_t)(row0 + q) * a.ldq + qc0;
                        if (PRUNED && !VWIN)
                            v = load8_guard(qrow, s * 32 + g4 * 8, nqk);
                        else
                            v = *reinterpret_cast<const f16x8 *>(qrow + s * 32 + g4 * 8);
                    }
                    qf[qs][s] = v * sc;
                }
            }
        };

        f32x4 ot[DV][QS];
        float m_run[QS];
        // What the key-tile loop needs of m_run in every tile, kept as state and touched only where a
        // maximum is raised (after the first tiles: almost never): the start vector of the score
        // products, four copies of -m (zero while the row has no maximum yet), and the amount a
        // tile's maximum has to exceed before the row's is raised (-inf until then, 8 binades after).
        // They save a dozen vector instructions per tile (padding mask: 1 x 1024 rows 14.7 -> 14.0 us, 2 x 1000 16.6 -> 15.8;
        // two subtiles a wave, 157 registers: 8 x 700 24.7 -> 23.9, 6 x 1024 31.3 -> 30.3).  The register-staged forms with a
        // mask, and heads of 128 with two subtiles, have none to spare and work both out from m_run in every tile.
        constexpr bool KEEP_START = (!MASK || (DMA && (QS == 1 || HD <= 64))) && !SHAREDQK;
        f32x4 neg_m4[QS];
        float raise_over[QS];
        f32x4 l_acc[QS]; // row sums of P, accumulated by the matrix unit (all 16 rows of the tile equal)
#pragma unroll
        for (int qs = 0; qs < QS; qs++) {
            m_run[qs] = -INFINITY;
            neg_m4[qs] = f32x4{-0.f, -0.f, -0.f, -0.f};
            raise_over[qs] = -INFINITY;
            l_acc[qs] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int d = 0; d < DV; d++)
                ot[d][qs] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const bool qk_vec = SHAREDQK && ((a.seq_len & 3) == 0) &&
                            ((reinterpret_cast<uintptr_t>(a.QK) & 7u) == 0);
        const bool qk_vec16 = qk_vec && ((a.seq_len & 7) == 0) && ((reinterpret_cast<uintptr_t>(a.QK) & 15u) == 0);
        const float ls = a.log2_scale;

        // ---- key/value tile staging: global -> registers -> LDS.  The
        // registers of tile t+1 are in flight while tile t is being consumed.
        constexpr int CPR = HD / 8;                                        // 16-byte chunks per K row
        constexpr int NKL = (AT_KT * CPR + AT_THREADS - 1) / AT_THREADS;   // K chunks per thread
        constexpr int DQ = HD / 4;                                         // 4-wide column groups of V
        constexpr int NVW = ((AT_KT / 4) * DQ + AT_THREADS - 1) / AT_THREADS; // V 4x4 blocks per thread
        f16x8 kreg[NKL];
        f16x4 vreg[NVW][4];
        // FULL: every key of the tile is valid, so no per-lane bounds checks
        auto load_tile = [&](int kb, auto full_c) {
            constexpr bool FULL = decltype(full_c)::value;
            if (!SHAREDQK) {
#pragma unroll
                for (int i = 0; i < NKL; i++) {
                    const int idx = tid + i * AT_THREADS;
                    const int key = idx / CPR, dc = idx % CPR;
                    f16x8 v = zero8;
                    if ((AT_KT * CPR % AT_THREADS == 0 || idx < AT_KT * CPR) && (FULL || kb + key < len)) {
                        const f16 *krow = a.K + (size_t)(row0 + kb + key) * a.ldq + qc0;
                        if (PRUNED)
                            v = load8_guard(krow, dc * 8, nqk);
                        else
                            v = *reinterpret_cast<const f16x8 *>(krow + dc * 8);
                    }
                    kreg[i] = v;
                }
            }
#pragma unroll
            for (int i = 0; i < NVW; i++) {
                const int w = tid + i * AT_THREADS;
                const int dq = w % DQ, kq = w / DQ;
#pragma unroll
                for (int kk = 0; kk < 4; kk++) {
                    const int key = kb + kq * 4 + kk;
                    f16x4 v = f16x4{0, 0, 0, 0};
                    if (((AT_KT / 4) * DQ % AT_THREADS == 0 || w < (AT_KT / 4) * DQ) &&
                        (FULL || key < len)) { // rows at or beyond len read as zero
                        const f16 *vrow = a.V + (size_t)(row0 + key) * a.ldv + vc0;
                        if (PRUNED) {
                            v = load4_guard(vrow, dq * 4, nv);
                        } else {
                            v = *reinterpret_cast<const f16x4 *>(vrow + dq * 4);
                        }
                    }
                    vreg[i][kk] = v;
                }
            }
        };
        auto store_tile = [&](int buf) {
            f16 *ks = smem + buf * (KBUF + VBUF);
            f16 *vt = ks + KBUF;
            if (!SHAREDQK) {
#pragma unroll
                for (int i = 0; i < NKL; i++) {
                    const int idx = tid + i * AT_THREADS;
                    const int key = idx / CPR, dc = idx % CPR;
                    if (AT_KT * CPR % AT_THREADS == 0 || idx < AT_KT * CPR)
                        *reinterpret_cast<f16x8 *>(ks + key * LDK + dc * 8) = kreg[i];
                }
            }
#pragma unroll
            for (int i = 0; i < NVW; i++) { // V goes in transposed: [d][key]
                const int w = tid + i * AT_THREADS;
                const int dq = w % DQ, kq = w / DQ;
                if ((AT_KT / 4) * DQ % AT_THREADS == 0 || w < (AT_KT / 4) * DQ) {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const f16x4 t = f16x4{vreg[i][0][e], vreg[i][1][e], vreg[i][2][e], vreg[i][3][e]};
                        *reinterpret_cast<f16x4 *>(vt + (dq * 4 + e) * LDV + kq * 4) = t;
                    }
                }
            }
        };
        // DMA staging of one tile: every instruction moves 64 x 16 bytes to 1 KB
        // of consecutive LDS, so a lane's LDS position decides which (row,
        // column) it fetches; lanes that land in the row padding fetch the
        // row's first bytes.  Rows at or beyond len re-read the last valid row
        // (their scores are masked to -inf / their P is 0).
        // For a tile whose 64 keys all exist, a lane's source is "tile base + an
        // offset that never changes": the offsets are worked out once (byte
        // offsets in 32 bits, relative to the first row of the tile in K or V)
        // and an instruction then costs no address arithmetic in the vector ALU -
        // it was a quarter of the loop's vector instructions.
        constexpr int DMA_ROWBK = LDK * 2, DMA_ROWBV = LDVN * 2; // LDS bytes per row
        constexpr int DMA_NK = (DMA && !SHAREDQK) ? AT_KT * DMA_ROWBK / 1024 : 0;
        constexpr int DMA_NV = DMA ? AT_KT * DMA_ROWBV / 1024 : 0;
        constexpr int DMA_NTOT = DMA_NK + DMA_NV;
        constexpr int DMA_PW = DMA ? (DMA_NTOT + AT_WAVES - 1) / AT_WAVES : 1; // instructions per wave
        unsigned dma_off[DMA_PW];
        if (DMA) {
#pragma unroll
            for (int j = 0; j < DMA_PW; j++) {
                const int i = j * AT_WAVES + wave;
                const bool isv = i >= DMA_NK;
                const int ii = isv ? i - DMA_NK : i;
                const int p = ii * 1024 + lane * 16;
                const int rowb = isv ? DMA_ROWBV : DMA_ROWBK;
                const int row = p / rowb, cb = p - row * rowb;
                int col = cb < (isv ? HD : HDK) * 2 ? (cb >> 1) : 0;
                if (VWIN && isv) // all 80 columns of a window row are data; pieces past the row pitch re-read its last one
                    col = min(cb >> 1, a.ldv - 8 - vc0);
                dma_off[j] = (unsigned)((row * (isv ? a.ldv : a.ldq) + col) * 2);
            }
        }
        auto dma_tile = [&](int kb, int buf) {
            static_assert(!DMA || (AT_KT * DMA_ROWBK % 1024 == 0 && AT_KT * DMA_ROWBV % 1024 == 0),
                          "a tile is a whole number of DMA instructions");
            f16 *ks = smem + buf * (KBUF + VBUF);
            f16 *vs = ks + KBUF;
            if (!PLAIN && __builtin_expect(kb + AT_KT > len, 0)) { // the last tile: rows that do not exist re-read the last one
#pragma unroll
                for (int j = 0; j < DMA_PW; j++) {
                    const int i = j * AT_WAVES + wave;
                    const bool isv = i >= DMA_NK;
                    const int p = (isv ? i - DMA_NK : i) * 1024 + lane * 16;
                    const int row = p / (isv ? DMA_ROWBV : DMA_ROWBK);
                    dma_off[j] -= (unsigned)(max(row - (len - 1 - kb), 0) * (isv ? a.ldv : a.ldq) * 2);
                }
            }
            const char *kbase = reinterpret_cast<const char *>(a.K + (size_t)(row0 + kb) * a.ldq + qc0);
            const char *vbase = reinterpret_cast<const char *>(a.V + (size_t)(row0 + kb) * a.ldv + vc0);
#pragma unroll
            for (int j = 0; j < DMA_PW; j++) {
                const int i = j * AT_WAVES + wave;
                if (DMA_NTOT % AT_WAVES != 0 && i >= DMA_NTOT)
                    break;
                const bool isv = i >= DMA_NK;
                const int ii = isv ? i - DMA_NK : i;
                // (kept opaque in place: otherwise the offsets are folded into 64-bit vector
                // addresses again, one 64-bit add per instruction and tile)
                asm("" : "+v"(dma_off[j]));
                load_lds16((isv ? vbase : kbase) + dma_off[j], (isv ? vs : ks) + ii * 512);
            }
        };
        typedef std::integral_constant<bool, true> yes_t;
        typedef std::integral_constant<bool, false> no_t;

        const int nt = (len + AT_KT - 1) / AT_KT;
        // all of this wave's query rows valid?  (wave-uniform)
        const bool wave_rows_ok = q0 + (wave + 1) * QS * 16 <= len;
        // any of them?  A wave without rows (short sequences) only takes part in the staging and the barriers
        const bool wave_idle = !PLAIN && q0 + wave * QS * 16 >= len;
        // value window: the output column (within the head) of every window column, -1 for the columns of
        // other heads; kept behind the tile buffers for the epilogue
        int *wcol = reinterpret_cast<int *>(at_smem + SM * 2);
        if (VWIN && tid < DV * 16) {
            int c = -1;
            if (tid >= vskip && tid < nv)
                c = (a.v_col_id ? a.v_col_id[vc0 + tid] : vc0 + tid) - h * HD;
            wcol[tid] = (c >= 0 && c < HD) ? c : -1;
        }
        // Does key tile t hold a non-zero mask element for this wave's query
        // rows?  (wave-uniform; all-zero tiles skip the mask loads and adds,
        // which changes no result bit: s + 0 == s.)  The summary words of the
        // first 64 tiles are fetched once, up front; longer sequences do not
        // use the summary.
        unsigned mw0 = 0xFFFFFFFFu, mw1 = 0xFFFFFFFFu;
        if (MASK && a.msum && a.msum_words <= 2) {
            typedef const __attribute__((address_space(4))) unsigned *UConst; // (scalar loads)
            const UConst ms = (UConst)a.msum;
            mw0 = mw1 = 0;
#pragma unroll
            for (int qs = 0; qs < QS; qs++) {
                const int g = (q0 + (wave * QS + qs) * 16) >> 4;
                if (g * 16 < a.seq_len) {
                    mw0 |= ms[g * a.msum_words];
                    if (a.msum_words > 1)
                        mw1 |= ms[g * a.msum_words + 1];
                }
            }
        }
        auto tile_has_mask = [&](int t) -> bool {
            return t >= 64 || (((t < 32 ? mw0 : mw1) >> (t & 31)) & 1u);
        };

        // Additive mask values of one tile.  They are requested one tile ahead (right after the previous tile consumed
        // its own) so the L2 latency is covered by a whole tile of work.
        // Whole mask rows of a tile are 128 bytes: a lane (row, g) takes keys 16g .. 16g+15 as two 16-byte loads, so
        // that the four lanes of a row read each of its lines once; the score layout wants keys 16k + 4g .. +3 for
        // k = 0..3, i.e. the 4 x 4 transpose of the 8-byte pieces across the row's four lanes, done with row swaps
        // when the values are consumed.  Four 8-byte loads per lane, the direct form, touch every line four times from
        // four requests: with twelve waves per CU the lines do not survive in L1 between them, and a dense mask then
        // costs more L2 traffic than K and V together.
        // Rows of any length come this way: the loads need no more than the 2-byte alignment of a half, and what they
        // read behind a row's end belongs to keys that do not exist (their scores become -inf).  Only the last few
        // elements of the array, where a whole load would pass its end, are fetched one by one.  (Element loads for
        // every row that is not 8-byte aligned or that ends inside the tile were sixteen dependent round trips: 2 x
        // 1021 rows, dense mask, 60 us against 23 for 2 x 1024.)
        f16x4 mk[QS][4];
        const f16 *mrow[QS]; // the lane's first key
        if (MASK && a.mask) {
#pragma unroll
            for (int qs = 0; qs < QS; qs++)
                mrow[qs] = a.mask + (size_t)min(q0 + (wave * QS + qs) * 16 + c16, a.seq_len - 1) * a.seq_len + g4 * 16;
        }
        auto load_mask = [&](int kb) {
#pragma unroll
            for (int qs = 0; qs < QS; qs++) {
                f16x8 l[2];
                const f16 *m = mrow[qs] + kb;
                if (kb + AT_KT <= a.seq_len) { // (wave-uniform)
                    l[0] = *reinterpret_cast<const f16x8_u *>(m);
                    l[1] = *reinterpret_cast<const f16x8_u *>(m + 8);
                } else {
                    const int left = (int)min(a.mask + (size_t)a.seq_len * a.seq_len - m, (ptrdiff_t)16);
                    l[0] = load8_guard(m, 0, left);
                    l[1] = load8_guard(m, 8, left);
                }
                mk[qs][0] = f16x4{l[0][0], l[0][1], l[0][2], l[0][3]};
                mk[qs][1] = f16x4{l[0][4], l[0][5], l[0][6], l[0][7]};
                mk[qs][2] = f16x4{l[1][0], l[1][1], l[1][2], l[1][3]};
                mk[qs][3] = f16x4{l[1][4], l[1][5], l[1][6], l[1][7]};
            }
        };
        // (query rows at or beyond len have no Q, and whatever they sum up is never stored; only stored scores are read)
        auto fast_tile = [&](int kb) { return kb + AT_KT <= len && (!SHAREDQK || (wave_rows_ok && qk_vec)); };
        bool has_mask_cur = false;
        auto mask_ahead = [&] { // the first tile's
            has_mask_cur = MASK && !wave_idle && a.mask && group < nt && tile_has_mask(group);
            if (has_mask_cur)
                load_mask(group * AT_KT);
        };

        // One key tile.  FAST: all 64 keys and all of the wave's query rows are
        // valid and the vector paths apply, so the body has no per-lane
        // predicates at all.
        bool has_mask_next = false;
        // (FAST and MASKED are wave-uniform run-time flags, not template
        // parameters: four inlined copies of this body made the register
        // allocator keep a second copy of every accumulator - 223 VGPRs against
        // 122 for one copy - which halved the waves per SIMD)
        auto tile_body = [&](int kb, const f16 *ks, const f16 *vt, const bool FAST, const bool MASKED) {
            // MASKED: this tile's mask values are in mk
            __builtin_amdgcn_s_setprio(AT_PRIO);
            // ---- scores, transposed: st[ksub][qs][r] = S[q = c16][key = 16 ksub + 4 g4 + r],
            // MINUS the row's running maximum: the matrix unit starts from -m
            // instead of zero, which costs nothing there and saves the vector
            // ALU one subtraction per score
            f32x4 st[4][QS];
            float m_ref[QS];
            f32x4 nm4[QS];
#pragma unroll
            for (int qs = 0; qs < QS; qs++) {
                if (KEEP_START) {
                    nm4[qs] = neg_m4[qs];
                    m_ref[qs] = -nm4[qs][0]; // (only used where a maximum is raised)
                } else {
                    m_ref[qs] = (m_run[qs] == -INFINITY) ? 0.f : m_run[qs];
                    nm4[qs] = f32x4{-m_ref[qs], -m_ref[qs], -m_ref[qs], -m_ref[qs]};
                }
            }
            if (!SHAREDQK) {
                // K fragments are read one 16-key subtile ahead of the MFMAs that
                // use them (two subtiles' worth of registers instead of four)
                f16x8 kfr[2][DK];
#pragma unroll
                for (int s = 0; s < DK; s++)
                    kfr[0][s] = *reinterpret_cast<const f16x8 *>(ks + c16 * LDK + s * 32 + g4 * 8);
#pragma unroll
                for (int ksub = 0; ksub < 4; ksub++) {
                    if (ksub + 1 < 4) {
#pragma unroll
                        for (int s = 0; s < DK; s++)
                            kfr[(ksub + 1) & 1][s] = *reinterpret_cast<const f16x8 *>(
                                ks + ((ksub + 1) * 16 + c16) * LDK + s * 32 + g4 * 8);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int s = 0; s < DK; s++)
#pragma unroll
                        for (int qs = 0; qs < QS; qs++) // (the first step reads -m as its C operand: no copies)
                            st[ksub][qs] = mfma16x16x32(kfr[ksub & 1][s], qf[qs][s], s == 0 ? nm4[qs] : st[ksub][qs]);
                }
            } else if (FAST && qk_vec16) {
                // stored scores of a full tile: line-wise like the mask (128 bytes per query row and tile)
#pragma unroll
                for (int qs = 0; qs < QS; qs++) {
                    const int q = q0 + (wave * QS + qs) * 16 + c16;
                    const f16 *src = a.QK + ((size_t)bh * a.seq_len + q) * a.seq_len + kb + g4 * 16;
                    const f16x8 l0 = *reinterpret_cast<const f16x8 *>(src);
                    const f16x8 l1 = *reinterpret_cast<const f16x8 *>(src + 8);
                    f16x4 pc[4] = {f16x4{l0[0], l0[1], l0[2], l0[3]}, f16x4{l0[4], l0[5], l0[6], l0[7]},
                                   f16x4{l1[0], l1[1], l1[2], l1[3]}, f16x4{l1[4], l1[5], l1[6], l1[7]}};
                    transpose_pieces_4x4(pc);
#pragma unroll
                    for (int ksub = 0; ksub < 4; ksub++)
                        st[ksub][qs] = __builtin_convertvector(pc[ksub], f32x4) - m_ref[qs];
                }
            } else {
#pragma unroll
                for (int qs = 0; qs < QS; qs++) {
                    const int q = q0 + (wave * QS + qs) * 16 + c16;
#pragma unroll
                    for (int ksub = 0; ksub < 4; ksub++) {
                        const int key = kb + ksub * 16 + g4 * 4;
                        f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
                        const f16 *src = a.QK + ((size_t)bh * a.seq_len + q) * a.seq_len + key;
                        if (FAST || (q < len && qk_vec && key + 3 < len)) {
                            const f16x4 t4 = *reinterpret_cast<const f16x4 *>(src);
#pragma unroll
                            for (int r = 0; r < 4; r++)
                                v[r] = (float)t4[r];
                        } else if (q < len) {
#pragma unroll
                            for (int r = 0; r < 4; r++)
                                if (key + r < len)
                                    v[r] = (float)src[r];
                        }
                        st[ksub][qs] = v - m_ref[qs];
                    }
                }
            }

            __builtin_amdgcn_s_setprio(0);
            // ---- mask, online softmax, pack P as the B operand.  The running
            // maximum is only raised when a row's new maximum exceeds it by
            // more than 8 binades (P then stays <= 256, exact enough in half),
            // so after the first tiles the accumulator rescale is skipped.
            f16x8 pf[QS][2];
            if (MASKED) { // the loads hold key blocks per lane: into the score layout
#pragma unroll
                for (int qs = 0; qs < QS; qs++)
                    transpose_pieces_4x4(mk[qs]);
            }
            if (MASKED) {
                // (the multiplier is exactly 1.0 but opaque to the optimiser,
                // which would otherwise turn the fused form back into a
                // conversion and an add)
                float one = 1.0f;
                asm("" : "+s"(one));
#pragma unroll
                for (int qs = 0; qs < QS; qs++)
#pragma unroll
                    for (int ksub = 0; ksub < 4; ksub++)
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            // (as a fused multiply-add by one: the mixed-precision
                            // form takes the half operand directly, no conversion)
                            st[ksub][qs][r] = __builtin_fmaf((float)mk[qs][ksub][r], one, st[ksub][qs][r]);
            }
            if (MASK && a.mask) { // next tile's mask
                has_mask_next = kb + KS * AT_KT < len && tile_has_mask((kb + KS * AT_KT) / AT_KT);
                if (has_mask_next)
                    load_mask(kb + KS * AT_KT);
            }
            // the lane's part of each row maximum (of s - m_ref); the row's other three
            // parts only matter when some row of the wave has to raise its maximum
            float pmx[QS];
            bool live = false;
#pragma unroll
            for (int qs = 0; qs < QS; qs++) {
                if (!FAST) {
#pragma unroll
                    for (int ksub = 0; ksub < 4; ksub++)
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            if (kb + ksub * 16 + g4 * 4 + r >= len)
                                st[ksub][qs][r] = -INFINITY;
                }
                float mx = -INFINITY;
#pragma unroll
                for (int ksub = 0; ksub < 4; ksub++) {
                    mx = fmaxf(fmaxf(mx, st[ksub][qs][0]), st[ksub][qs][1]);
                    mx = fmaxf(fmaxf(mx, st[ksub][qs][2]), st[ksub][qs][3]);
                }
                pmx[qs] = mx;
                // does this tile add anything to the row?  Not if every score is 160 binades or more under a
                // maximum the row already has: every exp2 is then exactly zero in fp32 (so is P, and the sums
                // and the output do not change).
                if (MASK)
                    live = live || m_run[qs] == -INFINITY || !(mx * ls < -160.0f);
            }
            // A tile that is dead for every row of the wave - the keys behind a padding mask - ends here: no
            // exponentials, no second product (wave-uniform; same bits as going through with P = 0).
            if (MASK && __builtin_amdgcn_ballot_w64(live) == 0)
                return;
#pragma unroll
            for (int qs = 0; qs < QS; qs++) {
                float mx = pmx[qs];
                // (a row without a maximum yet takes its first finite one: raise_over is -inf then)
                auto raises = [&](float v) {
                    if (KEEP_START)
                        return v * ls > raise_over[qs];
                    return (m_run[qs] == -INFINITY) ? (v > -INFINITY) : (v * ls > 8.0f);
                };
                const bool up_lane = raises(mx);
                if (__builtin_amdgcn_ballot_w64(up_lane) != 0) {
                    mx = xor_max_16_32(mx);
                    const bool up = raises(mx);
                    const float m_new = up ? mx + m_ref[qs] : m_run[qs];
                    const float m_fin = (m_new == -INFINITY) ? 0.f : m_new;
                    const float alpha = __builtin_amdgcn_exp2f((m_run[qs] - m_fin) * ls); // 1 where unchanged
                    const float shift = m_fin - m_ref[qs];                                // 0 where unchanged
                    m_run[qs] = m_new;
                    if (KEEP_START) {
                        neg_m4[qs] = f32x4{-m_fin, -m_fin, -m_fin, -m_fin};
                        raise_over[qs] = (m_new == -INFINITY) ? -INFINITY : 8.0f;
                    }
                    l_acc[qs] *= alpha;
#pragma unroll
                    for (int d = 0; d < DV; d++)
                        ot[d][qs] *= alpha;
#pragma unroll
                    for (int ksub = 0; ksub < 4; ksub++)
                        st[ksub][qs] -= shift;
                }
                if (ls != 1.0f) { // (wave-uniform; base-2 softmax needs no multiplication at all)
#pragma unroll
                    for (int ksub = 0; ksub < 4; ksub++)
                        st[ksub][qs] *= ls;
                }
                f16x2 ph[8];
#pragma unroll
                for (int ksub = 0; ksub < 4; ksub++)
#pragma unroll
                    for (int r2 = 0; r2 < 2; r2++) {
                        const float p0 = __builtin_amdgcn_exp2f(st[ksub][qs][2 * r2]);
                        const float p1 = __builtin_amdgcn_exp2f(st[ksub][qs][2 * r2 + 1]);
                        typedef float f32x2 __attribute__((ext_vector_type(2)));
                        ph[ksub * 2 + r2] = __builtin_convertvector(f32x2{p0, p1}, f16x2);
                    }
#pragma unroll
                for (int kk = 0; kk < 2; kk++)
                    pf[qs][kk] = f16x8{ph[kk * 4 + 0][0], ph[kk * 4 + 0][1], ph[kk * 4 + 1][0], ph[kk * 4 + 1][1],
                                       ph[kk * 4 + 2][0], ph[kk * 4 + 2][1], ph[kk * 4 + 3][0], ph[kk * 4 + 3][1]};
            }

            __builtin_amdgcn_s_setprio(AT_PRIO);
            // ---- O^T += V^T P^T, V^T fragments read one 16-column subtile ahead
            {
                auto load_v = [&](int d, f16x8 (&dst)[2]) {
#pragma unroll
                    for (int kk = 0; kk < 2; kk++) {
                        f16x4 v0, v1;
                        if (DMA) {
                            // natural layout [key][d]: the transpose read hands lane
                            // c of a 16-lane group the 4 consecutive keys of column
                            // d0+c when lane i of the group addresses row i/4,
                            // columns 4(i%4)..+3.  The B operand's 8 k-slots are
                            // keys 4g..4g+3 of subtile 2kk and of subtile 2kk+1.
                            typedef short s16x4 __attribute__((ext_vector_type(4)));
                            typedef __attribute__((address_space(3))) s16x4 *lds4;
                            const f16 *vrow = vt + (kk * 32 + g4 * 4 + (c16 >> 2)) * LDVN + d * 16 + (c16 & 3) * 4;
                            v0 = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)vrow));
                            v1 = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(vrow + 16 * LDVN)));
                        } else {
                            const f16 *vrow = vt + (d * 16 + c16) * LDV + kk * 32 + g4 * 4;
                            v0 = *reinterpret_cast<const f16x4 *>(vrow);
                            v1 = *reinterpret_cast<const f16x4 *>(vrow + 16);
                        }
                        dst[kk] = f16x8{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                    }
                };
                f16x8 vfr[2][2];
                load_v(0, vfr[0]);
#pragma unroll
                for (int d = 0; d < DV; d++) {
                    // (a head that keeps nv < 64 value columns has nothing in the
                    // subtiles from ceil(nv / 16) on: wave-uniform skip)
                    if (PRUNED && d * 16 >= nv)
                        break;
                    if (d + 1 < DV)
                        load_v(d + 1, vfr[(d + 1) & 1]);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int kk = 0; kk < 2; kk++)
#pragma unroll
                        for (int qs = 0; qs < QS; qs++)
                            ot[d][qs] = mfma16x16x32(vfr[d & 1][kk], pf[qs][kk], ot[d][qs]);
                }
                // the softmax denominators: ones^T P^T sums a query's 64
                // probabilities (as rounded to half for the product above)
                // without any vector adds or cross-lane steps
                const f16x8 ones8 = f16x8{1, 1, 1, 1, 1, 1, 1, 1};
#pragma unroll
                for (int kk = 0; kk < 2; kk++)
#pragma unroll
                    for (int qs = 0; qs < QS; qs++)
                        l_acc[qs] = mfma16x16x32(ones8, pf[qs][kk], l_acc[qs]);
            }
            __builtin_amdgcn_s_setprio(0);
        };

        // Everything the first tiles need is requested before anything is waited for: K and V of the first tile, Q, the
        // first mask values, K and V of the second tile (whose wait is the first tile's end).
        if (DMA) {
            if (KS == 1 || group < nt)
                dma_tile(group * AT_KT, 0);
            load_q();
            mask_ahead();
            if (nt > group + KS) {
                dma_tile((group + KS) * AT_KT, 1);
                constexpr int BEHIND = DMA_NTOT / AT_WAVES; // at least so many requests of this wave are the second tile's
                __builtin_amdgcn_s_waitcnt(0x0F70 | (BEHIND & 15) | (BEHIND >> 4 << 14)); // vmcnt(BEHIND)
            } else {
                __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
            }
        } else {
            if (AT_KT <= len)
                load_tile(0, yes_t{});
            else
                load_tile(0, no_t{});
            load_q();
            mask_ahead();
            store_tile(0);
        }
        __syncthreads();

        // Without a mask: the full tiles in a loop of their own, the last one behind it (the bounds as a branch inside
        // the loop cost 0.15 us a tile: 2 x 1024 rows with lengths 15.9 us, without 13.4).
        constexpr bool PEEL = DMA && !MASK && !SHAREDQK && !PLAIN && KS == 1;
        const int nloop = PEEL ? len / AT_KT : (nt + KS - 1) / KS;
        for (int t = 0; t < nloop; t++) {
            const int kb = (t * KS + group) * AT_KT;
            const f16 *ks = smem + (t & 1) * (KBUF + VBUF);
            const f16 *vt = ks + KBUF;
            const bool more = (t + 1) * KS + group < nt;
            // tile t+1 goes into the other buffer (last read in iteration t-1,
            // which every wave left before the previous barrier) while tile t is
            // consumed: by DMA straight away, or through registers that are
            // stored after the tile body
            if (more) {
                if (DMA && t > 0) // (the second tile is on its way)
                    dma_tile(kb + KS * AT_KT, (t + 1) & 1);
                else if (DMA)
                    ;
                else if (kb + 2 * AT_KT <= len)
                    load_tile(kb + AT_KT, yes_t{});
                else
                    load_tile(kb + AT_KT, no_t{});
            }
            if (KS > 1 && kb >= len) // (the other groups' last step)
                ;
            else if constexpr (PLAIN)
                tile_body(kb, ks, vt, true, false);
            else if (PEEL) {
                if (!wave_idle)
                    tile_body(kb, ks, vt, true, false);
            }
            else if (!wave_idle)
                tile_body(kb, ks, vt, fast_tile(kb), has_mask_cur);
            has_mask_cur = has_mask_next;
            if (more) {
                if (DMA)
                    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): this wave's part of tile t+1 has landed
                else
                    store_tile((t + 1) & 1);
            }
            __syncthreads();
        }
        if (PEEL && nloop < nt) {
            const f16 *ks = smem + (nloop & 1) * (KBUF + VBUF);
            if (!wave_idle)
                tile_body(nloop * AT_KT, ks, ks + KBUF, false, false);
            __syncthreads();
        }

        if constexpr (KS > 1) { // the groups' sums, each under its own maximum
            constexpr int PART = AT_THREADS * (DV * 4 + 2); // floats of a group
            static_assert(PART * 4 <= SM * 2, "a group's sums fit its tile buffers");
            f32x4 *const part = reinterpret_cast<f32x4 *>(smem);
            float *const stat = reinterpret_cast<float *>(part + DV * AT_THREADS);
            if (group > 0) {
#pragma unroll
                for (int d = 0; d < DV; d++)
                    part[d * AT_THREADS + tid] = ot[d][0];
                stat[tid] = m_run[0];
                stat[AT_THREADS + tid] = l_acc[0][0];
            }
            __syncthreads();
            if (group == 0) {
#pragma unroll
                for (int g = 1; g < KS; g++) {
                    const f32x4 *const other = part + g * (SM / 8);
                    const float *const ostat = stat + g * (SM / 2);
                    const float m_o = ostat[tid], m_new = fmaxf(m_run[0], m_o), m_fin = m_new == -INFINITY ? 0.f : m_new;
                    const float mine = __builtin_amdgcn_exp2f((m_run[0] - m_fin) * ls), its = __builtin_amdgcn_exp2f((m_o - m_fin) * ls);
                    m_run[0] = m_new;
                    l_acc[0] = l_acc[0] * mine + ostat[AT_THREADS + tid] * its;
#pragma unroll
                    for (int d = 0; d < DV; d++)
                        ot[d][0] = ot[d][0] * mine + other[d * AT_THREADS + tid] * its;
                }
            }
        }
        // ---- normalise and stage the output block in LDS (all waves are past
        // the loop's final barrier, so the tile buffers are free)
        f16 *os = smem - group * SM;
        if (PRUNED) { // columns that no kept V column maps to must read as zero
            for (int i = tid; i < SM_O / 8; i += AT_THREADS)
                reinterpret_cast<f16x8 *>(os)[i] = zero8;
            __syncthreads();
        }
        if (KS == 1 || group == 0)
#pragma unroll
            for (int qs = 0; qs < QS; qs++) {
            const float l = l_acc[qs][0];
            const float inv = l > 0.f ? 1.0f / l : 0.f;
            const int ql = (wave * QS + qs) * 16 + c16;
#pragma unroll
            for (int d = 0; d < DV; d++) {
                f16x4 o;
#pragma unroll
                for (int r = 0; r < 4; r++)
                    o[r] = (f16)(ot[d][qs][r] * inv);
                if (VWIN) {
                    typedef int i32x4 __attribute__((ext_vector_type(4)));
                    const i32x4 c4 = *reinterpret_cast<const i32x4 *>(wcol + d * 16 + g4 * 4);
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (c4[r] >= 0)
                            os[ql * LDO + c4[r]] = o[r];
                } else if (PRUNED) {
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int j = d * 16 + g4 * 4 + r;
                        if (j < nv) {
                            const int col = (a.v_col_id ? a.v_col_id[vc0 + j] : vc0 + j) - h * hw;
                            if (col >= 0 && col < hw)
                                os[ql * LDO + col] = o[r];
                        }
                    }
                } else {
                    *reinterpret_cast<f16x4 *>(os + ql * LDO + d * 16 + g4 * 4) = o;
                }
            }
        }
        __syncthreads();
        for (int idx = threadIdx.x; idx < QB * CPR; idx += NW * 64) {
            const int ql = idx / CPR, dc = idx % CPR;
            const int q = q0 + ql;
            if (q < rows_alloc && dc * 8 < hw) {
                f16x8 v = zero8;
                if (q < len)
                    v = *reinterpret_cast<const f16x8 *>(os + ql * LDO + dc * 8);
                store_out(obase + (size_t)q * a.ldo + dc * 8, v);
            }
        }
    } else {
        // whole query block is padding: rows exist (padded layout) and read as zero
        constexpr int CPR = HD / 8;
        for (int idx = threadIdx.x; idx < QB * CPR; idx += NW * 64) {
            const int ql = idx / CPR, dc = idx % CPR;
            const int q = q0 + ql;
            if (q < rows_alloc && dc * 8 < hw)
                store_out(obase + (size_t)q * a.ldo + dc * 8, zero8);
        }
    }
}

// LDS bytes of one workgroup (mirrors the constants inside attention_block)
template <int HD, int QS, int NW, bool PRUNED, int HDK = HD, bool VWIN = false, int KS = 1> constexpr size_t attn_lds_bytes() {
    // (must agree with the kernel's KBUF / VBUF)
    constexpr int KV = 2 * (AT_KT * (HDK + 16) + ((PRUNED && !VWIN) ? HD * (AT_KT + 8) : AT_KT * (HD + 16)));
    constexpr int O = NW / KS * 16 * QS * (HD + 8);
    return sizeof(f16) * (size_t)KS * (KV > O ? KV : O) + (VWIN ? 5 * 16 * sizeof(int) : 0); // (+ the window's column table)
}

// what a launcher fills in besides the operands (attention.hip): head scale,
// output pitch and the attached mask summary; returns whether the mask is known
// to be zero everywhere
bool attention_finish_args(AttnArgs &a, int d_model);

} // namespace et

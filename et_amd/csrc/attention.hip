// Fused multi-head self-attention for gfx950: on-the-fly (scores never leave
// the CU), attention-aware pruned (compact Q/K/V column sets per head) and the
// score-matrix-in-memory variant, all from one key-tiled online-softmax kernel.
//
// Reference math (kernels/attention.cu:51-120): Qs = half(Q*scale),
// S = Qs K^T + mask, P = softmax_base2(S), Z = P V, per head, per 16-row query
// block, with the whole 16 x seq_len score block in shared memory.  Here the
// keys are walked in tiles of 64 with a running max / running sum, so LDS use
// is independent of seq_len and no S x S block exists anywhere.
//
// Layout trick: both contractions are issued TRANSPOSED.
//   S^T(keys x queries) = K_tile * Qs^T : A = K rows from LDS, B = Q fragment
//     held in registers for the whole kernel.  A lane (c = lane%16, g =
//     lane/16) then holds, for ONE query c, four consecutive keys 4g..4g+3 of
//     each 16-key subtile, so row max / row sum need only two cross-lane steps
//     (xor 16, xor 32) and the running statistics are per-lane scalars.
//   O^T(d x queries) = V^T * P^T : the P values a lane already holds are, as
//     they stand, the B operand (8 k-slots = 4 keys of subtile 2kk + 4 keys
//     of subtile 2kk+1); the matching A operand is a V^T fragment, which the
//     LDS transpose read (ds_read_b64_tr_b16) produces from a V tile kept in
//     its natural [key][d] layout (the pruned variant transposes V while
//     staging it instead).  P never goes through LDS and the O accumulator's
//     query index is again the lane's c, so the online rescale is a per-lane
//     multiply.
// K and V tiles of the unpruned variants are staged by DMA (global -> LDS
// without registers), double-buffered, one tile ahead of the MFMAs.
#include "attention_block.h"

#include <mutex>
#include <vector>

namespace et {

// A workgroup's query block qb of pair bh; false: none.  Workgroup ids go round-robin over the 8 XCDs.  XCD x works on
// the (batch, head) pairs x, x+8, x+16, ... in that order, all query blocks of a pair together (they share its K and V in
// that XCD's L2): with sequences of different lengths every XCD gets an even mix, and pairs keep their order.
__device__ __forceinline__ bool attn_place(const AttnArgs &a, int &bh, int &qb) {
    const int xcd = blockIdx.x & 7, rest = blockIdx.x >> 3; // rest < per_xcd = ceil(pairs / 8) * nqb
    qb = rest % a.nqb;
    bh = (rest / a.nqb) * 8 + xcd;
    return bh < a.nhead * a.batch;
}

template <int HD, int QS, int NW, bool PRUNED, bool SHAREDQK, bool PLAIN = false, int HDK = HD, bool VWIN = false,
          bool MASK = !PLAIN>
__global__ void __launch_bounds__(NW * 64, (QS == 1 && HD <= 64) ? 4 : 2) attention_kernel(const AttnArgs a) {
    int bh, qb;
    if (attn_place(a, bh, qb))
        attention_block<HD, QS, NW, PRUNED, SHAREDQK, PLAIN, HDK, VWIN, false, MASK>(a, bh / a.nhead, bh % a.nhead, qb);
}

// the same in two groups of four waves over the key tiles of a block of 64 query rows (two_key_groups)
template <int HD, bool PLAIN, bool MASK>
__global__ void __launch_bounds__(512, 4) attention_two_groups_kernel(const AttnArgs a) {
    int bh, qb;
    if (attn_place(a, bh, qb))
        attention_block<HD, 1, 8, false, false, PLAIN, HD, false, false, MASK, 2>(a, bh / a.nhead, bh % a.nhead, qb);
}

// Packed sequences of different lengths (cu_seqlens): a grid of one workgroup per
// (sequence, head, query block of the LONGEST sequence) is mostly workgroups that
// find nothing to do, and dispatching those costs as much as the work of a batch
// of short sequences.  Here the grid is what the chip holds at once and every
// workgroup walks its share of the blocks that exist: XCD x owns the (sequence,
// head) pairs x, x+8, ... as above, their query blocks in order form that XCD's
// list, and workgroup k of the W on the XCD takes blocks k, k+W, k+2W, ... .
// A block's position in the list is found from the running block count per
// sequence, which every wave keeps in registers (lane l: sequences l, l+64, ...;
// at most 64*AT_PX sequences).
constexpr int AT_PX = 4;
// workgroups that a CU holds at once, by which the launcher sizes the grid: the registers have to allow them (the bound
// counts waves of a SIMD)
constexpr int packed_on_cu(int HD, int QS, int KS) { return QS == 2 ? 3 : HD <= 64 ? 4 / KS : 2; }
template <int HD, int QS, int NW, bool MASK, int KS = 1>
__global__ void __launch_bounds__(NW * 64, packed_on_cu(HD, QS, KS) * NW / 4) attention_packed_kernel(const AttnArgs a) {
    constexpr int QB = NW / KS * 16 * QS;
    const int lane = threadIdx.x & 63;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, W = gridDim.x >> 3;
    int px[AT_PX], nbv[AT_PX]; // blocks before sequence (l + 64 r) in this XCD's list; its query blocks
    int run = 0;
#pragma unroll
    for (int r = 0; r < AT_PX; r++) {
        const int s = lane + 64 * r;
        int nb = 0, v = 0;
        if (s < a.batch) {
            const int len = min(max(a.cu_seqlens[s + 1] - a.cu_seqlens[s], 0), a.seq_len);
            nb = (len + QB - 1) / QB;
            const int h0 = (xcd - s * a.nhead) & 7; // first head of the sequence whose pair lands on this XCD
            v = h0 < a.nhead ? nb * ((a.nhead - h0 + 7) >> 3) : 0;
        }
        int inc = v; // inclusive scan over the 64 lanes
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int t = __shfl_up(inc, d, 64);
            inc += lane >= d ? t : 0;
        }
        px[r] = s < a.batch ? run + inc - v : 0x7fffffff;
        nbv[r] = nb;
        run += __shfl(inc, 63, 64);
    }
    run = __builtin_amdgcn_readfirstlane(run);
    for (int i = slot; i < run; i += W) {
        // the sequence: the last one whose first block is at or before i (the counts never decrease, and a
        // sequence without blocks on this XCD shares its successor's count and is passed over)
        int cnt = 0;
#pragma unroll
        for (int r = 0; r < AT_PX; r++)
            cnt += __builtin_popcountll(__builtin_amdgcn_ballot_w64(px[r] <= i));
        const int b = cnt - 1; // (cnt >= 1: the first sequence's count is 0)
        int first = 0, nb = 1;
#pragma unroll
        for (int r = 0; r < AT_PX; r++)
            if ((b >> 6) == r) {
                first = __builtin_amdgcn_readlane(px[r], b & 63);
                nb = __builtin_amdgcn_readlane(nbv[r], b & 63);
            }
        const int rem = i - first;
        const int h = ((xcd - b * a.nhead) & 7) + 8 * (rem / max(nb, 1));
        if (nb <= 0 || rem < 0 || b >= a.batch || h >= a.nhead)
            continue; // (cannot happen with consistent counts; never index past the operands)
        attention_block<HD, QS, NW, false, false, false, HD, false, false, MASK, KS>(a, b, h, rem % nb);
        __syncthreads(); // the block's output staging in LDS is read before the next block's tiles land there
    }
}

// scaled Q K^T written to memory, [(b*nhead+h)][q][k]; one wave per 64 queries x 64 keys (the K fragments are
// fetched once and used for four tiles of 16 queries), transposed product so a lane owns 4 consecutive keys of
// one query.  A query's 64 scores of the tile are 128 bytes, one cache line: the lane's four 8-byte pieces are
// transposed over the query's four lanes so that every lane stores 32 contiguous bytes and the four of them the
// whole line (element-wise 2-byte stores of the same values took 129 us for batch 16 x seq 512, six times the
// time of writing 100 MB).
template <int HD>
__global__ void __launch_bounds__(256)
qk_scores_kernel(f16 *__restrict__ QK, const f16 *__restrict__ Q, const f16 *__restrict__ K,
                 int seq_len, int d_model, int nhead, float scale) {
    constexpr int DK = HD / 32;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
    const int bh = blockIdx.z, h = bh % nhead, b = bh / nhead;
    const int qb0 = blockIdx.y * 64;
    const int k0 = (blockIdx.x * 4 + wave) * 64;
    if (k0 >= seq_len)
        return;
    const size_t row0 = (size_t)b * seq_len;
    f16x8 kf[4][DK];
#pragma unroll
    for (int ksub = 0; ksub < 4; ksub++) {
        const int key = k0 + ksub * 16 + c16;
#pragma unroll
        for (int s = 0; s < DK; s++) {
            kf[ksub][s] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (key < seq_len)
                kf[ksub][s] = *reinterpret_cast<const f16x8 *>(K + (row0 + key) * d_model + h * HD + s * 32 + g4 * 8);
        }
    }
    // whole lines: all 64 keys exist and rows start on 16-byte boundaries (wave-uniform)
    const bool lines = k0 + 64 <= seq_len && (seq_len & 7) == 0 && (reinterpret_cast<uintptr_t>(QK) & 15u) == 0;
    for (int qt = 0; qt < 4; qt++) {
        if (qb0 + qt * 16 >= seq_len)
            break;
        const int q = qb0 + qt * 16 + c16;
        f16x8 qf[DK];
#pragma unroll
        for (int s = 0; s < DK; s++) {
            qf[s] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (q < seq_len)
                qf[s] = *reinterpret_cast<const f16x8 *>(Q + (row0 + q) * d_model + h * HD + s * 32 + g4 * 8);
        }
        f16x4 pc[4]; // piece ksub: keys k0 + 16 ksub + 4 g4 .. + 3 of query q
#pragma unroll
        for (int ksub = 0; ksub < 4; ksub++) {
            f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < DK; s++)
                acc = mfma16x16x32(kf[ksub][s], qf[s], acc);
            pc[ksub] = __builtin_convertvector(acc * scale, f16x4);
        }
        f16 *qrow = QK + ((size_t)bh * seq_len + q) * seq_len + k0;
        if (lines) {
            transpose_pieces_4x4(pc); // piece j: keys k0 + 16 g4 + 4 j .. + 3
            if (q < seq_len) {
                *reinterpret_cast<f16x8 *>(qrow + g4 * 16) =
                    f16x8{pc[0][0], pc[0][1], pc[0][2], pc[0][3], pc[1][0], pc[1][1], pc[1][2], pc[1][3]};
                *reinterpret_cast<f16x8 *>(qrow + g4 * 16 + 8) =
                    f16x8{pc[2][0], pc[2][1], pc[2][2], pc[2][3], pc[3][0], pc[3][1], pc[3][2], pc[3][3]};
            }
        } else if (q < seq_len) {
#pragma unroll
            for (int ksub = 0; ksub < 4; ksub++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (k0 + ksub * 16 + g4 * 4 + r < seq_len)
                        qrow[ksub * 16 + g4 * 4 + r] = pc[ksub][r];
        }
    }
}

template <auto KERN> static void attn_launch_grid(size_t lds, int threads, const AttnArgs &a, hipStream_t st) {
    launch_kernel<KERN>(dim3(a.per_xcd * 8), dim3(threads), lds, st, a);
}
template <int HD, int QS, int NW, bool PRUNED, bool SHAREDQK, bool PLAIN = false, int HDK = HD, bool VWIN = false,
          bool MASK = !PLAIN>
static void attn_launch_one(const AttnArgs &a, hipStream_t st) {
    constexpr auto kern = &attention_kernel<HD, QS, NW, PRUNED, SHAREDQK, PLAIN, HDK, VWIN, MASK>;
    attn_launch_grid<kern>(attn_lds_bytes<HD, QS, NW, PRUNED, HDK, VWIN>(), NW * 64, a, st);
}
template <int HD, bool PLAIN, bool MASK> static void attn_launch_two_groups(const AttnArgs &a, hipStream_t st) {
    constexpr auto kern = &attention_two_groups_kernel<HD, PLAIN, MASK>;
    attn_launch_grid<kern>(attn_lds_bytes<HD, 1, 8, false, HD, false, 2>(), 512, a, st);
}

// Blocks of 128 query rows for packed sequences without a mask: K and V are read from LDS once per 32 queries of a wave
// instead of 16, but a short last block wastes more and fewer blocks balance worse.  The lengths are on the device; the
// line is two rounds of the workgroups that the chip holds by the blocks of the LONGEST sequence.  12 heads, lengths
// uniform up to the second figure, blocks of 64 / 128 rows, us: 64 x 512 36.6 / 32.6, 200 x 300 55.4 / 50.8, 64 x 256
// 17.3 / 16.7, 40 x 512 27.3 / 27.4 (beyond the line); 64 x 128 9.1 / 9.1, 20 x 300 9.7 / 10.2, 16 x 512 13.1 / 14.9.
static bool packed_by_128(const AttnArgs &a) {
    return (long)((a.seq_len + 127) / 128) * a.nhead * a.batch >= 2 * 3 * (long)std::max(et_device_cu_count(), 1);
}

// Two groups of waves over the key tiles of a block of 64 query rows, where the chip has no block for its CUs' other
// waves: a wave alone on its SIMD waits out every tile's latencies.  64 wide heads, one group / two, us: 12 blocks of 64
// rows x 16 tiles (1 x 1024) no mask 11.5 / 9.9, padding 14.0 / 10.9, dense 17.1 / 13.1; 2 x 512 7.5 / 7.0, padding 8.5 /
// 7.6, dense 10.2 / 8.8; 1 x 200 dense 6.8 / 6.5, others alike.  With more blocks than CUs only where there are many tiles:
// 2 x 1000 (384 blocks) 14.4 / 13.7, padding 15.8 / 15.2, dense 19.6 / 18.0; 3 x 600 (360) 10.6 / 10.7, 11.7 / 11.7, 13.9 /
// 13.3; 4 x 384 (288) 7.7 / 8.2, 8.9 / 9.1; 4 x 1000 (768) 19.4 / 21.0.  Four groups are not faster anywhere.
static bool two_key_groups(const AttnArgs &a) {
    const long cus = std::max(et_device_cu_count(), 1), tiles = (a.seq_len + AT_KT - 1) / AT_KT;
    return (a.total <= cus && tiles >= 4) || (2 * a.total <= 3 * cus && tiles >= 12);
}

// packed sequences: as many workgroups (4 waves x 16 QS query rows) as the chip holds at once, or fewer: for every XCD as
// many as the blocks of the one with the most pairs.  (An even share of the blocks gives the XCDs with a pair more a second
// round while others idle: one sequence, 12 heads on 8 XCDs, 1024 rows 20.1 -> 11.9 us, padding mask 25.5 -> 14.6, 512
// rows 13.7 -> 8.4, 200 rows 10.8 -> 7.0; from two sequences on the same times.)
template <int HD, bool MASK, int QS = 1, int KS = 1>
static void attn_launch_packed(const AttnArgs &a, hipStream_t st) {
    // (32 query rows per wave with the mask's bookkeeping needed 207 registers, two waves per SIMD: 63 us against 48 us on
    // a batch of 64 sequences of 32..512 rows; without it 154 and three)
    static_assert(QS == 1 || !MASK, "two subtiles a wave: without a mask");
    constexpr size_t lds = attn_lds_bytes<HD, QS, 4 * KS, false, HD, false, KS>();
    constexpr auto kern = &attention_packed_kernel<HD, QS, 4 * KS, MASK, KS>;
    const long resident = (long)std::max(et_device_cu_count(), 1) * packed_on_cu(HD, QS, KS);
    const long wgs = std::min<long>(resident, 8L * a.per_xcd);
    launch_kernel<kern>(dim3((unsigned)((wgs + 7) / 8 * 8)), dim3(256 * KS), lds, st, a);
}

// variant 0: 4 waves x 32 query rows; 1: 8 waves x 16 rows; 2: 4 waves x 16 rows; 3: 4 waves x 16 rows in each of two key
// groups
template <int HD, bool PRUNED, bool SHAREDQK, int HDK = HD>
static void attn_launch_variant(int variant, bool plain, bool no_mask, const AttnArgs &a, hipStream_t st) {
    if constexpr (HD == 64 && HDK == 64 && !PRUNED && !SHAREDQK) {
        if (variant == 3) {
            if (plain)
                attn_launch_two_groups<HD, true, false>(a, st);
            else if (no_mask)
                attn_launch_two_groups<HD, false, false>(a, st);
            else
                attn_launch_two_groups<HD, false, true>(a, st);
            return;
        }
    }
    if constexpr (!PRUNED && !SHAREDQK) {
        if (plain) {
            if (variant == 0)
                attn_launch_one<HD, 2, 4, false, false, true, HDK>(a, st);
            else if (variant == 1)
                attn_launch_one<HD, 1, 8, false, false, true, HDK>(a, st);
            else
                attn_launch_one<HD, 1, 4, false, false, true, HDK>(a, st);
            return;
        }
        // ragged lengths without a mask: the plain form's loop, the last tile with its bounds behind it (12 heads:
        // 2 x 1021 rows 19.5 -> 14.5 us, 14 x 500 22.8 -> 18.9, 8 x 250 8.7 -> 7.2)
        if (no_mask) {
            if (variant == 0)
                attn_launch_one<HD, 2, 4, false, false, false, HDK, false, false>(a, st);
            else if (variant == 1)
                attn_launch_one<HD, 1, 8, false, false, false, HDK, false, false>(a, st);
            else
                attn_launch_one<HD, 1, 4, false, false, false, HDK, false, false>(a, st);
            return;
        }
    }
    if (variant == 0)
        attn_launch_one<HD, 2, 4, PRUNED, SHAREDQK, false, HDK>(a, st);
    else if (variant == 1)
        attn_launch_one<HD, 1, 8, PRUNED, SHAREDQK, false, HDK>(a, st);
    else
        attn_launch_one<HD, 1, 4, PRUNED, SHAREDQK, false, HDK>(a, st);
}

static int g_attn_variant = -1; // et_tuning_set("attn_variant"): -1 = automatic
static int g_attn_packed = 1;   // et_tuning_set("attn_packed"): 0 = packed sequences run one workgroup per possible query block
static int g_attn_vwin = 1;     // et_tuning_set("attn_vwin"): 0 = pruned attention always stages through registers

static float head_scale(int hd) {
    // half(sqrt(1/head_dim)), kernels/attention.cu:126
    return (float)(f16)sqrtf(1.0f / (float)hd);
}

// ---- mask summary: one bit per (16 query rows, 64-key tile) ----------------
// One workgroup of four waves per group of 16 rows, wave w takes the tiles w, w+4, ...; per tile a lane tests 16
// elements (row lane/4, keys 16*(lane%4)..+15: two 16-byte loads where rows are 16-byte aligned) and the wave's
// ballot gives the bit.  (One wave per group with 2-byte loads took 22 us for a 512 x 512 mask, as long as the
// attention launch that the entry point without allocations puts behind it.)
__global__ void __launch_bounds__(256) mask_summary_kernel(const f16 *mask, int seq_len, unsigned *out,
                                                           int words) {
    extern __shared__ unsigned ms_bits[]; // `words` entries
    const int g = blockIdx.x;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int w = threadIdx.x; w < words; w += 256)
        ms_bits[w] = 0;
    __syncthreads();
    const int row = g * 16 + (lane >> 2);
    const int nt = (seq_len + AT_KT - 1) / AT_KT;
    const uint16_t *m = reinterpret_cast<const uint16_t *>(mask);
    const bool vec = (seq_len & 7) == 0 && (reinterpret_cast<uintptr_t>(mask) & 15u) == 0;
    for (int t = wave; t < nt; t += 4) {
        bool nz = false; // anything but +0 / -0
        if (row < seq_len) {
            const int k0 = t * AT_KT + (lane & 3) * 16;
            if (vec && k0 + 16 <= seq_len) {
                const u32x4 *p = reinterpret_cast<const u32x4 *>(m + (size_t)row * seq_len + k0);
                const u32x4 v0 = p[0], v1 = p[1];
                nz = (((v0[0] | v0[1] | v0[2] | v0[3] | v1[0] | v1[1] | v1[2] | v1[3]) & 0x7FFF7FFFu) != 0);
            } else {
                for (int j = 0; j < 16; j++)
                    if (k0 + j < seq_len && (m[(size_t)row * seq_len + k0 + j] & 0x7FFFu) != 0)
                        nz = true;
            }
        }
        if (__builtin_amdgcn_ballot_w64(nz) != 0 && lane == 0)
            atomicOr(&ms_bits[t >> 5], 1u << (t & 31));
    }
    __syncthreads();
    for (int w = threadIdx.x; w < words; w += 256)
        out[(size_t)g * words + w] = ms_bits[w];
}

static int mask_summary_words(int seq_len) { return ((seq_len + AT_KT - 1) / AT_KT + 31) / 32; }

// summaries registered for a mask pointer (et_attention_mask_summary_attach)
struct MaskSummaryEntry {
    const void *mask;
    const unsigned *summary;
    int seq_len;
    bool all_zero; // no bit set: the mask adds nothing anywhere
};
static std::mutex g_msum_mutex;
static std::vector<MaskSummaryEntry> g_msum;

// returns whether the mask is known to be zero everywhere
static bool attach_mask_summary(AttnArgs &a) {
    a.msum = nullptr;
    a.msum_words = 0;
    if (!a.mask)
        return true;
    std::lock_guard<std::mutex> lock(g_msum_mutex);
    for (const MaskSummaryEntry &e : g_msum)
        if (e.mask == a.mask && e.seq_len == a.seq_len) {
            a.msum = e.summary;
            a.msum_words = mask_summary_words(a.seq_len);
            return e.all_zero;
        }
    return false;
}

bool attention_finish_args(AttnArgs &a, int d_model) {
    a.ldo = d_model;
    a.scale = head_scale(d_model / a.nhead);
    return attach_mask_summary(a);
}

// qk_width: columns per head in Q and K (0 = head_dim)
// given_summary: a summary of a.mask supplied by the caller of this function
// (it then replaces the lookup among the attached ones)
static int attention_check(const AttnArgs &a, int d_model, bool sharedqk, const char *who) {
    ET_REQUIRE(a.out && a.V, ET_ERR_INVALID_ARG, "%s: null pointer", who);
    ET_REQUIRE(sharedqk ? a.QK != nullptr : (a.Q && a.K), ET_ERR_INVALID_ARG, "%s: null pointer", who);
    ET_REQUIRE(a.seq_len > 0 && d_model > 0 && a.nhead > 0 && a.batch > 0, ET_ERR_INVALID_ARG,
               "%s: seq_len=%d d_model=%d nhead=%d batch=%d", who, a.seq_len, d_model, a.nhead, a.batch);
    ET_REQUIRE(d_model % a.nhead == 0, ET_ERR_INVALID_ARG, "%s: d_model %% nhead != 0", who);
    const int hd = d_model / a.nhead;
    ET_REQUIRE(hd % 16 == 0 && hd <= 128, ET_ERR_UNSUPPORTED,
               "%s: head_dim %d: multiples of 16 up to 128", who, hd);
    ET_REQUIRE(aligned16(a.out) && aligned16(a.Q) && aligned16(a.K) && aligned16(a.V),
               ET_ERR_ALIGNMENT, "%s: out/Q/K/V must be 16-byte aligned", who);
    return ET_OK;
}

static int attention_dispatch(AttnArgs a, int d_model, bool pruned, bool sharedqk,
                              hipStream_t st, const char *who, int qk_width = 0,
                              const unsigned *given_summary = nullptr) {
    {
        const int rc = attention_check(a, d_model, sharedqk, who);
        if (rc != ET_OK)
            return rc;
    }
    const int hd_data = d_model / a.nhead;
    // Kernels are built for heads of 32, 64 and 128 columns.  Any other multiple
    // of 16 up to 128 (the reference loops over head_dim in steps of 16,
    // kernels/attention.cu:86-90) runs on the register-staged kernel of the next
    // built width as ragged heads: it reads the columns beyond a head's end as
    // zeros and writes none of them.
    const bool odd_width = !(hd_data == 32 || hd_data == 64 || hd_data == 128);
    ET_REQUIRE(!odd_width || (hd_data % 16 == 0 && hd_data > 0 && hd_data < 128 && !sharedqk && !a.qk_head_ptr &&
                              !a.v_head_ptr && !a.cu_seqlens),
               ET_ERR_UNSUPPORTED,
               "%s: head_dim %d: multiples of 16 up to 128 (dense heads, padded batches) or 32 / 64 / 128", who, hd_data);
    const int hd = !odd_width ? hd_data : hd_data < 32 ? 32 : hd_data < 64 ? 64 : 128;
    if (odd_width) {
        pruned = true;
        a.head_width = hd_data;
    }
    if (!pruned) {
        ET_REQUIRE(a.ldq % 8 == 0 && a.ldv % 8 == 0, ET_ERR_ALIGNMENT,
                   "%s: d_model must be a multiple of 8", who);
    }
    a.ldo = d_model;
    a.scale = head_scale(hd_data);
    bool no_mask;
    if (given_summary && a.mask) {
        a.msum = given_summary;
        a.msum_words = mask_summary_words(a.seq_len);
        no_mask = false; // its bits are only known on the device
    } else {
        no_mask = attach_mask_summary(a);
    }
    // 128 query rows per workgroup when that still fills the chip, else 64
    int variant = 0;
    {
        const long wg128 = (long)((a.seq_len + 127) / 128) * a.nhead * a.batch;
        if (wg128 < 512)
            variant = 2;
        if (hd == 128)
            variant = 2;
        if (a.cu_seqlens)
            variant = 2; // packed sequences of different lengths: 64-row blocks waste fewer padded query rows
                         // (64 sequences of 32 to 512 rows: 50 us against 53-57 us with 128-row blocks)
        if (g_attn_variant == 3)
            variant = 2;
        if (g_attn_variant >= 0 && g_attn_variant <= 2 && !(hd == 128 && g_attn_variant == 0))
            variant = g_attn_variant;
    }
    const int QB = variant == 2 ? 64 : 128; // (3: chosen below, from 2)
    const bool plain = no_mask && !a.seq_lens && !a.cu_seqlens && a.seq_len % QB == 0;
    a.nqb = (a.seq_len + QB - 1) / QB;
    a.total = a.nqb * a.nhead * a.batch;
    a.per_xcd = (a.nhead * a.batch + 7) / 8 * a.nqb;
    if (variant == 2 && hd == 64 && hd_data == 64 && !pruned && !sharedqk && !(qk_width && qk_width != hd_data) &&
        (g_attn_variant < 0 ? two_key_groups(a) : g_attn_variant == 3))
        variant = 3;
#define ET_ATTN_CASE(HDV)                                                                         \
    if (hd == HDV) {                                                                              \
        if (sharedqk) attn_launch_variant<HDV, false, true>(variant, false, false, a, st);                     \
        else if (pruned) attn_launch_variant<HDV, true, false>(variant, false, false, a, st);                  \
        else attn_launch_variant<HDV, false, false>(variant, plain, no_mask, a, st);                             \
    }
    if (qk_width && qk_width != hd_data) {
        ET_REQUIRE(qk_width > 0 && qk_width < hd_data && qk_width % 16 == 0 && !sharedqk && !a.qk_head_ptr &&
                       !a.v_head_ptr && !a.cu_seqlens,
                   ET_ERR_UNSUPPORTED, "%s: %d of %d columns per head in Q and K: a multiple of 16 below the head width",
                   who, qk_width, hd_data);
        if (hd == 64 && qk_width == 32 && !pruned) { // the DMA-staged kernel with a 32-wide K tile
            attn_launch_variant<64, false, false, 32>(variant, plain, no_mask, a, st);
            return launch_status(who);
        }
        // any other width: ragged heads on the register-staged kernel
        pruned = true;
        a.qk_width = qk_width;
    }
    // packed sequences: the grid the chip holds, every workgroup walks its share of the query blocks that exist
    // (variant 2 counts the blocks of 64)
    if (a.cu_seqlens && !pruned && !sharedqk && variant >= 2 && a.batch <= 64 * AT_PX && g_attn_packed) {
        if (hd == 32)
            no_mask ? attn_launch_packed<32, false>(a, st) : attn_launch_packed<32, true>(a, st);
        else if (variant == 3)
            no_mask ? attn_launch_packed<64, false, 1, 2>(a, st) : attn_launch_packed<64, true, 1, 2>(a, st);
        else if (hd == 64)
            no_mask ? (packed_by_128(a) ? attn_launch_packed<64, false, 2>(a, st) : attn_launch_packed<64, false>(a, st)) : attn_launch_packed<64, true>(a, st);
        else
            no_mask ? attn_launch_packed<128, false>(a, st) : attn_launch_packed<128, true>(a, st);
        return launch_status(who);
    }
    // dense Q/K with compact V (the reference's pruned wiring): DMA-staged value windows
    if (pruned && hd == 64 && !a.qk_head_ptr && a.v_head_ptr && a.ldq % 8 == 0 && a.ldv % 8 == 0 && a.ldv >= 8 &&
        g_attn_vwin) {
        if (variant == 0 && plain)
            attn_launch_one<64, 2, 4, true, false, true, 64, true>(a, st);
        else if (variant == 0 && no_mask)
            attn_launch_one<64, 2, 4, true, false, false, 64, true, false>(a, st);
        else if (variant == 0)
            attn_launch_one<64, 2, 4, true, false, false, 64, true>(a, st);
        else if (variant == 1)
            attn_launch_one<64, 1, 8, true, false, false, 64, true>(a, st);
        else if (plain)
            attn_launch_one<64, 1, 4, true, false, true, 64, true>(a, st);
        else if (no_mask)
            attn_launch_one<64, 1, 4, true, false, false, 64, true, false>(a, st);
        else
            attn_launch_one<64, 1, 4, true, false, false, 64, true>(a, st);
        return launch_status(who);
    }
    ET_ATTN_CASE(32)
    ET_ATTN_CASE(64)
    ET_ATTN_CASE(128)
#undef ET_ATTN_CASE
    return launch_status(who);
}

void set_attn_variant(int v) { g_attn_variant = v; }
void set_attn_vwin(int v) { g_attn_vwin = v; }
void set_attn_packed(int v) { g_attn_packed = v; }

} // namespace et

extern "C" int et_OTF_attention(void *out, const void *Q, const void *K, const void *V,
                                const void *mask, int seq_len, int d_model, int nhead, int batch,
                                const int *seq_lens, float log2_scale, void *stream) {
    using namespace et;
    AttnArgs a = {};
    a.out = static_cast<f16 *>(out);
    a.Q = static_cast<const f16 *>(Q);
    a.K = static_cast<const f16 *>(K);
    a.V = static_cast<const f16 *>(V);
    a.mask = static_cast<const f16 *>(mask);
    a.seq_lens = seq_lens;
    a.ldq = a.ldv = d_model;
    a.seq_len = seq_len;
    a.nhead = nhead;
    a.batch = batch;
    a.log2_scale = log2_scale;
    return attention_dispatch(a, d_model, false, false, static_cast<hipStream_t>(stream),
                              "et_OTF_attention");
}

// ---- the entry point that allocates nothing --------------------------------
// Its scratch memory is the summary of the mask (one bit per 16 query rows x 64
// keys), which the other entry points keep in a buffer that the caller
// allocates and attaches.  Every GPU holds its own copy of the array at its own
// address: the address is looked up once per device and only that pointer is
// ever handed to a kernel (the array's name is a host-side stand-in).
namespace et {
constexpr int NOALLOC_MAX_SEQ = 4096; // 64 key tiles: what the kernels' two summary words per row group cover
constexpr int NOALLOC_WORDS = (NOALLOC_MAX_SEQ / 16) * 2;
static __device__ __align__(256) unsigned scratch[NOALLOC_WORDS]; // 2 KiB
constexpr int NOALLOC_MAX_DEVICES = 64;
static unsigned *g_scratch_ptr[NOALLOC_MAX_DEVICES];
static std::mutex g_scratch_mutex;

static int noalloc_scratch(unsigned **ptr, hipStream_t st) {
    int dev = -1;
    ET_HIP(stream_device(st, &dev));
    ET_REQUIRE(dev >= 0 && dev < NOALLOC_MAX_DEVICES, ET_ERR_UNSUPPORTED,
               "et_OTF_attention_noalloc: device index %d beyond %d", dev, NOALLOC_MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        const OnDevice on(dev);
        ET_HIP(on.error);
        ET_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        ET_REQUIRE(p != nullptr, ET_ERR_HIP, "et_OTF_attention_noalloc: no address for the scratch array");
        g_scratch_ptr[dev] = static_cast<unsigned *>(p);
    }
    *ptr = g_scratch_ptr[dev];
    return ET_OK;
}
} // namespace et

extern "C" int et_OTF_attention_noalloc(void *out, const void *Q, const void *K, const void *V,
                                        const void *mask, int seq_len, int d_model, int nhead,
                                        int batch, const int *seq_lens, float log2_scale,
                                        void *stream) {
    using namespace et;
    AttnArgs a = {};
    a.out = static_cast<f16 *>(out);
    a.Q = static_cast<const f16 *>(Q);
    a.K = static_cast<const f16 *>(K);
    a.V = static_cast<const f16 *>(V);
    a.mask = static_cast<const f16 *>(mask);
    a.seq_lens = seq_lens;
    a.ldq = a.ldv = d_model;
    a.seq_len = seq_len;
    a.nhead = nhead;
    a.batch = batch;
    a.log2_scale = log2_scale;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (!mask) // nothing to summarise: no scratch memory is touched
        return attention_dispatch(a, d_model, false, false, st, "et_OTF_attention_noalloc");
    {
        // everything the attention launch would refuse is refused before the scratch array is written
        const int rc = attention_check(a, d_model, false, "et_OTF_attention_noalloc");
        if (rc != ET_OK)
            return rc;
    }
    ET_REQUIRE(seq_len <= NOALLOC_MAX_SEQ, ET_ERR_UNSUPPORTED,
               "et_OTF_attention_noalloc: seq_len %d beyond the %d that the static scratch array covers",
               seq_len, NOALLOC_MAX_SEQ);
    unsigned *summary = nullptr;
    const int rc = noalloc_scratch(&summary, st);
    if (rc != ET_OK)
        return rc;
    // every word that the attention kernel reads for this seq_len is written
    // here first, so what an earlier call left in the array does not matter
    launch_kernel<&mask_summary_kernel>(dim3((seq_len + 15) / 16), dim3(256), mask_summary_words(seq_len) * sizeof(unsigned), st, a.mask, seq_len,
                       summary, mask_summary_words(seq_len));
    const int rs = launch_status("et_OTF_attention_noalloc summary launch");
    if (rs != ET_OK)
        return rs;
    return attention_dispatch(a, d_model, false, false, st, "et_OTF_attention_noalloc", 0, summary);
}

extern "C" int et_OTF_attention_summary(void *out, const void *Q, const void *K, const void *V,
                                        const void *mask, const void *mask_summary, int seq_len, int d_model,
                                        int nhead, int batch, const int *seq_lens, float log2_scale,
                                        void *stream) {
    using namespace et;
    AttnArgs a = {};
    a.out = static_cast<f16 *>(out);
    a.Q = static_cast<const f16 *>(Q);
    a.K = static_cast<const f16 *>(K);
    a.V = static_cast<const f16 *>(V);
    a.mask = static_cast<const f16 *>(mask);
    a.seq_lens = seq_lens;
    a.ldq = a.ldv = d_model;
    a.seq_len = seq_len;
    a.nhead = nhead;
    a.batch = batch;
    a.log2_scale = log2_scale;
    ET_REQUIRE(!mask_summary || mask, ET_ERR_INVALID_ARG, "et_OTF_attention_summary: a summary without a mask");
    return attention_dispatch(a, d_model, false, false, static_cast<hipStream_t>(stream), "et_OTF_attention_summary",
                              0, static_cast<const unsigned *>(mask_summary));
}

extern "C" int et_OTF_attention_qk_width(void *out, const void *Q, const void *K, const void *V,
                                         const void *mask, int qk_width, int seq_len, int d_model,
                                         int nhead, int batch, const int *seq_lens, float log2_scale,
                                         void *stream) {
    using namespace et;
    ET_REQUIRE(qk_width > 0 && nhead > 0, ET_ERR_INVALID_ARG, "et_OTF_attention_qk_width: qk_width=%d", qk_width);
    AttnArgs a = {};
    a.out = static_cast<f16 *>(out);
    a.Q = static_cast<const f16 *>(Q);
    a.K = static_cast<const f16 *>(K);
    a.V = static_cast<const f16 *>(V);
    a.mask = static_cast<const f16 *>(mask);
    a.seq_lens = seq_lens;
    a.ldq = nhead * qk_width;
    a.ldv = d_model;
    a.seq_len = seq_len;
    a.nhead = nhead;
    a.batch = batch;
    a.log2_scale = log2_scale;
    return attention_dispatch(a, d_model, false, false, static_cast<hipStream_t>(stream),
                              "et_OTF_attention_qk_width", qk_width);
}

extern "C" int et_OTF_attention_varlen(void *out, const void *Q, const void *K, const void *V,
                                       const void *mask, const int *cu_seqlens, int max_seq_len,
                                       int d_model, int nhead, int batch, float log2_scale,
                                       void *stream) {
    using namespace et;
    ET_REQUIRE(cu_seqlens, ET_ERR_INVALID_ARG, "et_OTF_attention_varlen: null cu_seqlens");
    AttnArgs a = {};
    a.out = static_cast<f16 *>(out);
    a.Q = static_cast<const f16 *>(Q);
    a.K = static_cast<const f16 *>(K);
    a.V = static_cast<const f16 *>(V);
    a.mask = static_cast<const f16 *>(mask);
    a.cu_seqlens = cu_seqlens;
    a.ldq = a.ldv = d_model;
    a.seq_len = max_seq_len;
    a.nhead = nhead;
    a.batch = batch;
    a.log2_scale = log2_scale;
    return attention_dispatch(a, d_model, false, false, static_cast<hipStream_t>(stream),
                              "et_OTF_attention_varlen");
}

extern "C" int et_Prune_attention(void *out, const void *Q, const void *K, const void *V,
                                  const int *qk_head_ptr, int ldqk, const int *v_col_id,
                                  const int *v_head_ptr, int ldv, const void *mask, int seq_len,
                                  int d_model, int nhead, int batch, const int *seq_lens,
                                  float log2_scale, void *stream) {
    using namespace et;
    AttnArgs a = {};
    a.out = static_cast<f16 *>(out);
    a.Q = static_cast<const f16 *>(Q);
    a.K = static_cast<const f16 *>(K);
    a.V = static_cast<const f16 *>(V);
    a.mask = static_cast<const f16 *>(mask);
    a.seq_lens = seq_lens;
    a.qk_head_ptr = qk_head_ptr;
    a.v_col_id = v_col_id;
    a.v_head_ptr = v_head_ptr;
    a.ldq = qk_head_ptr ? ldqk : d_model;
    a.ldv = v_head_ptr ? ldv : d_model;
    ET_REQUIRE(a.ldq > 0 && a.ldv > 0, ET_ERR_INVALID_ARG, "et_Prune_attention: ldqk=%d ldv=%d", ldqk, ldv);
    ET_REQUIRE(!v_col_id || v_head_ptr, ET_ERR_INVALID_ARG,
               "et_Prune_attention: v_col_id given without v_head_ptr");
    a.seq_len = seq_len;
    a.nhead = nhead;
    a.batch = batch;
    a.log2_scale = log2_scale;
    return attention_dispatch(a, d_model, true, false, static_cast<hipStream_t>(stream),
                              "et_Prune_attention");
}

extern "C" int et_sharedQK_attention(void *out, const void *QK, const void *V, const void *mask,
                                     int seq_len, int d_model, int nhead, int batch,
                                     const int *seq_lens, float log2_scale, void *stream) {
    using namespace et;
    AttnArgs a = {};
    a.out = static_cast<f16 *>(out);
    a.QK = static_cast<const f16 *>(QK);
    a.V = static_cast<const f16 *>(V);
    a.mask = static_cast<const f16 *>(mask);
    a.seq_lens = seq_lens;
    a.ldq = a.ldv = d_model;
    a.seq_len = seq_len;
    a.nhead = nhead;
    a.batch = batch;
    a.log2_scale = log2_scale;
    return attention_dispatch(a, d_model, false, true, static_cast<hipStream_t>(stream),
                              "et_sharedQK_attention");
}

extern "C" int et_qk_scores(void *QK, const void *Q, const void *K, int seq_len, int d_model,
                            int nhead, int batch, void *stream) {
    using namespace et;
    ET_REQUIRE(QK && Q && K, ET_ERR_INVALID_ARG, "et_qk_scores: null pointer");
    ET_REQUIRE(seq_len > 0 && d_model > 0 && nhead > 0 && batch > 0 && d_model % nhead == 0,
               ET_ERR_INVALID_ARG, "et_qk_scores: bad sizes");
    const int hd = d_model / nhead;
    ET_REQUIRE(hd == 32 || hd == 64 || hd == 128, ET_ERR_UNSUPPORTED,
               "et_qk_scores: head_dim %d not in {32,64,128}", hd);
    ET_REQUIRE(aligned16(Q) && aligned16(K) && d_model % 8 == 0, ET_ERR_ALIGNMENT,
               "et_qk_scores: Q/K must be 16-byte aligned");
    // scale = half(1/sqrt(head_dim)), encoder/encoder.cu:113
    const float scale = (float)(f16)(1.0f / sqrtf((float)hd));
    const dim3 grid((seq_len + 255) / 256, (seq_len + 63) / 64, batch * nhead), block(256);
    hipStream_t st = static_cast<hipStream_t>(stream);
    f16 *o = static_cast<f16 *>(QK);
    const f16 *q = static_cast<const f16 *>(Q), *k = static_cast<const f16 *>(K);
    if (hd == 32)
        hipLaunchKernelGGL(qk_scores_kernel<32>, grid, block, 0, st, o, q, k, seq_len, d_model, nhead, scale);
    else if (hd == 64)
        hipLaunchKernelGGL(qk_scores_kernel<64>, grid, block, 0, st, o, q, k, seq_len, d_model, nhead, scale);
    else
        hipLaunchKernelGGL(qk_scores_kernel<128>, grid, block, 0, st, o, q, k, seq_len, d_model, nhead, scale);
    return launch_status("et_qk_scores");
}

extern "C" size_t et_attention_mask_summary_bytes(int seq_len) {
    if (seq_len <= 0)
        return 0;
    return (size_t)((seq_len + 15) / 16) * et::mask_summary_words(seq_len) * sizeof(unsigned);
}

extern "C" int et_attention_mask_summary(const void *mask, int seq_len, void *summary, void *stream) {
    using namespace et;
    ET_REQUIRE(mask && summary, ET_ERR_INVALID_ARG, "et_attention_mask_summary: null pointer");
    ET_REQUIRE(seq_len > 0, ET_ERR_INVALID_ARG, "et_attention_mask_summary: seq_len=%d", seq_len);
    launch_kernel<&mask_summary_kernel>(dim3((seq_len + 15) / 16), dim3(256), mask_summary_words(seq_len) * sizeof(unsigned),
                       static_cast<hipStream_t>(stream), static_cast<const f16 *>(mask), seq_len,
                       static_cast<unsigned *>(summary), mask_summary_words(seq_len));
    return launch_status("et_attention_mask_summary launch");
}

extern "C" int et_attention_mask_summary_attach(const void *mask, int seq_len, const void *summary) {
    using namespace et;
    ET_REQUIRE(mask && seq_len > 0, ET_ERR_INVALID_ARG, "et_attention_mask_summary_attach: bad arguments");
    std::lock_guard<std::mutex> lock(g_msum_mutex);
    for (size_t i = 0; i < g_msum.size(); i++)
        if (g_msum[i].mask == mask && g_msum[i].seq_len == seq_len) {
            g_msum.erase(g_msum.begin() + i);
            break;
        }
    if (summary) {
        // read the summary back once: an all-zero mask selects the kernels
        // without any mask handling
        const size_t words = (size_t)((seq_len + 15) / 16) * mask_summary_words(seq_len);
        std::vector<unsigned> h(words);
        ET_HIP(hipDeviceSynchronize());
        ET_HIP(hipMemcpy(h.data(), summary, words * sizeof(unsigned), hipMemcpyDeviceToHost));
        bool all_zero = true;
        for (unsigned w : h)
            all_zero = all_zero && w == 0;
        g_msum.push_back({mask, static_cast<const unsigned *>(summary), seq_len, all_zero});
    }
    return ET_OK;
}

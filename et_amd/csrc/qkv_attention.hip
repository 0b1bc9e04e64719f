// Q/K/V projections and attention of a head in ONE launch, for short sequences
// (steps 1-5 of a layer, encoder/encoder.cu:22-32 of the reference).
//
// Why.  Up to some hundred rows both launches that this one replaces are chains
// of memory round trips behind 2.5 us of launch each, and with many short
// sequences they are the traffic of Q, K and V through the memory system.  A
// head's Q, K and V of up to 128 rows are 60 KB: they fit the LDS next to a
// panel of X, so a workgroup projects one head of one sequence and attends over
// it without writing any of the three.
//
// Mapping.  One workgroup of twelve waves per (sequence, head), qkv_block.h.  X is read once per head; the heads of a
// sequence share an XCD's L2 where that costs no round of workgroups.
#include "qkv_block.h"

#include <algorithm>
#include <cstring>

namespace et {

constexpr int QA_WAVES = 12;
constexpr int QA_PAIRS = 20; // tile pairs of a block-row (154 registers with a mask; twelve waves can have 168)

template <bool MASK>
__global__ void __launch_bounds__(QA_WAVES * 64) qkv_attention_kernel(const QaArgs a) {
    int b, h;
    if (a.by_seq) {
        const QuotRem of = quot_rem(blockIdx.x >> 3, a.nhead, a.nhead_magic);
        h = of.r;
        b = of.q * 8 + (blockIdx.x & 7);
    } else {
        const QuotRem of = quot_rem(blockIdx.x, a.nhead, a.nhead_magic);
        h = of.r;
        b = of.q;
    }
    if (b < a.batch)
        qkv_attention_block<QA_WAVES, QA_PAIRS, MASK, false>(a, b, h);
}

static int g_qkv_attn = -1; // et_tuning_set("qkv_attention"): 0 never, 1 wherever the form exists, -1 automatic
void set_qkv_attention(int v) { g_qkv_attn = v; }

bool qa_shapes(const et_tile_plan *q, const et_tile_plan *k, const et_tile_plan *v, int max_len, int d, int nheads, int pairs) {
    for (const et_tile_plan *p : {q, k, v})
        if (!p || p->in_feat != d || p->out_feat != d || p->nchunk != 1 || p->most_pairs > pairs)
            return false;
    return nheads > 0 && d == nheads * 64 && d <= 1024 && max_len > 0 && max_len <= QA_MOST;
}
void qa_operands(QaArgs &a, const et_tile_plan *q, const et_tile_plan *k, const et_tile_plan *v, int max_len, int d, size_t lds) {
    const et_tile_plan *ps[3] = {q, k, v};
    for (int i = 0; i < 3; i++)
        a.l[i] = QaLinear{ps[i]->d_data, ps[i]->d_cptr, ps[i]->d_row_offset, ps[i]->d_bias, ps[i]->npair};
    a.d = d;
    a.ldx = d + 16;
    a.max_len = max_len;
    a.rows32 = (max_len + 31) / 32 * 32;
    a.ring = qa_ring(d, max_len, lds);
}
} // namespace et

extern "C" int et_qkv_attention_pays(const et_tile_plan *q, const et_tile_plan *k, const et_tile_plan *v, int max_len,
                                     int d_model, int nheads, int batch) {
    using namespace et;
    if (g_qkv_attn == 0 || batch <= 0 || !qa_shapes(q, k, v, max_len, d_model, nheads, QA_PAIRS))
        return 0;
    if (g_qkv_attn == 1)
        return 1;
    // One launch instead of two, but one CU per head: a workgroup takes 5 us for 64 rows and 8 for 128, however many there
    // are, and beyond a round of workgroups (two of the short sequences') the joined projections share W and X better.
    // Longer lists cost it more than the other form, which spreads them over the chip.  Whole layers, two launches / one,
    // us (sequences x rows).  80 % pruned, 768 wide: 8 x 16 28.4 / 24.1, 20 x 33 35.0 / 29.9, 2 x 60 28.4 / 26.5, 20 x 80 51.1 /
    // 41.6, 40 x 80 62.8 / 60.0, 4 x 96 33.1 / 31.3, 12 x 100 45.3 / 39.1, 16 x 128 53.7 / 46.4; beyond the lines 1 x 128 27.8
    // / 30.1, 2 x 100 28.2 / 29.4, 40 x 106 65.0 / 65.9, 64 x 64 62.8 / 63.7, 300 x 16 74 / 83; 1024 wide: 20 x 33 42.2 / 41.5,
    // 12 x 100 54.0 / 49.6.  50 % pruned, 768 wide: 8 x 16 29.1 / 27.0, 20 x 33 40.3 / 37.0, 12 x 100 50.0 / 47.7; beyond: 2 x 60
    // 29.3 / 30.1, 5 x 88 38.7 / 39.1, 40 x 33 48.9 / 50.5; dense: 512 wide 6 x 100 38.2 / 41.3.
    const long wgs = (long)batch * nheads, cus = std::max(et_device_cu_count(), 1);
    const double pairs = 0.5 * std::max(std::max(q->ntile, k->ntile), v->ntile) / (d_model / 16); // of a block-row
    if (pairs <= 8.5)
        return max_len <= 88 ? wgs <= 2 * cus : wgs <= cus && wgs >= cus / 6;
    return pairs <= 13.0 && wgs <= cus && (max_len <= 32 || wgs >= cus / 2);
}

extern "C" int et_qkv_attention(void *out, const void *X, const et_tile_plan *q, const et_tile_plan *k,
                                const et_tile_plan *v, const void *mask, const int *seq_lens, const int *cu_seqlens,
                                int max_len, int seq_len, int d_model, int nheads, int batch, float log2_scale,
                                void *stream) {
    using namespace et;
    ET_REQUIRE(out && X && q && k && v, ET_ERR_INVALID_ARG, "et_qkv_attention: null pointer");
    ET_REQUIRE(batch > 0 && seq_len > 0 && max_len <= seq_len && (cu_seqlens || max_len == seq_len) &&
                   qa_shapes(q, k, v, max_len, d_model, nheads, QA_PAIRS),
               ET_ERR_UNSUPPORTED,
               "et_qkv_attention: heads of 64, up to 1024 columns in one chunk, sequences of up to %d rows", QA_MOST);
    ET_REQUIRE(aligned16(out) && aligned16(X), ET_ERR_ALIGNMENT, "et_qkv_attention: pointers must be 16-byte aligned");
    QaArgs a;
    memset(&a, 0, sizeof(a));
    AttnArgs at = {}; // (head scale and attached mask summary)
    at.mask = static_cast<const f16 *>(mask);
    at.seq_len = seq_len;
    at.nhead = nheads;
    a.mask = attention_finish_args(at, d_model) ? nullptr : at.mask;
    a.scale = at.scale;
    qa_operands(a, q, k, v, max_len, d_model, 160 * 1024);
    a.X = static_cast<const f16 *>(X);
    a.out = static_cast<f16 *>(out);
    a.seq_lens = cu_seqlens ? nullptr : seq_lens;
    a.cu_seqlens = cu_seqlens;
    a.seq_len = seq_len;
    a.nhead = nheads;
    a.batch = batch;
    a.nhead_magic = magic_of(nheads);
    a.log2_scale = log2_scale;
    const size_t lds = qa_lds(a.ring, d_model, max_len);
    {
        // workgroups of a sequence on one XCD: where the sequences divide among the XCDs evenly enough (the registers of
        // twelve waves leave no room for a second workgroup on a CU)
        const int cus = std::max(et_device_cu_count(), 8);
        auto rounds = [&](long wgs, int on) { return (wgs + on - 1) / on; };
        a.by_seq = rounds((batch + 7) / 8 * nheads, cus / 8) <= rounds((long)batch * nheads, cus);
    }
    const int grid = a.by_seq ? (batch + 7) / 8 * 8 * nheads : batch * nheads;
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto launch = [&](auto mask_c) -> int {
        constexpr auto kern = &qkv_attention_kernel<decltype(mask_c)::value>;
        launch_kernel<kern>(dim3(grid), dim3(QA_WAVES * 64), lds, s, a);
        return launch_status("et_qkv_attention launch");
    };
    return a.mask ? launch(std::true_type()) : launch(std::false_type());
}

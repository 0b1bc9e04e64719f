// Row-pruned linear + expansion to model width + skip connection + LayerNorm in
// one launch: out = LayerNorm(scatter(X W^T + bias) + skip), the steps behind
// attention and behind the feed-forward block of a layer whose output and second
// feed-forward linear keep some of their rows (row_mat; the compact result of
// kernels/linear.cu:30-32 of the reference).
//
// Why.  The compact result is narrow - 240 of 768 columns at 70 % - so one
// workgroup holds whole rows of it, and the launch that expanded and normalised
// them (skip_layernorm.hip) did little but wait for them again.
//
// Mapping.  A workgroup of eight waves per 16 * MS rows.  The rows of X come into
// LDS by DMA, the skip rows into registers; a wave makes NB block-rows of 16
// features, W in the plan's tile pairs (a full list: pair j of a block-row is
// columns 32j .. 32j + 31), four pairs of each block-row in flight.  The results
// are rounded to half and scattered over zeroed rows of model width in the
// panel's LDS; then a wave normalises 2 * MS rows, two at a time in 32 lanes each (row after row over 64 lanes a quarter of
// the vector work of a 768-wide row was for lanes without a piece: attention-aware layer 32 x 256 86.8 -> 85.5 us, 4 x 100 33.2 ->
// 32.6).
// What bounds it: one phase after the other in a workgroup - panel, W (370 KB for
// 240 x 768 past every workgroup, 3 us at 64 bytes a clock), LayerNorm (2 us for
// 32 rows on a CU), store.  Linear and expansion + LayerNorm as two launches / this
// one, back to back, us: 768 -> 240 (230 kept): 256 rows 8.9 / 7.5, 4096 11.8 / 9.1,
// 8192 16.8 / 12.5, 16384 25.0 / 21.7; 928 -> 240: 8192 17.6 / 14.0; 624 -> 160: 8192
// 15.7 / 11.2; 768 -> 384: 256 9.2 / 9.3, 8192 22.1 / 15.4, 16384 33.0 / 25.3.  Eight
// pairs in flight instead of four take registers from the second workgroup of a CU:
// 8192 rows 12.7, 16384 25.0.
#include "row_ln.h"
#include "tile_plan.h"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace et {

constexpr int RL_WAVES = 8;
constexpr int RL_DEPTH = 4; // pairs in flight per block-row
constexpr int RL_MAX_NB = 3;

struct RlArgs {
    const f16 *W, *bias, *X, *skip, *gamma, *beta;
    const int *col; // output column of a compact one
    f16 *out;
    int M, K, nbr, ppb, ncol, size, ldx, lde; // ppb: pairs per block-row; ldx, lde: halves per LDS row of X, of the result
    float inv_n;
};

template <int NB, int MS, int NP>
__global__ void __launch_bounds__(RL_WAVES * 64, NB < 3 ? 4 : 2) row_layernorm_kernel(
    // (what the first requests need arrives in registers with the wave)
    const f16 *hot_X, const f16 *hot_W, const f16 *hot_skip, int hot_M, int hot_K, int hot_nbr, int hot_ppb, int hot_size, int hot_ldx,
    const f16 *hot_bias, const RlArgs args) {
    RlArgs a = args;
    a.X = hot_X;
    a.W = hot_W;
    a.skip = hot_skip;
    a.M = hot_M;
    a.K = hot_K;
    a.nbr = hot_nbr;
    a.ppb = hot_ppb;
    a.size = hot_size;
    a.ldx = hot_ldx;
    a.bias = hot_bias;
    extern __shared__ __attribute__((aligned(16))) unsigned char rl_smem[];
    f16 *const xs = reinterpret_cast<f16 *>(rl_smem);
    constexpr int ROWS = 16 * MS / RL_WAVES; // of a wave: wave, wave + 8, ...
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c16 = lane & 15, g4 = lane >> 4, khalf8 = (g4 & 1) * 8, hi = lane >> 5;
    const int m0 = blockIdx.x * 16 * MS;
    const int kpiece = a.K >> 3, npiece = a.size >> 3;
    // (rows that do not exist re-read the last one; they are not written)
#pragma unroll
    for (int k = 0; k < ROWS; k++) {
        const int r = wave + k * RL_WAVES;
        const f16 *src = a.X + (size_t)min(m0 + r, a.M - 1) * a.K;
        if (lane < kpiece)
            load_lds16(src + lane * 8, xs + r * a.ldx);
        if (lane + 64 < kpiece)
            load_lds16(src + (lane + 64) * 8, xs + r * a.ldx + 512);
    }
    // (block-rows beyond the matrix re-read its last one; what comes of them is not written)
    const unsigned lane_w2 = (unsigned)(hi * 256 + c16 * 16 + khalf8) * 2;
    const char *wp[NB];
    f16x8 w[RL_DEPTH][NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
        wp[nb] = reinterpret_cast<const char *>(a.W) + (size_t)min(wave * NB + nb, a.nbr - 1) * a.ppb * 1024;
    auto request = [&](f16x8 (&dst)[NB], int s) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
            dst[nb] = *reinterpret_cast<const f16x8 *>(wp[nb] + (size_t)min(s, a.ppb - 1) * 1024 + lane_w2);
    };
#pragma unroll
    for (int i = 0; i < RL_DEPTH; i++)
        request(w[i], i);
    f16x4 bias[NB];
    int col[NB][4];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const int f = min(wave * NB + nb, a.nbr - 1) * 16 + g4 * 4;
        bias[nb] = *reinterpret_cast<const f16x4 *>(a.bias + f);
#pragma unroll
        for (int r = 0; r < 4; r++)
            col[nb][r] = a.col[min(f + r, a.ncol - 1)];
    }
    // (a pair of rows: 32 lanes each)
    RowPieces<NP> skip[ROWS / 2];
#pragma unroll
    for (int k = 0; k < ROWS / 2; k++)
        skip[k] = row_pieces<NP, 32>(a.skip + (size_t)min(m0 + wave + (2 * k + hi) * RL_WAVES, a.M - 1) * a.size, npiece, lane);
    const char *const xlane = reinterpret_cast<const char *>(xs + c16 * a.ldx + khalf8);
    f32x4 acc[NB][MS];
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
#pragma unroll
        for (int m = 0; m < MS; m++)
            acc[nb][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
    __syncthreads();
    for (int s0 = 0; s0 < a.ppb; s0 += RL_DEPTH) {
#pragma unroll
        for (int i = 0; i < RL_DEPTH; i++)
            if (s0 + i < a.ppb) { // (wave-uniform)
                const int s = s0 + i;
                // (an odd list's last tile stands alone: the zero weights beside it meet its own columns)
                const int k2 = min(s * 32 + hi * 16, a.K - 16) * 2;
                f16x8 x[MS];
#pragma unroll
                for (int m = 0; m < MS; m++)
                    x[m] = *reinterpret_cast<const f16x8 *>(xlane + m * 32 * a.ldx + k2);
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
#pragma unroll
                    for (int m = 0; m < MS; m++)
                        acc[nb][m] = mfma16x16x32(w[i][nb], x[m], acc[nb][m]);
                request(w[i], s + RL_DEPTH);
            }
    }
    const RowPieces<NP> gamma = row_pieces<NP, 32>(a.gamma, npiece, lane), beta = row_pieces<NP, 32>(a.beta, npiece, lane);
    __syncthreads(); // X has been read
#pragma unroll
    for (int k = 0; k < ROWS / 2; k++) {
        RowPieces<NP> zero;
#pragma unroll
        for (int i = 0; i < NP; i++)
            zero.p[i] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
        row_put<NP, 32>(xs + (wave + (2 * k + hi) * RL_WAVES) * a.lde, zero, npiece, lane);
    }
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const int f = (wave * NB + nb) * 16 + g4 * 4;
        const f32x4 b4 = __builtin_convertvector(bias[nb], f32x4);
#pragma unroll
        for (int m = 0; m < MS; m++) {
            const f16x4 v = __builtin_convertvector(acc[nb][m] + b4, f16x4);
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (f + r < a.ncol)
                    xs[(m * 16 + c16) * a.lde + col[nb][r]] = v[r];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ROWS / 2; k++) {
        const int r = wave + (2 * k + hi) * RL_WAVES;
        const RowPieces<NP> v = row_layernorm<NP, 32>(row_pieces<NP, 32>(xs + r * a.lde, npiece, lane), skip[k], gamma, beta, npiece, a.inv_n, lane);
        if (m0 + r < a.M)
            row_put<NP, 32>(a.out + (size_t)(m0 + r) * a.size, v, npiece, lane);
    }
}

static int g_row_ln = 1; // et_tuning_set("row_layernorm"): 0 never
void set_row_layernorm(int v) { g_row_ln = v; }

static size_t rl_lds(int ms, int K, int size) {
    return (size_t)16 * ms * std::max(K + ((K & 31) ? 0 : 16), size + 8) * sizeof(f16);
}
static bool rl_takes(const et_tile_plan *p, int n, int size, int M) {
    // A full list in one chunk, narrow enough for eight waves; with three block-rows a wave the two launches are as quick
    // up to a thousand rows (whole layers, half of the rows kept: 200 rows 35.5 / 36.4 us, 1024 48.2 / 48.1, 4096 73.6 /
    // 71.9).
    if (p->out_feat > RL_WAVES * 2 * 16 && M < 1024)
        return false;
    if (!g_row_ln || n <= 0 || p->nchunk != 1 || p->in_feat > 1024 || p->out_feat > RL_WAVES * RL_MAX_NB * 16 || size > 1024 ||
        p->ntile != p->out_feat / 16 * (p->in_feat / 16))
        return false;
    return true;
}
} // namespace et

extern "C" int et_tile_plan_run_scatter_ln(const et_tile_plan *plan, void *out, const void *X, void *compact, const int *col_id,
                                           int n, const void *skip, const void *gamma, const void *beta, int size, int M,
                                           void *stream) {
    using namespace et;
    ET_REQUIRE(plan && out && X && compact && col_id && skip && gamma && beta, ET_ERR_INVALID_ARG,
               "et_tile_plan_run_scatter_ln: null pointer");
    ET_REQUIRE(M >= 0 && size > 0 && size % 8 == 0 && n >= 0 && n <= plan->out_feat && n <= size, ET_ERR_INVALID_ARG,
               "et_tile_plan_run_scatter_ln: M=%d size=%d n=%d of %d", M, size, n, plan->out_feat);
    ET_REQUIRE(aligned16(out) && aligned16(X) && aligned16(compact) && aligned16(skip) && aligned16(gamma) && aligned16(beta),
               ET_ERR_ALIGNMENT, "et_tile_plan_run_scatter_ln: pointers must be 16-byte aligned");
    if (M == 0)
        return ET_OK;
    if (!rl_takes(plan, n, size, M)) { // the two steps, through the caller's buffer
        const int rc = et_tile_plan_run(plan, compact, X, M, 0, stream);
        return rc != ET_OK ? rc
                           : et_scatter_skip_layernorm(out, compact, col_id, n, plan->out_feat, skip, gamma, beta, M, size, stream);
    }
    RlArgs a;
    memset(&a, 0, sizeof(a));
    a.W = plan->d_data;
    a.bias = plan->d_bias;
    a.X = static_cast<const f16 *>(X);
    a.skip = static_cast<const f16 *>(skip);
    a.gamma = static_cast<const f16 *>(gamma);
    a.beta = static_cast<const f16 *>(beta);
    a.col = col_id;
    a.out = static_cast<f16 *>(out);
    a.M = M;
    a.K = plan->in_feat;
    a.nbr = plan->out_feat / 16;
    a.ppb = (a.K / 16 + 1) / 2;
    a.ncol = n;
    a.size = size;
    a.ldx = a.K + ((a.K & 31) ? 0 : 16); // row stride == 32 (mod 64) bytes: conflict-free
    a.lde = size + 8;
    a.inv_n = 1.0f / (float)size;
    // 16 rows a workgroup while that is one per CU, then 32: one per CU up to 8192 rows, beyond them two share its registers;
    // with three block-rows a wave they do not, and beyond a round 64 rows cost less: 16384 x 768 -> 384 29.4 -> 25.3 us, 8224 rows 23.7 -> 19.1
    // (with two block-rows 16384 rows 21.7 -> 22.1)
    const int nb = (a.nbr + RL_WAVES - 1) / RL_WAVES, cus = std::max(et_device_cu_count(), 1);
    const int ms = M <= 16 * cus ? 1 : M <= 32 * cus || nb < 3 ? 2 : 4;
    const size_t lds = rl_lds(ms, a.K, size);
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto launch = [&](auto nb_c, auto ms_c, auto np_c) -> int {
        constexpr auto kern = &row_layernorm_kernel<decltype(nb_c)::value, decltype(ms_c)::value, decltype(np_c)::value>;
        launch_kernel<kern>(dim3((M + 16 * ms - 1) / (16 * ms)), dim3(RL_WAVES * 64), lds, st, a.X, a.W, a.skip, a.M, a.K,
                           a.nbr, a.ppb, a.size, a.ldx, a.bias, a);
        return launch_status("row linear + LayerNorm launch");
    };
    typedef std::integral_constant<int, 1> c1;
    typedef std::integral_constant<int, 2> c2;
    typedef std::integral_constant<int, 3> c3;
    auto by_np = [&](auto nb_c, auto ms_c) { return size <= 512 ? launch(nb_c, ms_c, c2()) : size <= 768 ? launch(nb_c, ms_c, c3()) : launch(nb_c, ms_c, std::integral_constant<int, 4>()); };
    auto by_ms = [&](auto nb_c) { return ms == 1 ? by_np(nb_c, c1()) : by_np(nb_c, c2()); };
    if (ms == 4)
        return by_np(c3(), std::integral_constant<int, 4>());
    return nb == 1 ? by_ms(c1()) : nb == 2 ? by_ms(c2()) : by_ms(c3());
}

// skip connection + LayerNorm of one row, or two, by one wave, in registers (the math and the order of summation of
// skip_layernorm.hip: the same bits): for kernels that have the rows at hand.
#pragma once
#include "common.h"

namespace et {

// a row of up to LPR * 8 * NP halves in the LPR lanes of a wave, 64 or (two rows at once) 32: a lane's pieces of eight lie at
// lane, lane + LPR, ...; what is behind the row repeats its last piece and is not used
template <int NP> struct RowPieces {
    f16x8 p[NP];
};
template <int NP, int LPR = 64> __device__ __forceinline__ RowPieces<NP> row_pieces(const f16 *row, int npiece, int lane) {
    RowPieces<NP> v;
#pragma unroll
    for (int i = 0; i < NP; i++)
        v.p[i] = *reinterpret_cast<const f16x8 *>(row + min((lane & (LPR - 1)) + LPR * i, npiece - 1) * 8);
    return v;
}
template <int NP, int LPR = 64> __device__ __forceinline__ void row_put(f16 *row, const RowPieces<NP> &v, int npiece, int lane) {
#pragma unroll
    for (int i = 0; i < NP; i++)
        if ((lane & (LPR - 1)) + LPR * i < npiece)
            *reinterpret_cast<f16x8 *>(row + ((lane & (LPR - 1)) + LPR * i) * 8) = v.p[i];
}
template <int NP, int LPR = 64>
__device__ __forceinline__ RowPieces<NP> row_layernorm(RowPieces<NP> y, const RowPieces<NP> &skip, const RowPieces<NP> &gamma,
                                                       const RowPieces<NP> &beta, int npiece, float inv_n, int lane) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    constexpr int HALF = LPR == 32; // (the sums of what a whole wave would hold in its two halves are kept apart: half_wave_sum)
    const int l = lane & (LPR - 1);
    auto row_sum = [](const float (&v)[2]) { return LPR == 32 ? half_wave_sum(v[0], v[1]) : wave_sum(v[0]); };
    // (a half times 1.0 plus a float is one instruction; the multiplier is opaque, or it is a conversion and an addition)
    float one = 1.0f;
    asm("" : "+s"(one));
    float sum[2] = {0.f, 0.f}, var[2] = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NP; i++) {
        y.p[i] += skip.p[i]; // half add, one rounding
        if (l + LPR * i >= npiece)
            y.p[i] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 8; j += 2)
            sum[i & HALF] = __builtin_amdgcn_fdot2(h2{y.p[i][j], y.p[i][j + 1]}, h2{(f16)1, (f16)1}, sum[i & HALF], false);
    }
    const float mean = row_sum(sum) * inv_n;
#pragma unroll
    for (int i = 0; i < NP; i++)
        if (l + LPR * i < npiece) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float d = __builtin_fmaf((float)y.p[i][j], one, -mean);
                var[i & HALF] += d * d;
            }
        }
    const float rstd = __builtin_amdgcn_rsqf(row_sum(var) * inv_n + 1e-6f); // (never a denormal)
    const float shift = -mean * rstd;
#pragma unroll
    for (int i = 0; i < NP; i++)
#pragma unroll
        for (int j = 0; j < 8; j++)
            y.p[i][j] = (f16)(__builtin_fmaf((float)y.p[i][j], rstd, shift) * (float)gamma.p[i][j] + (float)beta.p[i][j]);
    return y;
}

} // namespace et

// What the kernels whose waves share the input channels of one set of results do at their end: add the waves' sums, take the
// statistics, apply the inference epilogue, store.  A lane holds TM channels x TN adjacent positions; wave v finishes the
// FM channels from v * FM on: TM / KSP, or one (then the waves from TM on finish none).
#pragma once
#include "common.hpp"

namespace adder {

// The sums of the KSP waves, added in the order of the waves; smem holds KSP * TM * TN * 64 floats (one wave: not used).
template <int TM, int KSP>
static constexpr int kFinished = TM >= KSP ? TM / KSP : 1;
template <int TM, int TN, int KSP>
__device__ __forceinline__ void add_waves(float *smem, int wave, int lane, const float (&tot)[TM][TN], float (&r)[kFinished<TM, KSP>][TN]) {
    if constexpr (KSP == 1) {
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int t = 0; t < TN; ++t) r[m][t] = tot[m][t];
        return;
    }
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t) smem[((wave * TM + m) * TN + t) * 64 + lane] = tot[m][t];
    __syncthreads();
    constexpr int FM = kFinished<TM, KSP>;
    const int m0 = FM * KSP > TM ? min(wave, TM - 1) : wave * FM;   // (a wave that finishes none repeats the last channel)
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            float v = smem[((m0 + f) * TN + t) * 64 + lane];
#pragma unroll
            for (int k = 1; k < KSP; ++k) v += smem[((k * TM + m0 + f) * TN + t) * 64 + lane];
            r[f][t] = v;
        }
}

// own: bit t of the positions that are this lane's; off: its first one in channel 0 of its image; L: positions per plane.
// stats (nullable): one slot per tile, sums of deviations from a pivot in fp32, moved back to the origin in fp64 (fwd.hip).
// EVAL: bn is applied (float storage).  whole: four positions are always this lane's own.
template <int FM, int TN, bool EVAL, class T>
__device__ __forceinline__ void finish_outputs(float (&r)[FM][TN], unsigned own, int co0, int Co, int L, int off, bool whole,
                                               T *__restrict__ y, double *__restrict__ stats, int tiles, int tile, int lane,
                                               const BnEval &bn) {
    if (stats) {
        const double count = (double)wave_sum_dpp((float)__popc(own));
        float sums[2 * FM], pivot[FM];
#pragma unroll
        for (int f = 0; f < FM; ++f) {
            pivot[f] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(r[f][0])));
            float s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int t = 0; t < TN; ++t)
                if (own >> t & 1) {
                    const float dv = r[f][t] - pivot[f];
                    s1 += dv;
                    s2 = fmaf(dv, dv, s2);
                }
            sums[2 * f] = s1;
            sums[2 * f + 1] = s2;
        }
        if constexpr (FM >= 2) {   // all sums in one reduce-scatter: lane l < 2 FM ends with number j(l), moment j % 2 of channel j / 2
            const float mine = wave_sum_scatter<2 * FM>(sums, lane), other = __shfl_xor(mine, FM, 64);
            const int j = wave_sum_scatter_index<2 * FM>(lane), f = j >> 1;
            float piv = pivot[0];
#pragma unroll
            for (int k = 1; k < FM; ++k) piv = f == k ? pivot[k] : piv;
            const double c = (double)piv;
            if (lane < 2 * FM && co0 + f < Co)
                stats[((size_t)(co0 + f) * tiles + tile) * 2 + (j & 1)] =
                    (j & 1) ? (double)mine + 2.0 * c * (double)other + count * c * c : (double)mine + count * c;
        } else {
            const double d1 = (double)wave_sum_dpp(sums[0]), d2 = (double)wave_sum_dpp(sums[1]), c = (double)pivot[0];
            if (lane == 0 && co0 < Co) {
                double *dst = stats + ((size_t)co0 * tiles + tile) * 2;
                dst[0] = d1 + count * c;
                dst[1] = d2 + 2.0 * c * d1 + count * c * c;
            }
        }
    }
    if constexpr (EVAL) {
        float a[FM][TN];
#pragma unroll
        for (int f = 0; f < FM; ++f) {   // (all loads before the first store: one counter serves both)
#pragma unroll
            for (int t = 0; t < TN; ++t) a[f][t] = 0.f;
            if (bn.res) ld_strip<TN>(bn.res + (size_t)min(co0 + f, Co - 1) * L + off, a[f]);
        }
#pragma unroll
        for (int f = 0; f < FM; ++f) {
            const BnEvalChannel ch(bn, min(co0 + f, Co - 1));
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                r[f][t] = ch(r[f][t]) + a[f][t];
                if (bn.relu) r[f][t] = relu_keep_nan(r[f][t]);
            }
        }
    }
#pragma unroll
    for (int f = 0; f < FM; ++f) {
        if (co0 + f >= Co) break;
        T *dst = y + (size_t)(co0 + f) * L + off;
        if (whole && own) {
            if constexpr (TN == 4 || TN == 2) st_strip<TN>(dst, r[f]);
        } else {
#pragma unroll
            for (int t = 0; t < TN; ++t)
                if (own >> t & 1) stf(dst + t, r[f][t]);
        }
    }
}

}  // namespace adder

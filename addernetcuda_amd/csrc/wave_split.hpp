// What the kernels whose waves share the input channels of one set of results do at their end: add the waves' sums, take the
// statistics, apply the inference epilogue, store.  A lane holds TM channels x TN adjacent positions; wave v finishes the
// FM channels from v * FM on: TM / KSP, or one (then the waves from TM on finish none).
#pragma once
#include "common.hpp"

namespace adder {

// The sums of the KSP waves, added in the order of the waves; smem holds KSP * TM * TN * 64 floats (one wave: not used, unless TURN).
// TURN: a lane's sums are those of positions lane, 64 + lane, ... of the tile; what it gets is those of TN adjacent ones.
template <int TM, int KSP>
static constexpr int kFinished = TM >= KSP ? TM / KSP : 1;
template <int TM, int TN, int KSP, bool TURN = false>
__device__ __forceinline__ void add_waves(float *smem, int wave, int lane, const float (&tot)[TM][TN], float (&r)[kFinished<TM, KSP>][TN]) {
    if constexpr (KSP == 1 && !TURN) {
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
            const int e = TURN ? lane * TN + t : t * 64 + lane;
            float v = smem[(m0 + f) * TN * 64 + e];
#pragma unroll
            for (int k = 1; k < KSP; ++k) v += smem[(k * TM + m0 + f) * TN * 64 + e];
            r[f][t] = v;
        }
}

// own: bit t of the positions that are this lane's; off: its first one in channel 0 of its image; L: positions per plane.
// stats (nullable): one slot per tile, sums of deviations from a pivot in fp32, moved back to the origin in fp64, so that the
// cancellation in E[y*y] - E[y]^2 happens in double precision.
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
        if constexpr (FM >= 2 && FM <= 8) {   // all sums in one reduce-scatter: lane l < 2 FM ends with number j(l), moment j % 2 of channel j / 2
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

// The same for input gradients: a second gradient (gadd, nullable) is added, the first pass of the BatchNorm in front of the layer is
// made where FUSE (the in_* fields of adder_bn_links: one slot of sums per tile; float storage), channels first <= c < Ci of the
// FM from ci0 on are stored.  off: the lane's first position in channel ci0.
template <int FM, int TN, bool FUSE, class T>
__device__ __forceinline__ void finish_grad_x(float (&r)[FM][TN], unsigned own, int ci0, int first, int Ci, int L, int off, bool whole,
                                              const T *__restrict__ x, T *__restrict__ gx, const T *__restrict__ gadd,
                                              const adder_bn_links &bn, int tiles, int tile, int lane) {
    // (all loads before the first store: one counter serves both; channels past Ci read the last one)
    float a[FM][TN];
    if (gadd) {
#pragma unroll
        for (int f = 0; f < FM; ++f) ld_strip<TN>(gadd + off + (size_t)min(f, Ci - 1 - ci0) * L, a[f]);
    }
    if constexpr (FUSE) {
        // x = relu(bn(in_x) [+ residual]): dz = (gx + gadd) * [x > 0] and per channel the sums of dz and dz * xhat.  xhat comes from x
        // where nothing but the ReLU followed the BatchNorm and |gamma| is large enough for the division, else from in_x.
        float xv[FM][TN];
#pragma unroll
        for (int f = 0; f < FM; ++f) ld_strip<TN>(x + off + (size_t)min(f, Ci - 1 - ci0) * L, xv[f]);
#pragma unroll
        for (int f = 0; f < FM; ++f) {
            const int c = min(ci0 + f, Ci - 1);
            const float g = bn.in_gamma ? as_uniform(bn.in_gamma)[c] : 0.f, be = bn.in_gamma ? as_uniform(bn.in_beta)[c] : 0.f;
            const bool from_x = bn.in_gamma && fabsf(g) >= 0x1p-6f * fmaxf(1.f, fabsf(be));
            float bx[TN];
#pragma unroll
            for (int t = 0; t < TN; ++t) bx[t] = xv[f][t];
            if (!from_x) ld_strip<TN>(bn.in_x + off + (size_t)(c - ci0) * L, bx);
            const float centre = from_x ? be : as_uniform(bn.in_mean)[c];
            const float scale = from_x ? __builtin_amdgcn_rcpf(g) : as_uniform(bn.in_rstd)[c];
            float a1 = 0.f, a2 = 0.f;
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                if (gadd) r[f][t] += a[f][t];
                const bool keep = (own >> t & 1) && !(bn.in_relu && !(xv[f][t] > 0.f));
                const float v = keep ? r[f][t] : 0.f;
                r[f][t] = v;
                a1 += v;
                a2 = fmaf(v, bx[t] - centre, a2);
            }
            const float s1 = wave_sum_dpp(a1), s2 = wave_sum_dpp(a2) * scale;
            if (lane == 0 && ci0 + f >= first && ci0 + f < Ci) {
                float *dst = bn.in_part + ((size_t)(ci0 + f) * tiles + tile) * 2;
                dst[0] = s1;
                dst[1] = s2;
            }
        }
    } else if (gadd) {
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int t = 0; t < TN; ++t) r[f][t] += a[f][t];
    }
#pragma unroll
    for (int f = 0; f < FM; ++f) {
        if (ci0 + f < first || ci0 + f >= Ci) continue;
        T *dst = gx + off + (size_t)f * L;
        if (whole && own) {
            if constexpr (TN == 2 || TN == 4) st_strip<TN>(dst, r[f]);
        } else {
#pragma unroll
            for (int t = 0; t < TN; ++t)
                if (own >> t & 1) stf(dst + t, r[f][t]);
        }
    }
}

}  // namespace adder

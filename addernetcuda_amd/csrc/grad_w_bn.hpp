// Shared by the weight-gradient kernels that form gy from the gradient of the BatchNorm behind their layer.
#pragma once
#include "common.hpp"

namespace adder {

// The four coefficients {k, c2, mu, km1} of the BatchNorm behind a layer, gy = k * dz + (c2 * (y - mu) - km1), for the workgroup's
// COB channels, from the sums the consumer's input-gradient kernel left (BnSums): 32 lanes add the slots of one channel, always in the same order, so every
// workgroup that needs a channel arrives at the same bits.  `write`: also store dgamma / dbeta of these channels
// (one workgroup per channel block does).  Stands in for a launch of its own between the two kernels.
template <class G>
__device__ __forceinline__ void bn_coef_from_sums(const BnSums &b, int co0, int Co, float4 *coef, bool write) {
    constexpr int GROUPS = G::NTHREADS / 32;
    constexpr int CHUNK = 16;
    const int sub = threadIdx.x & 31, grp = threadIdx.x >> 5;
    for (int cb = 0; cb < G::COB; cb += GROUPS) {
        const int c = cb + grp;
        if (G::COB % GROUPS == 0 || c < G::COB) {
            const int co = min(co0 + c, Co - 1);
            const float rs = b.rstd[co], gm = b.gamma[co], mu = b.mean[co];
            const float2 *p = reinterpret_cast<const float2 *>(b.part) + (size_t)co * b.slots;
            double s1 = 0.0, s2 = 0.0;
            for (int s0 = sub; s0 < b.slots; s0 += 32 * CHUNK) {   // CHUNK loads in flight, then added in slot order
                float2 v[CHUNK];
#pragma unroll
                for (int j = 0; j < CHUNK; ++j) v[j] = p[min(s0 + 32 * j, b.slots - 1)];   // (unconditional: no waits between them)
#pragma unroll
                for (int j = 0; j < CHUNK; ++j) {
                    const bool in = s0 + 32 * j < b.slots;
                    s1 += in ? (double)v[j].x : 0.0;
                    s2 += in ? (double)v[j].y : 0.0;
                }
            }
#pragma unroll
            for (int m = 16; m >= 1; m >>= 1) {   // (stays inside the 32-lane half)
                s1 += __shfl_xor(s1, m, 64);
                s2 += __shfl_xor(s2, m, 64);
            }
            if (sub == 0) {
                const float m1 = (float)(s1 / b.count), m2 = (float)(s2 / b.count);
                const float k = gm * rs;
                coef[c] = make_float4(k, -k * rs * m2, mu, k * m1);
                if (write && co0 + c < Co) {
                    b.dbeta[co] = (float)s1;
                    b.dgamma[co] = (float)s2;
                }
            }
        }
    }
}

}  // namespace adder

// Forward AdderNet convolution, NCHW in -> NCHW out, implicit im2col.
//   y[n,co,ho,wo] = - sum_{ci,i,j} | w[co,ci,i,j] - xpad[n,ci,ho*s+i-p,wo*s+j-p] |
// Replaces adder_cuda/adder.cu:19-70 (CONV) together with the unfold + permute
// copies of adder.py:32-33,38-39 that feed it.
//
// Which kernel a layer takes, and the one for any layer.  The inner operation is two fp32 VALU instructions per (co,k,position) term
// -- v_sub_f32 d, s_w, v_x ; v_sub_f32 acc, acc, |d| -- and cannot use FMA or MFMA, so the kernels of fwd_nine.hip (3x3, 5x5),
// fwd_tap.hip (1x1) and fwd_tile.hip (with statistics) keep everything else off the vector ALU: lanes own output positions, weights are wave-uniform and arrive
// through the scalar cache as SGPR operands.
#include "common.hpp"

#include <type_traits>

namespace adder {

// ---------------------------------------------------------------------------
// Generic kernel: any kernel size / stride / padding / channel count.
// One output position per lane, TM output channels per lane, input read
// straight from global memory with bounds checks.
// ---------------------------------------------------------------------------
template <int TM, class T = float>
__global__ __launch_bounds__(256) void fwd_generic_kernel(const T *__restrict__ x,
                                                          const float *__restrict__ w,
                                                          T *__restrict__ y, ConvDims d, const BnEval bn) {
    const int total = d.N * d.Ho * d.Wo;
    int pos = blockIdx.x * 256 + threadIdx.x;
    const bool active = pos < total;
    if (!active) pos = total - 1;
    const int wo = pos % d.Wo;
    const int ho = (pos / d.Wo) % d.Ho;
    const int n = pos / (d.Wo * d.Ho);
    const int co0 = blockIdx.y * TM;
    const int K = d.K();
    uniform_f32_ptr wc = as_uniform(w);

    float acc[TM], tot[TM];   // acc: at most 16 channels' taps, tot: the rest (keeps fp32 error small for large K)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[m] = tot[m] = 0.f;

    int wrow[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) wrow[m] = min(co0 + m, d.Co - 1) * K;

    const T *xn = x + (size_t)n * d.Ci * d.H * d.W;
    for (int ci = 0; ci < d.Ci; ++ci) {
        for (int i = 0; i < d.kh; ++i) {
            const int hi = ho * d.stride + i - d.pad;
            const bool hv = hi >= 0 && hi < d.H;
            for (int j = 0; j < d.kw; ++j) {
                const int wi = wo * d.stride + j - d.pad;
                const bool v = hv && wi >= 0 && wi < d.W;
                const float xv = v ? ldf(xn + ((size_t)ci * d.H + hi) * d.W + wi) : 0.f;
                const int k = (ci * d.kh + i) * d.kw + j;
#pragma unroll
                for (int m = 0; m < TM; ++m) acc[m] -= fabsf(wc[wrow[m] + k] - xv);
            }
        }
        if ((ci & 15) == 15 || ci + 1 == d.Ci) {
#pragma unroll
            for (int m = 0; m < TM; ++m) { tot[m] += acc[m]; acc[m] = 0.f; }
        }
    }
    if (active) {
#pragma unroll
        for (int m = 0; m < TM; ++m)
            if (co0 + m < d.Co) {
                const size_t off = (((size_t)n * d.Co + co0 + m) * d.Ho + ho) * d.Wo + wo;
                if (sizeof(T) == 4 && bn.gamma) {
                    tot[m] = BnEvalChannel(bn, co0 + m)(tot[m]);
                    if (bn.res) tot[m] += bn.res[off];
                    if (bn.relu) tot[m] = relu_keep_nan(tot[m]);
                }
                stf(y + off, tot[m]);
            }
    }
}

// Which kernel a forward without statistics takes; y aligned to groups of four.  (The others take bases of any alignment.)
static FwdKernel choose_fwd(const ConvDims &d, bool y_aligned) {
    if (fwd_strided_tile_supported(d) && (d.Ho * d.Wo % 4 != 0 || y_aligned)) return FwdKernel::strided_tile;
    if (fwd_tap_supported(d)) return FwdKernel::tap;
    if (fwd_nine_supported(d)) return FwdKernel::nine;
    return conv1x1_supported(d, nullptr, nullptr) ? FwdKernel::plain_1x1 : FwdKernel::general;
}

int fwd_kernel(const ConvDims &d) {
    const FwdKernel kernel = choose_fwd(d, true);
    const LaneShape shape = kernel == FwdKernel::tap ? fwd_tap_shape(d) : kernel == FwdKernel::nine ? fwd_nine_shape(d) : LaneShape{0, 0, 0};
    return static_cast<int>(kernel) * 100000 + shape.tm * 1000 + shape.tn * 100 + shape.waves;
}

// Both storage types take the same kernels and shapes: the arithmetic, which bounds them, is the same fp32.
// (bfloat16 layers other than 3x3 once went to the generic kernel: 128 -> 512 1x1 @28x28, 32 images, 561 us.)
template <class T>
int launch_fwd(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn) {
    switch (choose_fwd(d, aligned_groups(y))) {
        case FwdKernel::strided_tile: return launch_fwd_strided_tile(x, w, y, d, s, bn);
        case FwdKernel::tap: return launch_fwd_tap(x, w, y, d, s, bn);
        case FwdKernel::nine: return launch_fwd_nine(x, w, y, d, s, bn);
        case FwdKernel::plain_1x1: return launch_fwd_1x1(x, w, y, nullptr, d, s, bn);
        case FwdKernel::general: break;
    }
    constexpr int TM = 8;
    const long total = (long)d.N * d.Ho * d.Wo;
    hipLaunchKernelGGL((fwd_generic_kernel<TM, T>), dim3((unsigned)ceil_div_l(total, 256), ceil_div(d.Co, TM)),
                       dim3(256), 0, s, x, w, y, d, bn);
    return check_launch();
}
template int launch_fwd<float>(const float *, const float *, float *, const ConvDims &, hipStream_t, const BnEval &);
template int launch_fwd<bf16_t>(const bf16_t *, const float *, bf16_t *, const ConvDims &, hipStream_t, const BnEval &);

}  // namespace adder

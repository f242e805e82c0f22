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

// A class of sizes (0 = none): 1..3 3x3 stride 1 by output width, 4..5 3x3 stride 2 (all fwd_nine.hip),
// 6..7 1x1 stride 1 from 64 channels on by plane size, 8..9 1x1 with a stride, 10..13 = 6..9 for channels that are no multiple of 8 (all
// fwd_tap.hip), 14..18 5x5 (stride 1 by output width, then stride 2; fwd_nine.hip)
static int fwd_tiled_variant(const ConvDims &d) {
    if (d.kh == 1 && d.kw == 1 && d.pad == 0 && d.Ci % 4 == 0 && d.Ci >= 64) {
        const int quad = d.Ci % 8 ? 4 : 0, plane = d.Ho * d.Wo;
        const bool wide = ceil_div(plane, 256) * 256 <= ceil_div(plane, 64) * 64;
        if (d.stride == 1) return (wide ? 6 : 7) + quad;
        return (wide ? 8 : 9) + quad;
    }
    if (d.kh == 5 && d.kw == 5 && d.pad == 2) {
        if (d.stride == 1) return d.Wo > 16 ? 14 : (d.Wo > 8 ? 15 : 16);
        if (d.stride == 2) return d.Wo > 8 ? 17 : 18;
        return 0;
    }
    if (d.kh != 3 || d.kw != 3 || d.pad != 1) return 0;
    if (d.stride == 1) return d.Wo > 16 ? 1 : (d.Wo > 8 ? 2 : 3);
    if (d.stride == 2) return d.Wo > 8 ? 4 : 5;
    return 0;
}

// Whether a 3x3 or 1x1 layer has few positions: a class of sizes that fwd_kernel tells apart, and whose statistics are offered for bases of
// any alignment.  fwd_nine.hip and fwd_tap.hip choose their shapes by rules of their own.
static bool few_positions(const ConvDims &d, int variant) {
    if (variant == 0 || variant >= 14 || ceil_div(d.Co, 4) > kMaxGridY) return false;
    const int per_lane = variant >= 3 && variant <= 5 ? 8 : variant == 8 || variant == 9 ? 32 : 16;
    const int chunk = variant == 1 || variant == 4 || variant == 8 || variant == 9 || (variant == 5 && d.Ci >= 128) ? 8 : 16;
    const float terms = (float)d.K() * d.Co * d.N * d.Ho * d.Wo;
    const float tiled = 0.006f * d.K() * per_lane;
    const float share = (float)(ceil_div(ceil_div(d.Ci, chunk), 8) * chunk);
    const float few = 2.f + (d.kh == 3 ? 0.4f * share + terms / 10.9e6f : 0.25f * share + terms / 3.2e6f);
    return few < 0.9f * tiled;
}

// rows per tile (16, 8 or 4) that pad a map of H rows least; the larger tile on a tie
static int rows_per_tile_w32(int H) {
    const int p16 = round_up(H, 16), p8 = round_up(H, 8), p4 = round_up(H, 4);
    return p16 <= p8 && p16 <= p4 ? 16 : (p8 <= p4 ? 8 : 4);
}

// Which kernel launch_fwd runs without statistics and for bases aligned to groups of four: 0 general, 1 plain 1x1, 2 few
// positions, else 10 * variant + a class of sizes (3x3 on wide maps: whole groups of 16 / 8 / 4 rows 0 / 1 / 2; 5: channels from 128 on 1).
// One kernel, with shapes of its own, runs all the classes of the 3x3 layers (fwd_nine.hip), and one those of the 1x1 layers
// (fwd_tap.hip; plain ones, 1, too unless they are wide maps of few channels), number 2 included.
int fwd_kernel(const ConvDims &d) {
    const int variant = fwd_tiled_variant(d);
    if (few_positions(d, variant)) return 2;
    if (variant == 0) return conv1x1_supported(d, nullptr, nullptr) ? 1 : 0;
    const int rows = rows_per_tile_w32(d.Ho);
    return 10 * variant + (variant == 1 ? (rows == 16 ? 0 : rows == 8 ? 1 : 2) : variant == 5 && d.Ci >= 128 ? 1 : 0);
}

// Both storage types take the same kernels and shapes: the arithmetic, which bounds them, is the same fp32.
// (bfloat16 layers other than 3x3 once went to the generic kernel: 128 -> 512 1x1 @28x28, 32 images, 561 us.)
template <class T>
int launch_fwd(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn) {
    if (fwd_strided_tile_supported(d) && (d.Ho * d.Wo % 4 != 0 || aligned_groups(y))) return launch_fwd_strided_tile(x, w, y, d, s, bn);
    if (fwd_tap_supported(d)) return launch_fwd_tap(x, w, y, d, s, bn);
    if (fwd_nine_supported(d)) return launch_fwd_nine(x, w, y, d, s, bn);
    if (conv1x1_supported(d, x, y)) return launch_fwd_1x1(x, w, y, nullptr, d, s, bn);
    constexpr int TM = 8;
    const long total = (long)d.N * d.Ho * d.Wo;
    hipLaunchKernelGGL((fwd_generic_kernel<TM, T>), dim3((unsigned)ceil_div_l(total, 256), ceil_div(d.Co, TM)),
                       dim3(256), 0, s, x, w, y, d, bn);
    return check_launch();
}
template int launch_fwd<float>(const float *, const float *, float *, const ConvDims &, hipStream_t, const BnEval &);
template int launch_fwd<bf16_t>(const bf16_t *, const float *, bf16_t *, const ConvDims &, hipStream_t, const BnEval &);

}  // namespace adder

// Forward AdderNet convolution, NCHW in -> NCHW out, implicit im2col.
//   y[n,co,ho,wo] = - sum_{ci,i,j} | w[co,ci,i,j] - xpad[n,ci,ho*s+i-p,wo*s+j-p] |
// Replaces adder_cuda/adder.cu:19-70 (CONV) together with the unfold + permute
// copies of adder.py:32-33,38-39 that feed it.
//
// The inner operation is two fp32 VALU instructions per (co,k,position) term
// -- v_sub_f32 d, s_w, v_x ; v_sub_f32 acc, acc, |d| -- and cannot use FMA or
// MFMA, so the kernels are built to keep everything else off the vector ALU:
//   * lanes own output positions, weights are wave-uniform and arrive through
//     the scalar cache as SGPR operands (no VGPRs, no LDS bandwidth);
//   * the haloed input tile of a workgroup is staged once in LDS with the
//     padding zeros materialised, and each lane reads its (TN+2)-wide strips
//     with ds_read_b128/b64 at immediate offsets;
//   * each lane keeps TM x TN accumulators so one strip read feeds 9*TM*TN terms.
#include "common.hpp"
#include "tile3x3.hpp"

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

// ---------------------------------------------------------------------------
// Tiled kernel for 5x5 / pad 2, stride S = 1 or 2, and single taps with a stride.
//
// A workgroup owns NIMG images x a TH x TW patch of output positions and
// TM*COW output channels.  TW = TN*SPR: each lane owns a strip of TN adjacent
// outputs in one row, SPR strips side by side.  The 64*POSW position lanes are
// replicated COW times, each replica ("co-wave group") taking its own TM
// output channels and sharing the LDS tile.
//
// LDS tile: [img][cc][TH+2][PITCH] floats, double buffered over chunks of CC
// input channels.  Column 0 of a row is input column w0*S-1, so a lane's strip
// starts at column strip*TN*S, which is 16-byte aligned when TN*S is a multiple of 4.
// ---------------------------------------------------------------------------
// T: storage type of x and y (float, or bf16_t for the reduced-storage mode); the arithmetic is fp32 either way.
// EVAL: bn is applied to the results (float storage; an instance of its own, so that the others keep their registers).
template <class C, bool VEC, class T, bool EVAL>
__global__ __launch_bounds__(C::NTHREADS) void fwd_3x3_kernel(const T *__restrict__ x,
                                                                const float *__restrict__ w,
                                                                T *__restrict__ y,
                                                                double *__restrict__ stats, int N, int Ci,
                                                                int H, int W, int Co, int Ho, int Wo,
                                                                int tilesH, int tilesW,
                                                                const BnEval bn) {
    constexpr int TN = C::TN, TM = C::TM, CQ = C::CQ, S = C::S, STRIP = C::STRIP, KS = C::KS, KK = C::KK;
    extern __shared__ __align__(16) float smem[];

    int b = blockIdx.x;
    const int tw = b % tilesW; b /= tilesW;
    const int th = b % tilesH; b /= tilesH;
    const int n0 = b * C::NIMG;
    const int h0 = th * C::TH, w0 = tw * C::TW;

    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int pw = wave % C::POSW, cw = wave / C::POSW;
    int p = pw * 64 + lane;
    const bool lane_ok = p < C::LANES;
    if (!lane_ok) p = C::LANES - 1;
    const int strip = p % C::SPR;
    const int row = (p / C::SPR) % C::TH;
    const int img = p / (C::SPR * C::TH);
    const int co_base = (blockIdx.y * C::COW + cw) * TM;
    const int K = Ci * KK;
    uniform_f32_ptr wc = as_uniform(w);

    // wave-uniform weight row offsets (clamped so tail channels read valid memory)
    int wrow[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m)
        wrow[m] = __builtin_amdgcn_readfirstlane(min(co_base + m, Co - 1) * K);
    // two-level sum: `acc` collects one channel chunk (<= 9*CC terms), `tot` the chunks, so the
    // rounding error grows with the square roots of the two lengths instead of with K
    float acc[TM][TN], tot[TM][TN];
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t) acc[m][t] = tot[m][t] = 0.f;

    const int lane_off = img * C::CC * C::PLANE + row * S * C::PITCH + strip * TN * S;
    const int nchunks = ceil_div(Ci, C::CC);

    TileStage<typename C::Patch> st;
    tile_fetch<typename C::Patch, VEC, false, T>(st, x, 0, Ci, n0, N, h0 * S - C::PAD, w0 * S, H, W);
    {   // this workgroup's output channels: one contiguous run of weights
        const int co_blk = blockIdx.y * C::COW * TM;
        l2_warm(w + (size_t)co_blk * K, 1, 0, min(C::COW * TM, Co - co_blk) * K);
    }
    tile_commit<typename C::Patch>(st, smem);
    __syncthreads();

    for (int c = 0; c < nchunks; ++c) {
        const int ci0 = c * C::CC;
        if (c + 1 < nchunks) tile_fetch<typename C::Patch, VEC, false, T>(st, x, ci0 + C::CC, Ci, n0, N, h0 * S - C::PAD, w0 * S, H, W);

        const float *lbase = smem + (c & 1) * C::BUF + lane_off;
        const int ccnt = min(C::CC, Ci - ci0);
        // Software pipeline over the input channels of the chunk: the strips of channel
        // group cc+CQ and the weights of the next output channel are requested right after
        // the first subtract of the current one, i.e. after the wait for the current
        // operands and with the rest of the arithmetic still ahead to hide the latency.
        float xr[2][CQ][KS][STRIP];
        float wv[2][CQ * KK];
#pragma unroll
        for (int q = 0; q < CQ; ++q)
#pragma unroll
            for (int i = 0; i < KS; ++i)
                lds_read_strip<STRIP, C::STRIP_ALIGN>(lbase + q * C::PLANE + i * C::PITCH, xr[0][q][i]);
#pragma unroll
        for (int e = 0; e < CQ * KK; ++e) wv[0][e] = wc[wrow[0] + ci0 * KK + e];

        auto half = [&](const int cc, const int cur) {
            // cur = 0/1: which xr buffer holds channel group cc
            const int kofs = (ci0 + cc) * KK;
            const bool more = cc + CQ < ccnt;
            const int knext = more ? kofs + CQ * KK : kofs;  // clamped: stays inside the weight row
#pragma unroll
            for (int m = 0; m < TM; ++m) {
#pragma unroll
                for (int idx = 0; idx < CQ * KK * TN; ++idx) {
                    const int t = idx % TN, j = (idx / TN) % KS, i = (idx / TN / KS) % KS, q = idx / TN / KK;
                    acc[m][t] -= fabsf(wv[m & 1][q * KK + i * KS + j] - xr[cur][q][i][t * S + j]);
                    if (idx == 0) {
                        __builtin_amdgcn_sched_barrier(0);
                        if (m + 1 < TM) {
#pragma unroll
                            for (int e = 0; e < CQ * KK; ++e) wv[(m + 1) & 1][e] = wc[wrow[m + 1] + kofs + e];
                        } else {
#pragma unroll
                            for (int e = 0; e < CQ * KK; ++e) wv[(m + 1) & 1][e] = wc[wrow[0] + knext + e];
                        }
                        if (m == 0 && more) {
#pragma unroll
                            for (int q2 = 0; q2 < CQ; ++q2)
#pragma unroll
                                for (int i2 = 0; i2 < KS; ++i2)
                                    lds_read_strip<STRIP, C::STRIP_ALIGN>(
                                        lbase + (cc + CQ + q2) * C::PLANE + i2 * C::PITCH, xr[cur ^ 1][q2][i2]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        };
        static_assert(TM % 2 == 0, "weight double buffer assumes an even number of channels per lane");
#pragma unroll 1
        for (int cc = 0; cc < ccnt; cc += 2 * CQ) {
            half(cc, 0);
            if (cc + CQ < ccnt) half(cc + CQ, 1);
        }

        // (25 taps: a chunk is 200 terms already.  Of one-signed terms n2 sums of n1 round to sqrt(n1 / n2 + n2), which for more
        // than 34 chunks is less with two of them per sum: 813 channels 1.6e-7 -> 1.2e-7 of the result)
        if (KS != 5 || nchunks <= 34 || (c & 1) || c + 1 == nchunks) {
#pragma unroll
            for (int m = 0; m < TM; ++m)
#pragma unroll
                for (int t = 0; t < TN; ++t) { tot[m][t] += acc[m][t]; acc[m][t] = 0.f; }
        }

        if (c + 1 < nchunks) tile_commit<typename C::Patch>(st, smem + ((c + 1) & 1) * C::BUF);
        __syncthreads();
    }

    const int n = n0 + img, ho = h0 + row, wo = w0 + strip * TN;
    if (stats) {
        // BatchNorm statistics of the layer's output on the way out: per wave and output channel the sums of
        // y and y*y over the wave's valid positions, in the partial-sum layout of the BatchNorm kernels
        // (slot = position wave of this launch, stats[(co * slots + slot) * 2 + {0, 1}]).
        // The lanes sum deviations from a pivot (lane 0's first value) in fp32 and lane 0 moves the sums back
        // to the origin in fp64, so the cancellation in E[y*y] - E[y]^2 happens in double precision.
        const bool row_ok = lane_ok && n < N && ho < Ho;
        const int slots = gridDim.x * C::POSW, slot = blockIdx.x * C::POSW + pw;
        float cnt = 0.f;
#pragma unroll
        for (int t = 0; t < TN; ++t) cnt += (row_ok && wo + t < Wo) ? 1.f : 0.f;
        const double count = (double)wave_sum_dpp(cnt);
        if constexpr (TM == 2 || TM == 4 || TM == 8) {
            // all 2 TM sums of the wave in one reduce-scatter: lane l < 2 TM ends with sum number j(l) (channel j / 2,
            // first or second moment j % 2), fetches the other moment of its channel from the lane that holds it,
            // and moves its own one back to the origin
            float sums[2 * TM], pivot[TM];
#pragma unroll
            for (int m = 0; m < TM; ++m) {
                pivot[m] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(tot[m][0])));
                float s1 = 0.f, s2 = 0.f;
#pragma unroll
                for (int t = 0; t < TN; ++t)
                    if (row_ok && wo + t < Wo) {
                        const float dv = tot[m][t] - pivot[m];
                        s1 += dv;
                        s2 = fmaf(dv, dv, s2);
                    }
                sums[2 * m] = s1;
                sums[2 * m + 1] = s2;
            }
            const float mine = wave_sum_scatter<2 * TM>(sums, lane);
            constexpr int TOP = TM;   // lane bit that j % 2 comes from: j is the bit reversal of the lane
            const float other = __shfl_xor(mine, TOP, 64);
            const int j = wave_sum_scatter_index<2 * TM>(lane), m = j >> 1;
            float piv = pivot[0];
#pragma unroll
            for (int k = 1; k < TM; ++k) piv = m == k ? pivot[k] : piv;
            const double c = (double)piv;
            const int co = co_base + m;
            if (lane < 2 * TM && co < Co) {
                // j % 2 == 0: sum of y = d1 + n c;  else: sum of y*y = d2 + 2 c d1 + n c*c
                const double v = (j & 1) ? (double)mine + 2.0 * c * (double)other + count * c * c : (double)mine + count * c;
                stats[((size_t)co * slots + slot) * 2 + (j & 1)] = v;
            }
        } else {
#pragma unroll
            for (int m = 0; m < TM; ++m) {
                const float pivot = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(tot[m][0])));
                float s1 = 0.f, s2 = 0.f;
#pragma unroll
                for (int t = 0; t < TN; ++t)
                    if (row_ok && wo + t < Wo) {
                        const float dv = tot[m][t] - pivot;
                        s1 += dv;
                        s2 = fmaf(dv, dv, s2);
                    }
                const double d1 = (double)wave_sum_dpp(s1), d2 = (double)wave_sum_dpp(s2), c = (double)pivot;
                const int co = co_base + m;
                if (lane == 0 && co < Co) {
                    stats[((size_t)co * slots + slot) * 2] = d1 + count * c;
                    stats[((size_t)co * slots + slot) * 2 + 1] = d2 + 2.0 * c * d1 + count * c * c;
                }
            }
        }
    }
    if (lane_ok && n < N && ho < Ho) {
        const bool vec = TN % 4 == 0 && (Wo & 3) == 0 && wo + TN <= Wo;
        if constexpr (EVAL) {
            static_assert(sizeof(T) == 4, "inference epilogue: float storage");
            // Inference: the BatchNorm behind the layer, the shortcut and the ReLU on the way out instead of three more passes
            // over the map (two launches and a fill for the BatchNorm, one each for add and ReLU): ResNet-50, 32 images,
            // 9.53 -> 8.31 ms, of which 1.65 ms were those passes; ResNet-20, one image, 90 -> 25 launches, 870 -> 470 us.
            {
                float r[TM][TN];
#pragma unroll
                for (int m = 0; m < TM; ++m) {   // (all loads before the first store: one counter serves both)
                    const float *src = bn.res + (((size_t)n * Co + min(co_base + m, Co - 1)) * Ho + ho) * Wo + wo;
#pragma unroll
                    for (int t = 0; t < TN; ++t) r[m][t] = 0.f;
                    if (bn.res && vec && bn.res_vec) {
                        if constexpr (TN % 4 == 0) global_read_strip<TN, 4>(src, r[m]);
                    } else if (bn.res) {
#pragma unroll
                        for (int t = 0; t < TN; ++t)
                            if (wo + t < Wo) r[m][t] = src[t];
                    }
                }
#pragma unroll
                for (int m = 0; m < TM; ++m) {
                    const BnEvalChannel ch(bn, min(co_base + m, Co - 1));
#pragma unroll
                    for (int t = 0; t < TN; ++t) {
                        tot[m][t] = ch(tot[m][t]) + r[m][t];
                        if (bn.relu) tot[m][t] = relu_keep_nan(tot[m][t]);
                    }
                }
            }
        }
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            const int co = co_base + m;
            if (co < Co) {
                T *dst = y + (((size_t)n * Co + co) * Ho + ho) * Wo + wo;
                if (vec) {
#pragma unroll
                    for (int t = 0; t + 3 < TN; t += 4)
                        stf4(dst + t, make_float4(tot[m][t], tot[m][t + 1], tot[m][t + 2], tot[m][t + 3]));
                } else {
#pragma unroll
                    for (int t = 0; t < TN; ++t)
                        if (wo + t < Wo) stf(dst + t, tot[m][t]);
                }
            }
        }
    }
}

template <class C, bool VEC, class T>
static int launch_fwd_3x3_v(const T *x, const float *w, T *y, double *stats, const ConvDims &d,
                            hipStream_t s, const BnEval &bn) {
    const int tilesH = ceil_div(d.Ho, C::TH), tilesW = ceil_div(d.Wo, C::TW);
    const long gx = (long)ceil_div(d.N, C::NIMG) * tilesH * tilesW;
    const int gy = ceil_div(d.Co, C::TM * C::COW);
    if (gx > 0x7fffffffL) return ADDER_ERR_TOO_LARGE;
    auto launch = [&](auto eval) {
        constexpr bool EVAL = decltype(eval)::value;
        if (int rc = allow_dynamic_lds<&fwd_3x3_kernel<C, VEC, T, EVAL>>(C::LDS_BYTES)) return rc;
        hipLaunchKernelGGL((fwd_3x3_kernel<C, VEC, T, EVAL>), dim3((unsigned)gx, gy), dim3(C::NTHREADS),
                           C::LDS_BYTES, s, x, w, y, stats, d.N, d.Ci, d.H, d.W, d.Co, d.Ho, d.Wo, tilesH, tilesW, bn);
        return check_launch();
    };
    if constexpr (sizeof(T) == 4) {
        if (bn.gamma) return launch(std::true_type{});
    }
    return launch(std::false_type{});
}

template <class C, class T = float>
static int launch_fwd_3x3(const T *x, const float *w, T *y, double *stats, const ConvDims &d,
                          hipStream_t s, const BnEval &bn) {
    // element-wise tile loads when the rows of the staged tensor are not whole groups of four
    if (d.W % 4 == 0) return launch_fwd_3x3_v<C, true, T>(x, w, y, stats, d, s, bn);
    return launch_fwd_3x3_v<C, false, T>(x, w, y, stats, d, s, bn);
}

// 5x5 taps: a unit is one output channel x one input channel as well (25 weights, 50*TN vector instructions); five
// strips of eight values per buffer leave room for two output channels per lane.  Two vector instructions per term
// bound it: 32 -> 64 @16x16, 64 images (0.84e9 terms, 27 us at the issue ceiling): generic kernel 247 us, this 40 us.
using Fwd5W32   = Tile3x3Cfg<4, 8, 8, 1, 2, 8, 8, 1, 1, 5>;     // 8 rows of one image x 16 channels
using Fwd5W16   = Tile3x3Cfg<4, 4, 16, 1, 2, 8, 8, 1, 1, 5>;    // outputs 9..16 wide: one image x 16 channels
using Fwd5W8    = Tile3x3Cfg<4, 2, 8, 4, 2, 8, 8, 1, 1, 5>;     // outputs up to 8 wide: four images x 16 channels
using Fwd5W16S2 = Tile3x3Cfg<2, 8, 8, 1, 2, 8, 8, 1, 2, 5>;     // stride 2: 8 rows x 16 outputs of one image
using Fwd5W8S2  = Tile3x3Cfg<2, 4, 8, 2, 2, 8, 8, 1, 2, 5>;     // stride 2, outputs up to 8 wide: two images

// which tiled kernel serves these dimensions (0 = none): 1..3 3x3 stride 1 by output width, 4..5 3x3 stride 2 (all fwd_nine.hip),
// 6..7 1x1 stride 1 from 64 channels on by plane size, 8..9 1x1 with a stride, 10..13 = 6..9 for channels that are no multiple of 8 (all
// fwd_tap.hip), 14..18 5x5 (stride 1 by output width, then stride 2)
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

// A strided 3x3 / pad 1 layer and the strided 1x1 / pad 0 layer beside it (same x, same Co, Ho, Wo) in one launch;
// d describes the 3x3 layer.  Both outputs with their statistics (fwd_stats_slots(d) slots each).  Rows of whole
// float4 groups only; ADDER_ERR_UNSUPPORTED otherwise.
bool fwd_pair_supported(const ConvDims &d) {
    return fwd_nine_supported(d) && d.stride == 2 && d.W % 4 == 0 && d.H % 2 == 0;
}

int launch_fwd_pair(const float *x, const float *w, const float *w_side, float *y, float *y_side, double *stats,
                    double *stats_side, const ConvDims &d, hipStream_t s) {
    if (!fwd_pair_supported(d)) return ADDER_ERR_UNSUPPORTED;
    return launch_fwd_nine<float>(x, w, y, stats, d, s, kNoBnEval, false, w_side, y_side, stats_side);
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

int fwd_stats_slots(const ConvDims &d) {
    if (fwd_tap_supported(d)) return d.stride <= 2 || fwd_tiled_variant(d) ? fwd_tap_stats_slots(d) : 0;
    if (fwd_nine_supported(d)) return fwd_nine_stats_slots(d);
    return conv1x1_supported(d, nullptr, nullptr) ? fwd_1x1_stats_slots(d) : 0;
}

// stats (nullable): per-channel partial sums of y and y*y, fwd_stats_slots(d) > 0 slots per channel.
// Both storage types take the same kernels and tile shapes: the arithmetic, which bounds them, is the same fp32.
// (bfloat16 layers other than 3x3 once went to the generic kernel: 128 -> 512 1x1 @28x28, 32 images, 561 us.)
template <class T>
int launch_fwd(const T *x, const float *w, T *y, double *stats, const ConvDims &d, hipStream_t s, const BnEval &bn) {
    // rows that are whole groups of four are moved as such and need bases aligned to a group
    const bool rows_ok = (d.W % 4 != 0 || aligned_groups(x)) && (d.Wo % 4 != 0 || aligned_groups(y));
    const int variant = fwd_tiled_variant(d);
    const bool few = few_positions(d, variant);
    if (fwd_tap_supported(d)) {
        // (it takes bases of any alignment; from 64 channels on statistics for planes of whole groups are offered for aligned ones only, below
        // for strides up to two)
        const bool aligned = (d.stride > 1 || aligned_groups(x)) && aligned_groups(y);
        if (stats && (variant ? !few && d.Ho * d.Wo % 4 == 0 && !aligned : d.stride > 2)) return ADDER_ERR_UNSUPPORTED;
        return launch_fwd_tap(x, w, y, stats, d, s, bn);
    }
    if (fwd_nine_supported(d)) {
        if (stats && !rows_ok) return ADDER_ERR_UNSUPPORTED;   // (it takes bases of any alignment; statistics are offered for aligned ones)
        return launch_fwd_nine(x, w, y, stats, d, s, bn);
    }
    if (rows_ok && !stats) {   // 5x5 taps; statistics are offered for 3x3 and 1x1 layers
        switch (variant) {
            case 14: return launch_fwd_3x3<Fwd5W32>(x, w, y, stats, d, s, bn);
            case 15: return launch_fwd_3x3<Fwd5W16>(x, w, y, stats, d, s, bn);
            case 16: return launch_fwd_3x3<Fwd5W8>(x, w, y, stats, d, s, bn);
            case 17: return launch_fwd_3x3<Fwd5W16S2>(x, w, y, stats, d, s, bn);
            case 18: return launch_fwd_3x3<Fwd5W8S2>(x, w, y, stats, d, s, bn);
            default: break;
        }
    }
    if (conv1x1_supported(d, x, y)) return launch_fwd_1x1(x, w, y, stats, d, s, bn);
    if (stats) return ADDER_ERR_UNSUPPORTED;   // the generic kernel has no statistics epilogue
    constexpr int TM = 8;
    const long total = (long)d.N * d.Ho * d.Wo;
    hipLaunchKernelGGL((fwd_generic_kernel<TM, T>), dim3((unsigned)ceil_div_l(total, 256), ceil_div(d.Co, TM)),
                       dim3(256), 0, s, x, w, y, d, bn);
    return check_launch();
}
template int launch_fwd<float>(const float *, const float *, float *, double *, const ConvDims &, hipStream_t, const BnEval &);
template int launch_fwd<bf16_t>(const bf16_t *, const float *, bf16_t *, double *, const ConvDims &, hipStream_t,
                                const BnEval &);

// An ordinary convolution y = sum w * x through the 3x3 forward kernel: 3x3 / stride 1 / pad 1 only
// (ADDER_ERR_UNSUPPORTED elsewhere).  stats as in launch_fwd; the slot count is fwd_stats_slots(d).
int launch_mulconv_fwd(const float *x, const float *w, float *y, double *stats, const ConvDims &d, hipStream_t s) {
    const bool ok = d.kh == 3 && d.kw == 3 && d.pad == 1 && d.stride == 1 &&
                    (d.W % 4 != 0 || ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15) == 0);
    if (!ok) return ADDER_ERR_UNSUPPORTED;
    if (!fwd_nine_supported(d)) return ADDER_ERR_UNSUPPORTED;
    return launch_fwd_nine<float>(x, w, y, stats, d, s, kNoBnEval, true);
}

}  // namespace adder

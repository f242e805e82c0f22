// Forwards with the BatchNorm statistics of their output, and the ordinary convolution of a network's stem: 3x3 / pad 1 of stride 1
// or 2 and 1x1 / pad 0, float storage, tiles of x in LDS.  The forwards without statistics are those of fwd_nine.hip and fwd_tap.hip,
// which have the same bits: every result adds its channels' terms in chunks (fwd_chunk) and the chunks in channel order.
//
// Why the tiles: a slot of statistics sums the results of one wave, and the strips of those kernels, which line up over all images,
// group the results otherwise than a tile does.  The sums then differ in their last bits, the normalised maps behind them with them,
// and a deep network amplifies that: the logits of an untrained ResNet-50 whose BatchNorm statistics came from either grouping lie up to
// 0.07 of their root mean square apart.  So the grouping stays the tiles' whichever kernel makes the results: launches that leave the
// tiles half empty run the kernel without tiles, and tile_stats_kernel sums its y as the tiles would have (statistics_apart).  us for a training step,
// all forwards in tiles -> this: ResNet-20, 8 images 1427 -> 957, 47 images 1466 -> 1173, 128 images 1626 -> 1569, VGG-small, 8 images 2357 -> 1224, 30
// 3324 -> 2839 (input gradients without tiles among them; with the statistics in the kernels without tiles and their grouping 849, 1127, 1508, 1195, 2848).
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

// BatchNorm statistics of a layer's output: per wave and output channel the sums of y and y*y over the wave's positions, in the partial-sum
// layout of the BatchNorm kernels (slot = position wave of the launch, stats[(co * slots + slot) * 2 + {0, 1}]).
// The lanes sum deviations from a pivot (lane 0's first value) in fp32 and lane 0 moves the sums back
// to the origin in fp64, so the cancellation in E[y*y] - E[y]^2 happens in double precision.
// row_ok: the lane's row is inside the map; wo: its first column; co_base: the first of the wave's TM channels.
template <int TM, int TN>
__device__ __forceinline__ void tile_stats(const float (&tot)[TM][TN], const bool row_ok, const int wo, const int Wo, const int co_base, const int Co,
                                           const int slots, const int slot, const int lane, double *__restrict__ stats) {
    float cnt = 0.f;
#pragma unroll
    for (int t = 0; t < TN; ++t) cnt += (row_ok && wo + t < Wo) ? 1.f : 0.f;
    const double count = (double)wave_sum_dpp(cnt);
    static_assert(TM == 2 || TM == 4 || TM == 8, "channels per lane of the tile shapes");
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
}

// ---------------------------------------------------------------------------
// Tiled kernel for 3x3 / pad 1, stride S = 1 or 2, and 1x1 / pad 0 (the figures are the 3x3 ones).
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
// MUL: the same kernel as an ordinary convolution, y = sum w * x (one v_fmac per term), for the regular
// stem layer that precedes the adder layers of a network.
// SUB: a strided 1x1 layer, whose sampled positions are walked as one long row.
// T: storage type of x and y.  EVAL: the inference epilogue.
// PAIR (3x3 taps at stride 2 only): the strided 1x1 layer that reads the same x beside this layer (the downsample
// branch of a residual block, resnet20.py:66-70) is computed along with it -- its one tap is the centre tap of the
// 3x3 window, so the x values are in registers already: weights w_side (Co, Ci), output y_side and statistics
// stats_side shaped like y and stats.
template <class C, bool VEC = true, bool SUB = false, bool MUL = false, bool PAIR = false, class T = float, bool EVAL = false>
__global__ __launch_bounds__(C::NTHREADS) void fwd_tile_kernel(const T *__restrict__ x,
                                                               const float *__restrict__ w,
                                                               T *__restrict__ y,
                                                               double *__restrict__ stats, int N, int Ci,
                                                               int H, int W, int Co, int Ho, int Wo,
                                                               int tilesH, int tilesW, const Subsample sub, const BnEval bn,
                                                               const float *__restrict__ w_side = nullptr,
                                                               T *__restrict__ y_side = nullptr,
                                                               double *__restrict__ stats_side = nullptr) {
    static_assert(!PAIR || (C::S == 2 && C::KS == 3 && !MUL && !SUB), "the side layer is a strided 1x1 beside a strided 3x3");
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
    uniform_f32_ptr wsc = as_uniform(w_side);
    int wsrow[PAIR ? TM : 1];
    float tots[PAIR ? TM : 1][TN];   // PAIR: the side layer's sums (Ci terms each: one level)
    if constexpr (PAIR) {
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            wsrow[m] = __builtin_amdgcn_readfirstlane(min(co_base + m, Co - 1) * Ci);
#pragma unroll
            for (int t = 0; t < TN; ++t) tots[m][t] = 0.f;
        }
    }

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
    tile_fetch<typename C::Patch, VEC, SUB, T>(st, x, 0, Ci, n0, N, h0 * S - C::PAD, w0 * S, H, W, sub);
    {   // this workgroup's output channels: one contiguous run of weights
        const int co_blk = blockIdx.y * C::COW * TM;
        l2_warm(w + (size_t)co_blk * K, 1, 0, min(C::COW * TM, Co - co_blk) * K);
    }
    tile_commit<typename C::Patch>(st, smem);
    __syncthreads();

    for (int c = 0; c < nchunks; ++c) {
        const int ci0 = c * C::CC;
        if (c + 1 < nchunks) tile_fetch<typename C::Patch, VEC, SUB, T>(st, x, ci0 + C::CC, Ci, n0, N, h0 * S - C::PAD, w0 * S, H, W, sub);

        const float *lbase = smem + (c & 1) * C::BUF + lane_off;
        const int ccnt = min(C::CC, Ci - ci0);
        // Software pipeline over the input channels of the chunk: the strips of channel
        // group cc+CQ and the weights of the next output channel are requested right after
        // the first subtract of the current one, i.e. after the wait for the current
        // operands and with the rest of the arithmetic still ahead to hide the latency.
        float xr[2][CQ][KS][STRIP];
        float wv[2][CQ * KK];
        float wsv[2][CQ];   // PAIR: the side layer's weights, buffered like wv
#pragma unroll
        for (int q = 0; q < CQ; ++q)
#pragma unroll
            for (int i = 0; i < KS; ++i)
                lds_read_strip<STRIP, C::STRIP_ALIGN>(lbase + q * C::PLANE + i * C::PITCH, xr[0][q][i]);
#pragma unroll
        for (int e = 0; e < CQ * KK; ++e) wv[0][e] = wc[wrow[0] + ci0 * KK + e];
        if constexpr (PAIR) {
#pragma unroll
            for (int q = 0; q < CQ; ++q) wsv[0][q] = wsc[wsrow[0] + ci0 + q];
        }

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
                    if constexpr (MUL)
                        acc[m][t] = fmaf(wv[m & 1][q * KK + i * KS + j], xr[cur][q][i][t * S + j], acc[m][t]);
                    else
                        acc[m][t] -= fabsf(wv[m & 1][q * KK + i * KS + j] - xr[cur][q][i][t * S + j]);
                    if (idx == 0) {
                        __builtin_amdgcn_sched_barrier(0);
                        if (m + 1 < TM) {
#pragma unroll
                            for (int e = 0; e < CQ * KK; ++e) wv[(m + 1) & 1][e] = wc[wrow[m + 1] + kofs + e];
                            if constexpr (PAIR) {
#pragma unroll
                                for (int q2 = 0; q2 < CQ; ++q2) wsv[(m + 1) & 1][q2] = wsc[wsrow[m + 1] + ci0 + cc + q2];
                            }
                        } else {
#pragma unroll
                            for (int e = 0; e < CQ * KK; ++e) wv[(m + 1) & 1][e] = wc[wrow[0] + knext + e];
                            if constexpr (PAIR) {
#pragma unroll
                                for (int q2 = 0; q2 < CQ; ++q2)
                                    wsv[(m + 1) & 1][q2] = wsc[wsrow[0] + ci0 + (more ? cc + CQ : cc) + q2];
                            }
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
                if constexpr (PAIR) {   // the centre tap (1, 1) is the strided 1x1 layer's only tap
#pragma unroll
                    for (int q = 0; q < CQ; ++q)
#pragma unroll
                        for (int t = 0; t < TN; ++t) tots[m][t] -= fabsf(wsv[m & 1][q] - xr[cur][q][1][t * S + 1]);
                }
            }
        };
        static_assert(TM % 2 == 0, "weight double buffer assumes an even number of channels per lane");
#pragma unroll 1
        for (int cc = 0; cc < ccnt; cc += 2 * CQ) {
            half(cc, 0);
            if (cc + CQ < ccnt) half(cc + CQ, 1);
        }

#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int t = 0; t < TN; ++t) { tot[m][t] += acc[m][t]; acc[m][t] = 0.f; }

        if (c + 1 < nchunks) tile_commit<typename C::Patch>(st, smem + ((c + 1) & 1) * C::BUF);
        __syncthreads();
    }

    const int n = n0 + img, ho = h0 + row, wo = w0 + strip * TN;
    auto finish = [&](float (&tot)[TM][TN], T *__restrict__ y, double *__restrict__ stats) {
    if (stats)
        tile_stats<TM, TN>(tot, lane_ok && n < N && ho < Ho, wo, Wo, co_base, Co, (int)gridDim.x * C::POSW, (int)blockIdx.x * C::POSW + pw, lane, stats);
    if (lane_ok && n < N && ho < Ho) {
        const bool vec = TN % 4 == 0 && (Wo & 3) == 0 && wo + TN <= Wo;
        if constexpr (EVAL) {
            float r[TM][TN];
#pragma unroll
            for (int m = 0; m < TM; ++m) {   // (all loads before the first store: one counter serves both)
                const size_t at = (((size_t)n * Co + min(co_base + m, Co - 1)) * Ho + ho) * Wo + wo;
#pragma unroll
                for (int t = 0; t < TN; ++t) r[m][t] = bn.res && wo + t < Wo ? bn.res[at + t] : 0.f;
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
    };
    finish(tot, y, stats);
    if constexpr (PAIR) finish(tots, y_side, stats_side);
}

// ---------------------------------------------------------------------------
// 1x1 layers of few positions: one output position x TM output channels per lane, the waves of a workgroup share the input channels.
//
// A tile gives a lane 8-16 results and walks all input channels in one wave; one image leaves a handful of workgroups, and the launch
// lasts as long as that serial chain.  Here wave v of a workgroup takes the channel chunks v, v + waves, ...; after each round the
// chunk sums go through LDS and are added in channel order.  x is read from global memory (a map this small sits in L1 / L2) one
// channel ahead of the arithmetic, as are the weights.  1024 -> 256 @14x14, 1 / 4 images, 105 -> 34, 105 -> 94 us.
// ---------------------------------------------------------------------------
static constexpr int kFewTM = 4;
__global__ __launch_bounds__(512) void fwd_few_kernel(const float *__restrict__ x, const float *__restrict__ w, float *__restrict__ y,
                                                      double *__restrict__ stats, ConvDims d, int chunk) {
    constexpr int TM = kFewTM, G = 8;
    __shared__ float part[8][TM][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int plane = d.H * d.W, L = d.Ho * d.Wo, total = d.N * L, co0 = blockIdx.y * TM;
    const int pos = min((int)blockIdx.x * 64 + lane, total - 1);
    const int n = pos / L, ho = pos % L / d.Wo, wo = pos % L % d.Wo;
    const int off = n * d.Ci * plane + ho * d.stride * d.W + wo * d.stride;
    uniform_f32_ptr wc = as_uniform(w);
    int wrow[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) wrow[m] = min(co0 + m, d.Co - 1) * d.Ci;
    const int nchunks = ceil_div(d.Ci, chunk);
    float tot[TM];   // of result threadIdx.x + k * blockDim.x of the workgroup's TM x 64
#pragma unroll
    for (int k = 0; k < TM; ++k) tot[k] = 0.f;

    for (int c0 = 0; c0 < nchunks; c0 += waves) {
        const int c = c0 + wave;
        if (c < nchunks) {
            const int first = c * chunk, end = min(first + chunk, d.Ci);
            float acc[TM], xv[2][G], wv[2][TM * G];
#pragma unroll
            for (int m = 0; m < TM; ++m) acc[m] = 0.f;
            auto load = [&](const int b, const int ci) {
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const int cc = min(ci + g, end - 1);
#pragma unroll
                    for (int m = 0; m < TM; ++m) wv[b][m * G + g] = wc[wrow[m] + cc];
                    xv[b][g] = x[(size_t)cc * plane + off];
                }
            };
            auto add = [&](const int b, const int ci) {
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    if (ci + g >= end) break;
#pragma unroll
                    for (int m = 0; m < TM; ++m) acc[m] -= fabsf(wv[b][m * G + g] - xv[b][g]);
                }
            };
            load(0, first);
#pragma unroll 1
            for (int ci = first; ci < end; ci += 2 * G) {
                load(1, ci + G);
                __builtin_amdgcn_sched_barrier(0);
                add(0, ci);
                load(0, ci + 2 * G);
                __builtin_amdgcn_sched_barrier(0);
                add(1, ci + G);
            }
#pragma unroll
            for (int m = 0; m < TM; ++m) part[wave][m][lane] = acc[m];
        }
        __syncthreads();
        const int here = min(waves, nchunks - c0);
#pragma unroll
        for (int k = 0; k < TM; ++k) {
            const int e = threadIdx.x + k * blockDim.x;
            if (e < TM * 64)
                for (int v = 0; v < here; ++v) tot[k] += part[v][e >> 6][e & 63];
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < TM; ++k) {
        const int e = threadIdx.x + k * blockDim.x, p = blockIdx.x * 64 + (e & 63), co = co0 + (e >> 6);
        if (e < TM * 64 && co < d.Co) {   // (wave-uniform: a wave holds 64 positions of one channel)
            const double v = p < total ? (double)tot[k] : 0.0, s1 = wave_sum(v), s2 = wave_sum(v * v);
            if (lane == 0) {
                double *dst = stats + ((size_t)co * gridDim.x + blockIdx.x) * 2;
                dst[0] = s1;
                dst[1] = s2;
            }
            if (p < total) y[((size_t)(p / L) * d.Co + co) * L + p % L] = tot[k];
        }
    }
}

// The statistics of a y that another kernel left, a wave per slot and TM channels: each wave has the results that a wave of
// fwd_tile_kernel<C> has, in the same lanes, so that the statistics are the same bits.  One read of y and about 3 us.
template <class C>
__global__ __launch_bounds__(256) void tile_stats_kernel(const float *__restrict__ y, double *__restrict__ stats, int N, int Co, int Ho, int Wo, int tilesH, int tilesW,
                                                         int slots) {
    constexpr int TM = C::TM, TN = C::TN;
    static_assert(C::LANES % 64 == 0, "whole waves of positions");
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6))), lane = threadIdx.x & 63;
    const int co_base = wave / slots * TM, slot = wave % slots;
    if (co_base >= Co) return;
    int b = slot / C::POSW;
    const int tw = b % tilesW; b /= tilesW;
    const int th = b % tilesH; b /= tilesH;
    const int p = slot % C::POSW * 64 + lane;
    const int n = b * C::NIMG + p / (C::SPR * C::TH), ho = th * C::TH + p / C::SPR % C::TH, wo = tw * C::TW + p % C::SPR * TN;
    const bool row_ok = n < N && ho < Ho;
    const float *src = y + ((size_t)min(n, N - 1) * Co * Ho + min(ho, Ho - 1)) * Wo;
    float tot[TM][TN];
#pragma unroll
    for (int m = 0; m < TM; ++m) {
        const float *row = src + (size_t)min(co_base + m, Co - 1) * Ho * Wo;
        if (Wo % TN == 0) {   // (a strip lies inside the row or beside it)
            ld_strip<TN>(row + min(wo, Wo - TN), tot[m]);
        } else {
#pragma unroll
            for (int t = 0; t < TN; ++t) tot[m][t] = row[min(wo + t, Wo - 1)];
        }
    }
    if (!row_ok) {
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int t = 0; t < TN; ++t) tot[m][t] = 0.f;
    }
    tile_stats<TM, TN>(tot, row_ok, wo, Wo, co_base, Co, slots, slot, lane, stats);
}

template <class C>
static int launch_tile_stats(const float *y, double *stats, const ConvDims &d, hipStream_t s) {
    const int tilesH = ceil_div(d.Ho, C::TH), tilesW = ceil_div(d.Wo, C::TW), slots = ceil_div(d.N, C::NIMG) * tilesH * tilesW * C::POSW;
    hipLaunchKernelGGL((tile_stats_kernel<C>), dim3((unsigned)ceil_div_l((long)slots * ceil_div(d.Co, C::TM), 4)), dim3(256), 0, s, y, stats, d.N, d.Co, d.Ho, d.Wo, tilesH,
                       tilesW, slots);
    return check_launch();
}

template <class C, bool VEC, bool SUB = false, bool MUL = false, bool PAIR = false, bool EVAL = false, class T = float>
static int launch_tile_v(const T *x, const float *w, T *y, double *stats, const ConvDims &d, hipStream_t s,
                         const Subsample sub = Subsample{1, 0, 0, 0}, const BnEval &bn = kNoBnEval, const float *w_side = nullptr,
                         T *y_side = nullptr, double *stats_side = nullptr) {
    const int tilesH = ceil_div(d.Ho, C::TH), tilesW = ceil_div(d.Wo, C::TW);
    const long gx = (long)ceil_div(d.N, C::NIMG) * tilesH * tilesW;
    const int gy = ceil_div(d.Co, C::TM * C::COW);
    if (gx > 0x7fffffffL) return ADDER_ERR_TOO_LARGE;
    if (int rc = allow_dynamic_lds<&fwd_tile_kernel<C, VEC, SUB, MUL, PAIR, T, EVAL>>(C::LDS_BYTES)) return rc;
    hipLaunchKernelGGL((fwd_tile_kernel<C, VEC, SUB, MUL, PAIR, T, EVAL>), dim3((unsigned)gx, gy), dim3(C::NTHREADS), C::LDS_BYTES, s, x, w, y,
                       stats, d.N, d.Ci, d.H, d.W, d.Co, d.Ho, d.Wo, tilesH, tilesW, sub, bn, w_side, y_side, stats_side);
    return check_launch();
}

// element-wise tile loads when the rows of the staged tensor are not whole groups of four
template <class C, bool MUL = false>
static int launch_tile(const float *x, const float *w, float *y, double *stats, const ConvDims &d, hipStream_t s) {
    return d.W % 4 == 0 ? launch_tile_v<C, true, false, MUL>(x, w, y, stats, d, s) : launch_tile_v<C, false, false, MUL>(x, w, y, stats, d, s);
}

// partial-sum slots per channel the statistics epilogue of this tile shape writes
template <class C>
static int tile_slots(const ConvDims &d) {
    const long gx = (long)ceil_div(d.N, C::NIMG) * ceil_div(d.Ho, C::TH) * ceil_div(d.Wo, C::TW);
    return (int)(gx * C::POSW);
}

// Tile shapes per output width, picked by timing sweeps on MI355X.  What they have in common: a ResNet-20
// layer at batch 256 launches 2048-4096 waves in 256-512 workgroups of eight waves; a lane keeps only
// 2-4 output channels x 4 positions (few registers, short dependent chains); one pipeline unit is one
// output channel x one input channel (CQ = 1: 9 weights, 18*TN vector instructions), which keeps the two
// weight buffers far from the 102-SGPR limit (spilled SGPRs come back as v_readlane inside the hot loop)
// and works for odd channel counts too.
//                           TN SPR TH NIMG TM COW CC CQ S
using FwdW32   = Tile3x3Cfg<4, 8, 16, 1, 4, 4, 8, 1, 1>;    // outputs 32 wide: half an image x 16 channels
using FwdW16   = Tile3x3Cfg<4, 4, 16, 1, 4, 8, 16, 1, 1>;   // outputs 16 wide: one image x 32 channels
using FwdW8    = Tile3x3Cfg<4, 2, 8, 4, 2, 8, 16, 1, 1>;    // outputs 8 wide: four images x 16 channels
using FwdW16S2 = Tile3x3Cfg<2, 8, 16, 1, 4, 8, 8, 1, 2>;    // stride 2, outputs 16 wide: one image x 32 channels
using FwdW8S2  = Tile3x3Cfg<2, 4, 8, 2, 4, 8, 16, 1, 2>;    // stride 2, outputs 8 wide: two images x 32 channels
// ... with chunks of 8 input channels: two workgroups fit a CU's LDS instead of one, which pays from 128
// input channels on (512 -> 512 @14x14, batch 64: 740 -> 530 us; at 32 channels the extra barriers cost 2 %)
using FwdW8S2L = Tile3x3Cfg<2, 4, 8, 2, 4, 8, 8, 1, 2>;
// 1x1, stride 1: every (H, W) plane is one row of H*W positions; a unit is one output channel x 8 input
// channels (8 weights, 64 vector instructions), eight output-channel waves share the staged x tile.
using Fwd1x1   = Tile3x3Cfg<4, 64, 1, 1, 4, 8, 16, 8, 1, 1>;   // 256 positions of one image x 32 channels
using Fwd1x1s  = Tile3x3Cfg<4, 16, 1, 4, 4, 8, 16, 8, 1, 1>;   // planes of <= 64 positions: four images
// 1x1 with a stride: the tile loader gathers the sampled x element by element, which costs several times what the
// aligned float4 loads of a stride-1 plane cost, so a workgroup takes 64 output channels per staged tile instead of
// 32 (eight per lane, chunks of eight input channels to stay within 128 registers); ResNet-50's three downsample
// layers at batch 64: 538 -> 319, 621 -> 376, 591 -> 374 us.  (On stride-1 planes this shape is slower.)
using Fwd1x1sub = Tile3x3Cfg<4, 16, 1, 4, 8, 8, 8, 8, 1, 1>;   // 64 sampled positions of four images x 64 channels
// the same two with units of four input channels, for channel counts that are multiples of 4 but not of 8
// (DenseNet's multiples of 12)
using Fwd1x1q  = Tile3x3Cfg<4, 64, 1, 1, 4, 8, 16, 4, 1, 1>;
using Fwd1x1sq = Tile3x3Cfg<4, 16, 1, 4, 4, 8, 16, 4, 1, 1>;

// ... the same register tile in workgroups of four waves that cover fewer rows, for maps whose height is not a
// multiple of 16: 56 rows are 7 x 8, 28 rows 7 x 4 (ResNet-50 at batch 64: 64 -> 64 @56x56 340 -> 294 us,
// 128 -> 128 @28x28 330 -> 298 us); on 32 rows they are no faster than FwdW32
using FwdW32H8 = Tile3x3Cfg<4, 8, 8, 1, 4, 4, 8, 1, 1>;    // 8 rows of one image x 16 channels
using FwdW32H4 = Tile3x3Cfg<4, 8, 4, 2, 4, 4, 8, 1, 1>;    // 4 rows of two images x 16 channels
// rows per tile (16, 8 or 4) that pad a map of H rows least; the larger tile on a tie
static int rows_per_tile_w32(int H) {
    const int p16 = round_up(H, 16), p8 = round_up(H, 8), p4 = round_up(H, 4);
    return p16 <= p8 && p16 <= p4 ? 16 : (p8 <= p4 ? 8 : 4);
}

// which tiled kernel serves these dimensions (0 = none): 1..3 3x3 stride 1 by output width, 4..5 3x3 stride 2,
// 6..7 1x1 stride 1 by plane size, 8..9 1x1 with a stride (the sampled positions walked like a stride-1 plane),
// 10..13 = 6..9 with units of four input channels
static int tile_variant(const ConvDims &d) {
    // (below 64 input channels the plain 1x1 kernel of conv1x1.hip is as fast or faster)
    if (d.kh == 1 && d.kw == 1 && d.pad == 0 && d.Ci % Fwd1x1q::CQ == 0 && d.Ci >= 64) {
        const int quad = d.Ci % Fwd1x1::CQ ? 4 : 0;
        // 256 positions of one image per workgroup, or 64 positions of four: whichever pads the plane less
        // (28x28 = 784 positions fill 64-wide tiles to 94 %, 256-wide ones to 77 %: 216 -> 169 us for 128 -> 512)
        const int plane = d.Ho * d.Wo;
        const bool wide = ceil_div(plane, Fwd1x1::TW) * Fwd1x1::TW <= ceil_div(plane, Fwd1x1s::TW) * Fwd1x1s::TW;
        if (d.stride == 1) return (wide ? 6 : 7) + quad;
        return (wide ? 8 : 9) + quad;
    }
    if (d.kh != 3 || d.kw != 3 || d.pad != 1) return 0;
    if (d.stride == 1) return d.Wo > 16 ? 1 : (d.Wo > 8 ? 2 : 3);
    if (d.stride == 2) return d.Wo > 8 ? 4 : 5;
    return 0;
}

// Input channels per first-level sum of a layer's results, in every forward kernel.  (25 taps: a chunk of eight is 200 terms already.  Of
// one-signed terms n2 sums of n1 round to sqrt(n1 / n2 + n2), which for more than 34 chunks is less with 16 channels each: 813
// channels 1.6e-7 -> 1.2e-7 of the result.)
int fwd_chunk(const ConvDims &d) {
    if (d.kh == 5 && d.kw == 5) return ceil_div(d.Ci, 8) > 34 ? 16 : 8;
    switch (tile_variant(d)) {
        case 0: return conv1x1_supported(d, nullptr, nullptr) ? 64 : 16;
        case 1: return FwdW32::CC;
        case 2: return FwdW16::CC;
        case 3: return FwdW8::CC;
        case 4: return FwdW16S2::CC;
        case 5: return d.Ci >= 128 ? FwdW8S2L::CC : FwdW8S2::CC;
        case 8: case 9: return Fwd1x1sub::CC;
        default: return Fwd1x1::CC;
    }
}
static_assert(FwdW32::CC == FwdW32H8::CC && FwdW32::CC == FwdW32H4::CC && Fwd1x1::CC == Fwd1x1s::CC &&
              Fwd1x1::CC == Fwd1x1q::CC && Fwd1x1::CC == Fwd1x1sq::CC, "one chunk length per variant");

// Whether the kernel for few positions takes a 1x1 layer.  The tiled kernels last as long as one wave's chain of
// channels x results per lane, 6 ns a term, until the chip is full; this one has a chain of its share of the
// channels (0.25 us each) and then works at 3.2 terms per ps.  Beyond the line the tiled kernels win: 1024 -> 256
// @14x14, 16 images, 106 against 281 us.  (The plain 1x1 kernel has short chains.)
static bool few_positions(const ConvDims &d, int variant) {
    if (variant < 6 || ceil_div(d.Co, kFewTM) > kMaxGridY) return false;
    const int per_lane = variant == 8 || variant == 9 ? Fwd1x1sub::TM * Fwd1x1sub::TN : Fwd1x1::TM * Fwd1x1::TN;
    const float terms = (float)d.K() * d.Co * d.N * d.Ho * d.Wo;
    const int chunk = fwd_chunk(d);
    const float tiled = 0.006f * d.K() * per_lane;
    const float share = (float)(ceil_div(ceil_div(d.Ci, chunk), 8) * chunk);
    const float few = 2.f + (0.25f * share + terms / 3.2e6f);
    return few < 0.9f * tiled;
}

// a 1x1 layer seen as N x Ci "images" of one row of Ho*Wo positions (the whole plane when the stride is 1)
static ConvDims as_one_row(const ConvDims &d) {
    ConvDims f = d;
    f.H = f.Ho = 1;
    f.W = f.Wo = d.Ho * d.Wo;
    f.stride = 1;
    return f;
}
static Subsample sampling_of(const ConvDims &d) { return Subsample{d.stride, d.Wo, d.W, d.H * d.W}; }

// A strided 3x3 / pad 1 layer and the strided 1x1 / pad 0 layer beside it (same x, same Co, Ho, Wo) in one launch;
// d describes the 3x3 layer.  Both outputs with their statistics (fwd_stats_slots(d) slots each).  Rows of whole
// float4 groups only; ADDER_ERR_UNSUPPORTED otherwise.
bool fwd_pair_supported(const ConvDims &d) {
    return d.kh == 3 && d.kw == 3 && d.pad == 1 && d.stride == 2 && d.W % 4 == 0 && d.H % 2 == 0;
}

int launch_fwd_pair(const float *x, const float *w, const float *w_side, float *y, float *y_side, double *stats,
                    double *stats_side, const ConvDims &d, hipStream_t s) {
    if (!fwd_pair_supported(d)) return ADDER_ERR_UNSUPPORTED;
    auto run = [&](auto cfg) {
        return launch_tile_v<decltype(cfg), true, false, false, true>(x, w, y, stats, d, s, Subsample{1, 0, 0, 0}, kNoBnEval, w_side, y_side, stats_side);
    };
    if (d.Wo > 8) return run(FwdW16S2{});
    return d.Ci >= 128 ? run(FwdW8S2L{}) : run(FwdW8S2{});
}

// f(tile shape, dimensions): of a layer's variant, 1x1 layers as one row
template <class F>
static auto with_tile(const ConvDims &d, int variant, F f) {
    switch (variant) {
        case 1: switch (rows_per_tile_w32(d.Ho)) {
            case 16: return f(FwdW32{}, d);
            case 8: return f(FwdW32H8{}, d);
            default: return f(FwdW32H4{}, d);
        }
        case 2: return f(FwdW16{}, d);
        case 3: return f(FwdW8{}, d);
        case 4: return f(FwdW16S2{}, d);
        case 5: return d.Ci >= 128 ? f(FwdW8S2L{}, d) : f(FwdW8S2{}, d);
        case 6: return f(Fwd1x1{}, as_one_row(d));
        case 7: return f(Fwd1x1s{}, as_one_row(d));
        case 8: case 9: return f(Fwd1x1sub{}, as_one_row(d));
        case 10: case 12: return f(Fwd1x1q{}, as_one_row(d));
        default: return f(Fwd1x1sq{}, as_one_row(d));
    }
}

int fwd_stats_slots(const ConvDims &d) {
    const int variant = tile_variant(d);
    if (few_positions(d, variant)) return ceil_div(d.N * d.Ho * d.Wo, 64);
    if (variant == 0) return conv1x1_supported(d, nullptr, nullptr) ? fwd_1x1_stats_slots(d) : 0;
    return with_tile(d, variant, [](auto cfg, const ConvDims &f) { return tile_slots<decltype(cfg)>(f); });
}

// Whether a forward with statistics is the kernel without tiles and, behind it, tile_stats_kernel: where the tiles leave half of the CUs without a workgroup, or
// a good share of their lanes without a position and the layer is long enough for that to outweigh the read of y.  us, tiles / plain forward, to which
// the statistics add 3 to 4 and a read of y: 16 -> 16 @32x32, 64 images, 128 workgroups, 15.7 / 11.1, 128 images 16.6 / 16.0; 64 -> 64 @8x8, 8 images 28 / 7.3, 128 28.6 / 18.2,
// 256 29.1 / 26.1, stride 2 32 -> 64 @16x16, 32 images, 18.6 / 11.2, 64 18.7 / 16.5; 64 -> 64 @56x56 (88 % of the lanes), 32 images, 160 / 136, 512 -> 512 @7x7 (77 %) 285 / 180, stride 2 128 -> 128 @56x56 (77 %) 221 / 153;
// 512 -> 512 @8x8, 32 images, 256 workgroups, 276 / 182; whole tiles, 128 -> 128 @32x32, 128 images, 654 / 622 with 67 MB of y; 1x1, 1024 -> 256 @14x14 (77 %), 128 images, 336 / 297,
// 512 -> 128 @28x28 (94 %), 32 images, 93 / 86.
static bool statistics_apart(const ConvDims &d, int variant) {
    if (variant == 0 || few_positions(d, variant) || d.K() < 100) return false;
    if (variant < 6 ? !fwd_nine_supported(d) : !fwd_tap_supported(d) || fwd_strided_tile_supported(d)) return false;
    return with_tile(d, variant, [&](auto cfg, const ConvDims &f) {
        using C = decltype(cfg);
        const long tiles = (long)ceil_div(f.N, C::NIMG) * ceil_div(f.Ho, C::TH) * ceil_div(f.Wo, C::TW), wgs = tiles * ceil_div(f.Co, C::TM * C::COW);
        if (tiles * C::POSW * ceil_div(f.Co, C::TM) * 64 > kMaxThreads - 256) return false;
        constexpr int waves = C::NTHREADS / 64 < 8 ? C::NTHREADS / 64 : 8;
        if (wgs * waves <= (d.K() >= 2000 ? 2048 : variant == 5 ? 384 : 1024)) return true;
        return d.K() >= 500 && 100L * f.N * f.Ho * f.Wo < (d.kh == 3 ? 90 : 80) * tiles * (C::NIMG * C::TH * C::TW);
    });
}

int fwd_stats_kernel(const ConvDims &d) {
    const int variant = tile_variant(d), rows = rows_per_tile_w32(d.Ho);
    if (few_positions(d, variant)) return 2;
    if (variant == 0) return conv1x1_supported(d, nullptr, nullptr) ? 1 : 0;
    return (statistics_apart(d, variant) ? 1000 : 0) + 10 * variant + (variant == 1 ? (rows == 16 ? 0 : rows == 8 ? 1 : 2) : variant == 5 && d.Ci >= 128 ? 1 : 0);
}

// stats: per-channel partial sums of y and y*y, fwd_stats_slots(d) > 0 slots per channel.
int launch_fwd_stats(const float *x, const float *w, float *y, double *stats, const ConvDims &d, hipStream_t s) {
    const int variant = tile_variant(d);
    if (few_positions(d, variant)) {
        const int chunk = fwd_chunk(d), chunks = ceil_div(d.Ci, chunk);
        hipLaunchKernelGGL(fwd_few_kernel, dim3(ceil_div(d.N * d.Ho * d.Wo, 64), ceil_div(d.Co, kFewTM)), dim3(64 * (chunks < 8 ? chunks : 8)),
                           0, s, x, w, y, stats, d, chunk);
        return check_launch();
    }
    if (variant == 0) return conv1x1_supported(d, x, y) ? launch_fwd_1x1(x, w, y, stats, d, s, kNoBnEval) : static_cast<int>(ADDER_ERR_UNSUPPORTED);
    // rows (1x1: planes) that are whole groups of four are moved as such and need bases aligned to a group; x of a strided 1x1 layer is read element by element
    const ConvDims f = variant >= 6 ? as_one_row(d) : d;
    const bool strided = variant >= 6 && d.stride > 1;
    if ((!strided && f.W % 4 == 0 && !aligned_groups(x)) || (f.Wo % 4 == 0 && !aligned_groups(y))) return ADDER_ERR_UNSUPPORTED;
    if (statistics_apart(d, variant)) {
        if (int rc = variant < 6 ? launch_fwd_nine(x, w, y, d, s, kNoBnEval) : launch_fwd_tap(x, w, y, d, s, kNoBnEval)) return rc;
        return with_tile(d, variant, [&](auto cfg, const ConvDims &g) { return launch_tile_stats<decltype(cfg)>(y, stats, g, s); });
    }
    switch (variant) {
        case 1: switch (rows_per_tile_w32(d.Ho)) {
            case 16: return launch_tile<FwdW32>(x, w, y, stats, d, s);
            case 8: return launch_tile<FwdW32H8>(x, w, y, stats, d, s);
            default: return launch_tile<FwdW32H4>(x, w, y, stats, d, s);
        }
        case 2: return launch_tile<FwdW16>(x, w, y, stats, d, s);
        case 3: return launch_tile<FwdW8>(x, w, y, stats, d, s);
        case 4: return launch_tile<FwdW16S2>(x, w, y, stats, d, s);
        case 5: return d.Ci >= 128 ? launch_tile<FwdW8S2L>(x, w, y, stats, d, s) : launch_tile<FwdW8S2>(x, w, y, stats, d, s);
        case 6: return launch_tile<Fwd1x1>(x, w, y, stats, f, s);
        case 7: return launch_tile<Fwd1x1s>(x, w, y, stats, f, s);
        case 8: case 9: return launch_tile_v<Fwd1x1sub, false, true>(x, w, y, stats, f, s, sampling_of(d));
        case 10: return launch_tile<Fwd1x1q>(x, w, y, stats, f, s);
        case 11: return launch_tile<Fwd1x1sq>(x, w, y, stats, f, s);
        case 12: return launch_tile_v<Fwd1x1q, false, true>(x, w, y, stats, f, s, sampling_of(d));
        default: return launch_tile_v<Fwd1x1sq, false, true>(x, w, y, stats, f, s, sampling_of(d));
    }
}

// Strided 1x1 layers without statistics that stay in tiles: chunks of eight channels, whose sums the waves of fwd_tap.hip would have to bring together after 16
// terms each, and a workgroup per CU.  us, tiles / fwd_tap.hip: 32 images 256 -> 512 @56x56 188 / 225, 512 -> 1024 @28x28 200 / 250, 1024 -> 2048 @14x14
// 276 / 291; four images, 104 and 64 workgroups, 72 / 46, 116 / 53.
bool fwd_strided_tile_supported(const ConvDims &d) {
    const int variant = tile_variant(d);
    if (variant != 8 && variant != 9) return false;
    const long blocks = ceil_div(d.Co, Fwd1x1sub::TM * Fwd1x1sub::COW), wgs = (long)ceil_div(d.N, Fwd1x1sub::NIMG) * ceil_div(d.Ho * d.Wo, Fwd1x1sub::TW) * blocks;
    return blocks <= kMaxGridY && wgs >= 256 && wgs * Fwd1x1sub::NTHREADS <= 0xffffffffL;
}

template <class T>
int launch_fwd_strided_tile(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn) {
    const ConvDims f = as_one_row(d);
    if constexpr (sizeof(T) == 4) {
        if (bn.gamma) return launch_tile_v<Fwd1x1sub, false, true, false, false, true, T>(x, w, y, nullptr, f, s, sampling_of(d), bn);
    }
    return launch_tile_v<Fwd1x1sub, false, true, false, false, false, T>(x, w, y, nullptr, f, s, sampling_of(d));
}
template int launch_fwd_strided_tile<float>(const float *, const float *, float *, const ConvDims &, hipStream_t, const BnEval &);
template int launch_fwd_strided_tile<bf16_t>(const bf16_t *, const float *, bf16_t *, const ConvDims &, hipStream_t, const BnEval &);

// An ordinary convolution y = sum w * x through the tiled forward kernels: 3x3 / stride 1 / pad 1 only
// (ADDER_ERR_UNSUPPORTED elsewhere).  stats as in launch_fwd_stats (nullable); the slot count is fwd_stats_slots(d).
int launch_mulconv_fwd(const float *x, const float *w, float *y, double *stats, const ConvDims &d, hipStream_t s) {
    const bool ok = d.kh == 3 && d.kw == 3 && d.pad == 1 && d.stride == 1 &&
                    (d.W % 4 != 0 || ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15) == 0);
    if (!ok) return ADDER_ERR_UNSUPPORTED;
    switch (tile_variant(d)) {
        case 1: switch (rows_per_tile_w32(d.Ho)) {   // (the statistics slots are counted per tile shape)
            case 16: return launch_tile<FwdW32, true>(x, w, y, stats, d, s);
            case 8: return launch_tile<FwdW32H8, true>(x, w, y, stats, d, s);
            default: return launch_tile<FwdW32H4, true>(x, w, y, stats, d, s);
        }
        case 2: return launch_tile<FwdW16, true>(x, w, y, stats, d, s);
        case 3: return launch_tile<FwdW8, true>(x, w, y, stats, d, s);
        default: return ADDER_ERR_UNSUPPORTED;
    }
}

}  // namespace adder

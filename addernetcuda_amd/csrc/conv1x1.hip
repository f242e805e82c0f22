// 1x1 AdderNet convolution, pad 0, stride S = 1 or 2 (the ResNet downsample
// path, resnet20.py:66-70): the same three operations as the 3x3 kernels with
// K = Ci, so there is no halo and no LDS tile -- every lane reads its own
// float4 of the source row and keeps a TM x TN register tile; weights are
// wave-uniform SGPR operands.
//   forward  y[n,co,ho,wo]  = -sum_ci |w[co,ci] - x[n,ci,ho*S,wo*S]|
//   grad_x   gx[n,ci,hi,wi] =  sum_co hardtanh(w[co,ci] - x) * gy[n,co,hi/S,wi/S]  on the sampled
//                              grid, exactly 0 on the positions stride 2 skips
//   grad_w   gw[co,ci]      =  sum x*gy - w * sum gy   (see the kernel for the precision of its partial sums)
// Replaces adder.cu:19-70 / 194-272 for these shapes together with the
// unfold/fold copies of adder.py:32-33,38-39.
#include "common.hpp"

#include <type_traits>

namespace adder {

// A lane owns 4/S adjacent outputs of one output row: one float4 of the source row.
template <int S>
struct Lane1x1 {
    static constexpr int TN = 4 / S;
    int n, ho, wo0;   // first output of the lane
    bool ok;
    __device__ __forceinline__ Lane1x1(int g, int groups, int gpr, int Ho) {
        ok = g < groups;
        if (!ok) g = groups - 1;
        const int q = g % gpr;
        ho = (g / gpr) % Ho;
        n = g / (gpr * Ho);
        wo0 = q * TN;
    }
};

// Four consecutive elements of a row as floats.  VEC: one aligned group of four.  Otherwise (stride 1 on planes whose
// size is not a multiple of 4, walked as one long row) element by element, `valid` of them inside the row.
// T: storage type of the activations (float or bf16_t); arithmetic is fp32 either way.
template <bool VEC, class T>
__device__ __forceinline__ float4 ld4(const T *p, int valid) {
    if constexpr (VEC) return ldf4(p);
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (valid > 0) v.x = ldf(p);
    if (valid > 1) v.y = ldf(p + 1);
    if (valid > 2) v.z = ldf(p + 2);
    if (valid > 3) v.w = ldf(p + 3);
    return v;
}
template <bool VEC, class T>
__device__ __forceinline__ void st4(T *p, const float4 v, int valid) {
    if constexpr (VEC) {
        stf4(p, v);
    } else {
        if (valid > 0) stf(p, v.x);
        if (valid > 1) stf(p + 1, v.y);
        if (valid > 2) stf(p + 2, v.z);
        if (valid > 3) stf(p + 3, v.w);
    }
}

template <bool VEC, class T>
__device__ __forceinline__ float2 ld2(const T *p, int valid) {
    if constexpr (VEC) return ldf2(p);
    float2 v = make_float2(0.f, 0.f);
    if (valid > 0) v.x = ldf(p);
    if (valid > 1) v.y = ldf(p + 1);
    return v;
}
template <bool VEC, class T>
__device__ __forceinline__ void st2(T *p, const float2 v, int valid) {
    if constexpr (VEC) {
        stf2(p, v);
    } else {
        if (valid > 0) stf(p, v.x);
        if (valid > 1) stf(p + 1, v.y);
    }
}

template <int S, int TM, bool VEC = true, class T = float>
__global__ __launch_bounds__(256) void fwd_1x1_kernel(const T *__restrict__ x, const float *__restrict__ w,
                                                      T *__restrict__ y, double *__restrict__ stats, int N, int Ci,
                                                      int H, int W, int Co, int Ho, int Wo, int gpr, int groups,
                                                      const BnEval bn) {
    constexpr int TN = 4 / S;
    const Lane1x1<S> L(blockIdx.x * 256 + threadIdx.x, groups, gpr, Ho);
    const int co0 = blockIdx.y * TM;
    uniform_f32_ptr wc = as_uniform(w);
    int wrow[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) wrow[m] = min(co0 + m, Co - 1) * Ci;
    float acc[TM][TN], tot[TM][TN];   // two-level sum: acc holds at most 64 channels
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t) acc[m][t] = tot[m][t] = 0.f;

    l2_warm(w + (size_t)co0 * Ci, 1, 0, min(TM, Co - co0) * Ci);   // the scalar weight loads below run one step ahead

    const size_t plane = (size_t)H * W;
    const T *xp = x + (size_t)L.n * Ci * plane + (size_t)(L.ho * S) * W + L.wo0 * S;
    const int valid = L.ok ? W - L.wo0 * S : 0;   // only read when !VEC
    int ci = 0;
    for (; ci + 4 <= Ci; ci += 4) {
        if ((ci & 63) == 0) {
#pragma unroll
            for (int m = 0; m < TM; ++m)
#pragma unroll
                for (int t = 0; t < TN; ++t) { tot[m][t] += acc[m][t]; acc[m][t] = 0.f; }
        }
        float4 xv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) xv[e] = ld4<VEC>(xp + (size_t)(ci + e) * plane, valid);
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float wv = wc[wrow[m] + ci + e];
                const float xs[4] = {xv[e].x, xv[e].y, xv[e].z, xv[e].w};
#pragma unroll
                for (int t = 0; t < TN; ++t) acc[m][t] -= fabsf(wv - xs[t * S]);
            }
    }
    for (; ci < Ci; ++ci) {
        const float4 v = ld4<VEC>(xp + (size_t)ci * plane, valid);
        const float xs[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            const float wv = wc[wrow[m] + ci];
#pragma unroll
            for (int t = 0; t < TN; ++t) acc[m][t] -= fabsf(wv - xs[t * S]);
        }
    }
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t) tot[m][t] += acc[m][t];
    if (stats) {
        // BatchNorm statistics of the output on the way out, as in the tiled forward kernels: per wave and output
        // channel the sums of y and y*y over the wave's valid outputs (deviations from a pivot in fp32, moved
        // back to the origin in fp64), slot = wave of this launch
        const int lane = threadIdx.x & 63;
        const int slots = gridDim.x * 4, slot = blockIdx.x * 4 + (threadIdx.x >> 6);
        const int nvalid = L.ok ? min(TN, Wo - L.wo0) : 0;
        const double count = (double)wave_sum_dpp((float)nvalid);
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            const float pivot = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(tot[m][0])));
            float s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int t = 0; t < TN; ++t)
                if (t < nvalid) {
                    const float dv = tot[m][t] - pivot;
                    s1 += dv;
                    s2 = fmaf(dv, dv, s2);
                }
            const double d1 = (double)wave_sum_dpp(s1), d2 = (double)wave_sum_dpp(s2), c = (double)pivot;
            if (lane == 0 && co0 + m < Co) {
                stats[((size_t)(co0 + m) * slots + slot) * 2] = d1 + count * c;
                stats[((size_t)(co0 + m) * slots + slot) * 2 + 1] = d2 + 2.0 * c * d1 + count * c * c;
            }
        }
    }
    if (L.ok) {
        if constexpr (sizeof(T) == 4) {
            if (bn.gamma) {   // inference: the BatchNorm behind the layer, the shortcut and the ReLU on the way out
#pragma unroll
                for (int m = 0; m < TM; ++m) {
                    const int co = min(co0 + m, Co - 1);
                    const BnEvalChannel ch(bn, co);
                    const float *res = bn.res + (((size_t)L.n * Co + co) * Ho + L.ho) * Wo + L.wo0;
#pragma unroll
                    for (int t = 0; t < TN; ++t) {
                        tot[m][t] = ch(tot[m][t]);
                        if (bn.res && L.wo0 + t < Wo) tot[m][t] += res[t];
                        if (bn.relu) tot[m][t] = relu_keep_nan(tot[m][t]);
                    }
                }
            }
        }
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            if (co0 + m >= Co) continue;
            T *dst = y + (((size_t)L.n * Co + co0 + m) * Ho + L.ho) * Wo + L.wo0;
            if constexpr (TN == 4)
                st4<VEC>(dst, make_float4(tot[m][0], tot[m][1], tot[m][2], tot[m][3]), valid);
            else
                st2<VEC>(dst, make_float2(tot[m][0], tot[m][1]), L.ok ? Wo - L.wo0 : 0);
        }
    }
}

template <int S, int TM, bool VEC = true, class T = float>
__global__ __launch_bounds__(256) void grad_x_1x1_kernel(const T *__restrict__ gy,
                                                         const T *__restrict__ x,
                                                         const float *__restrict__ w, T *__restrict__ gx,
                                                         int N, int Ci, int H, int W, int Co, int Ho, int Wo,
                                                         int gpr, int groups) {
    constexpr int TN = 4 / S;
    const Lane1x1<S> L(blockIdx.x * 256 + threadIdx.x, groups, gpr, Ho);
    const int ci0 = blockIdx.y * TM;
    uniform_f32_ptr wc = as_uniform(w);
    const size_t plane = (size_t)H * W;
    const size_t xoff = (size_t)L.n * Ci * plane + (size_t)(L.ho * S) * W + L.wo0 * S;
    const int valid = L.ok ? W - L.wo0 * S : 0;   // only read when !VEC
    // clamp(w - x, -1, 1) = 2 * sat(0.5 w + cr) - 1 with cr = 0.5 - 0.5 x and sat the [0, 1] clamp modifier of
    // v_fma_f32: two instructions per term; sg collects the gy sum that the "- 1" multiplies
    float cr[TM][TN], acc[TM][TN], tot[TM][TN];   // two-level sum: acc holds at most 64 output channels
    float sg[TN], sgt[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t) sg[t] = sgt[t] = 0.f;
#pragma unroll
    for (int m = 0; m < TM; ++m) {
        const float4 v = ld4<VEC>(x + xoff + (size_t)min(ci0 + m, Ci - 1) * plane, valid);
        const float xs[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int t = 0; t < TN; ++t) { cr[m][t] = fmaf(-0.5f, xs[t * S], 0.5f); acc[m][t] = tot[m][t] = 0.f; }
    }
    l2_warm(w + min(ci0, Ci - 1), Co, Ci, min(TM, Ci - ci0));   // one run of TM weights per output channel
    const size_t gplane = (size_t)Ho * Wo;
    const T *gp = gy + (size_t)L.n * Co * gplane + (size_t)L.ho * Wo + L.wo0;
    // eight output channels per round: their gy loads are issued together (little arithmetic per load, so
    // the loop is bound by how many loads are in flight); channels past Co load nothing and count as gy = 0
    constexpr int UN = 8;
    for (int co0 = 0; co0 < Co; co0 += UN) {
        float g[UN][TN];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const bool live = co0 + u < Co;
            const T *src = gp + (size_t)min(co0 + u, Co - 1) * gplane;
            if constexpr (TN == 4) {
                const float4 v = ld4<VEC>(src, live ? valid : 0);
                g[u][0] = v.x; g[u][1] = v.y; g[u][2] = v.z; g[u][3] = v.w;
            } else {
                const float2 v = ld2<VEC>(src, live && L.ok ? Wo - L.wo0 : 0);
                g[u][0] = v.x; g[u][1] = v.y;
            }
            if (VEC && !live) {
#pragma unroll
                for (int t = 0; t < TN; ++t) g[u][t] = 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int co = min(co0 + u, Co - 1);
#pragma unroll
            for (int m = 0; m < TM; ++m) {
                const float wv = wc[co * Ci + min(ci0 + m, Ci - 1)];
#pragma unroll
                for (int t = 0; t < TN; ++t) acc[m][t] = fmaf(sat01(fmaf(wv, 0.5f, cr[m][t])), g[u][t], acc[m][t]);
            }
#pragma unroll
            for (int t = 0; t < TN; ++t) sg[t] += g[u][t];
        }
        if ((co0 & 63) == 64 - UN || co0 + UN >= Co) {
#pragma unroll
            for (int m = 0; m < TM; ++m)
#pragma unroll
                for (int t = 0; t < TN; ++t) { tot[m][t] += acc[m][t]; acc[m][t] = 0.f; }
#pragma unroll
            for (int t = 0; t < TN; ++t) { sgt[t] += sg[t]; sg[t] = 0.f; }
        }
    }
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t) tot[m][t] = fmaf(2.f, tot[m][t], -sgt[t]);
    if (L.ok) {
        const bool row2 = S == 2 && L.ho * 2 + 1 < H;  // the odd row below: never sampled by stride 2
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            if (ci0 + m >= Ci) continue;
            T *dst = gx + xoff + (size_t)(ci0 + m) * plane;
            if constexpr (S == 1) {
                st4<VEC>(dst, make_float4(tot[m][0], tot[m][1], tot[m][2], tot[m][3]), valid);
            } else {
                st4<VEC>(dst, make_float4(tot[m][0], 0.f, tot[m][1], 0.f), valid);
                if (row2) st4<VEC>(dst + W, make_float4(0.f, 0.f, 0.f, 0.f), valid);
            }
        }
    }
}

// grad_w: a wave owns TM output channels x TC input channels; its lanes walk over position
// groups, then the 64 lanes are folded through LDS (16 sums per round).
// float storage: fp32 sums and slabs, as many slabs as keep a lane's sums short.  bfloat16 storage (fp64 accumulation is what
// its entry point promises): the lanes are folded into fp64 every 64 positions per lane, and the slabs are fp64.  gw
// (bfloat16 storage, one slab): the finished gradient sum x g - w sum g goes there, and there are no slabs.
template <class T> using GwSum1x1 = std::conditional_t<sizeof(T) == 4, float, double>;

template <int S, int TM, int TC, bool VEC = true, class T = float>
__global__ __launch_bounds__(256) void grad_w_1x1_kernel(const T *__restrict__ gy, const T *__restrict__ x,
                                                         GwSum1x1<T> *__restrict__ part, GwSum1x1<T> *__restrict__ sgpart,
                                                         const float *__restrict__ w, float *__restrict__ gw, int N, int Ci,
                                                         int H, int W, int Co, int Ho, int Wo, int gpr, int groups) {
    using P = GwSum1x1<T>;
    constexpr bool WIDE = sizeof(P) == 8;
    constexpr int TN = 4 / S, A = TM * TC, TOT = A + TM, RUN = 64 / TN;   // RUN: position groups between two folds (WIDE)
    const int co0 = blockIdx.y * TM, ci0 = blockIdx.z * TC;
    const size_t plane = (size_t)H * W, gplane = (size_t)Ho * Wo;
    __shared__ float red[4][64 * 17];
    __shared__ P wsum[4][TOT];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    float acc[TM][TC], sg[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) {
        sg[m] = 0.f;
#pragma unroll
        for (int c = 0; c < TC; ++c) acc[m][c] = 0.f;
    }
    auto fold = [&](const bool first) {   // the sums of the wave's lanes into (first) or onto wsum; acc and sg restart
        float all[TOT];
#pragma unroll
        for (int a = 0; a < A; ++a) { all[a] = acc[a / TC][a % TC]; acc[a / TC][a % TC] = 0.f; }
#pragma unroll
        for (int m = 0; m < TM; ++m) { all[A + m] = sg[m]; sg[m] = 0.f; }
        constexpr int ROUNDS = ceil_div(TOT, 16);
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
#pragma unroll
            for (int e = 0; e < 16; ++e) red[wave][lane * 17 + e] = (r * 16 + e < TOT) ? all[(r * 16 + e) % TOT] : 0.f;
            __syncthreads();
            const int e = lane & 15, rg = lane >> 4;
            P s = P(0);
#pragma unroll
            for (int k = 0; k < 16; ++k) s += (P)red[wave][(rg * 16 + k) * 17 + e];
            s += __shfl_xor(s, 16, 64);
            s += __shfl_xor(s, 32, 64);
            if (rg == 0 && r * 16 + e < TOT) wsum[wave][r * 16 + e] = first ? s : wsum[wave][r * 16 + e] + s;
            __syncthreads();
        }
    };
    auto step = [&](const int g0) {
        const Lane1x1<S> L(g0, groups, gpr, Ho);
        const T *xp = x + (size_t)L.n * Ci * plane + (size_t)(L.ho * S) * W + L.wo0 * S;
        const T *gp = gy + (size_t)L.n * Co * gplane + (size_t)L.ho * Wo + L.wo0;
        const int valid = W - L.wo0 * S;   // only read when !VEC
        float xs[TC][TN], gs[TM][TN];
#pragma unroll
        for (int c = 0; c < TC; ++c) {
            const float4 v = ld4<VEC>(xp + (size_t)min(ci0 + c, Ci - 1) * plane, valid);
            const float t4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int t = 0; t < TN; ++t) xs[c][t] = t4[t * S];
        }
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            const T *p = gp + (size_t)min(co0 + m, Co - 1) * gplane;
            if constexpr (TN == 4) {
                const float4 v = ld4<VEC>(p, valid);
                gs[m][0] = v.x; gs[m][1] = v.y; gs[m][2] = v.z; gs[m][3] = v.w;
            } else {
                const float2 v = ld2<VEC>(p, Wo - L.wo0);
                gs[m][0] = v.x; gs[m][1] = v.y;
            }
        }
#pragma unroll
        for (int m = 0; m < TM; ++m) {
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                sg[m] += gs[m][t];
#pragma unroll
                for (int c = 0; c < TC; ++c) acc[m][c] = fmaf(gs[m][t], xs[c][t], acc[m][c]);
            }
        }
    };
    bool first = true;
    if constexpr (WIDE) {
        int run = 0;
        for (int base = blockIdx.x * 256; base < groups; base += gridDim.x * 256) {   // (uniform: fold has barriers)
            if (base + (int)threadIdx.x < groups) step(base + threadIdx.x);
            if (++run == RUN) { fold(first); first = false; run = 0; }
        }
    } else {
        for (int g0 = blockIdx.x * 256 + threadIdx.x; g0 < groups; g0 += gridDim.x * 256) step(g0);
    }
    // the last positions, then the 4 waves of the workgroup
    fold(first);
    if (threadIdx.x < TOT) {
        const int a = threadIdx.x;
        const P s = (wsum[0][a] + wsum[1][a]) + (wsum[2][a] + wsum[3][a]);
        const int co = co0 + (a < A ? a / TC : a - A), ci = ci0 + a % TC;
        if (WIDE && gw) {
            if (a < A && co < Co && ci < Ci) {
                const int b = A + a / TC;
                const P sum_g = (wsum[0][b] + wsum[1][b]) + (wsum[2][b] + wsum[3][b]);
                gw[(size_t)co * Ci + ci] = (float)(s - (P)w[(size_t)co * Ci + ci] * sum_g);
            }
        } else if (a < A) {
            if (co < Co && ci < Ci) part[(size_t)blockIdx.x * Co * Ci + (size_t)co * Ci + ci] = s;
        } else if (blockIdx.z == 0) {
            if (co < Co) sgpart[(size_t)blockIdx.x * Co + co] = s;
        }
    }
}

// ---- host side ------------------------------------------------------------------
// Stride 1: positions are independent, so every (H, W) plane is walked as one row of H*W elements; planes
// whose size is not a multiple of 4 (7x7) or whose base is not 16-byte aligned take the element-wise loads.
// Stride 2: one float4 of the source row per lane (two of its elements are sampled) and a float2 of the
// output row; rows that are not whole aligned groups (W % 4, Wo % 2, base pointers) are read element-wise.
// (For bfloat16 storage the groups of four are 8 bytes.)
bool conv1x1_supported(const ConvDims &d, const void *, const void *) {
    return d.kh == 1 && d.kw == 1 && d.pad == 0 && (d.stride == 1 || d.stride == 2);
}

// dimensions the kernels are launched with
static ConvDims lane_dims(const ConvDims &d) {
    ConvDims f = d;
    if (d.stride == 1) { f.H = 1; f.W = d.H * d.W; f.Ho = 1; f.Wo = d.H * d.W; }
    return f;
}

template <class T>
static bool vec_ok(const ConvDims &f, const T *a, const T *b, const T *c) {
    const bool aligned = aligned_groups(a) && aligned_groups(b) && aligned_groups(c);
    if (f.stride == 2) return f.W % 4 == 0 && f.Wo % 2 == 0 && aligned;
    return f.W % 4 == 0 && aligned;
}

static void lane_space(const ConvDims &f, int &gpr, int &groups) {
    gpr = ceil_div(f.Wo, 4 / f.stride);
    groups = f.N * f.Ho * gpr;
}

// partial-sum slots per channel of the statistics epilogue (one per wave of the launch)
int fwd_1x1_stats_slots(const ConvDims &d) {
    const ConvDims f = lane_dims(d);
    int gpr, groups;
    lane_space(f, gpr, groups);
    return ceil_div(groups, 256) * 4;
}

// stats (nullable): per-channel partial sums of y and y*y, fwd_1x1_stats_slots(d) slots per channel
template <class T>
int launch_fwd_1x1(const T *x, const float *w, T *y, double *stats, const ConvDims &d, hipStream_t s, const BnEval &bn) {
    constexpr int TM = 8;
    const ConvDims f = lane_dims(d);
    int gpr, groups;
    lane_space(f, gpr, groups);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(ceil_div(groups, 256), ceil_div(f.Co, TM)), dim3(256), 0, s, x, w, y, stats, f.N, f.Ci,
                           f.H, f.W, f.Co, f.Ho, f.Wo, gpr, groups, bn);
        return check_launch();
    };
    const bool vec = vec_ok<T>(f, x, y, nullptr);
    if (f.stride == 2) return vec ? launch(fwd_1x1_kernel<2, TM, true, T>) : launch(fwd_1x1_kernel<2, TM, false, T>);
    return vec ? launch(fwd_1x1_kernel<1, TM, true, T>) : launch(fwd_1x1_kernel<1, TM, false, T>);
}
template int launch_fwd_1x1<float>(const float *, const float *, float *, double *, const ConvDims &, hipStream_t, const BnEval &);
template int launch_fwd_1x1<bf16_t>(const bf16_t *, const float *, bf16_t *, double *, const ConvDims &, hipStream_t,
                                    const BnEval &);

template <class T>
int launch_grad_x_1x1(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s) {
    constexpr int TM = kGx1x1TM;
    const ConvDims f = lane_dims(d);
    int gpr, groups;
    lane_space(f, gpr, groups);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(ceil_div(groups, 256), ceil_div(f.Ci, TM)), dim3(256), 0, s, gy, x, w, gx, f.N, f.Ci,
                           f.H, f.W, f.Co, f.Ho, f.Wo, gpr, groups);
        return check_launch();
    };
    const bool vec = vec_ok<T>(f, gy, x, gx);
    if (f.stride == 2) return vec ? launch(grad_x_1x1_kernel<2, TM, true, T>) : launch(grad_x_1x1_kernel<2, TM, false, T>);
    return vec ? launch(grad_x_1x1_kernel<1, TM, true, T>) : launch(grad_x_1x1_kernel<1, TM, false, T>);
}
template int launch_grad_x_1x1<float>(const float *, const float *, const float *, float *, const ConvDims &, hipStream_t);
template int launch_grad_x_1x1<bf16_t>(const bf16_t *, const bf16_t *, const float *, bf16_t *, const ConvDims &, hipStream_t);

static constexpr int kGw1x1TM = 8, kGw1x1TC = 8;

int grad_w_1x1_slots(const ConvDims &d) {
    const ConvDims f = lane_dims(d);
    int gpr, groups;
    lane_space(f, gpr, groups);
    const int blocks_yz = ceil_div(f.Co, kGw1x1TM) * ceil_div(f.Ci, kGw1x1TC);
    int want = ceil_div(1024, blocks_yz);                 // ~4 workgroups per CU
    const int cap = ceil_div(groups, 256 * 4);            // at least 4 position groups per lane
    if (want > cap) want = cap;
    return want < 1 ? 1 : want;
}

// bfloat16 storage, 48 -> 48 @64x64, 64 images: generic kernel 1219 us, fp32 sums and slabs 52, fp64 ones 52.5; 32 -> 1024 @28x28, 256
// images: 11 125, 354 and 376.
template <class T, class P>
int launch_grad_w_1x1(const T *gy, const T *x, P *part, P *sgpart, const float *w, float *gw, int slots, const ConvDims &d,
                      hipStream_t s) {
    static_assert(std::is_same<P, GwSum1x1<T>>::value, "fp32 slabs for float storage, fp64 for bfloat16");
    constexpr int TM = kGw1x1TM, TC = kGw1x1TC;
    const ConvDims f = lane_dims(d);
    int gpr, groups;
    lane_space(f, gpr, groups);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(slots, ceil_div(f.Co, TM), ceil_div(f.Ci, TC)), dim3(256), 0, s, gy, x, part, sgpart, w,
                           gw, f.N, f.Ci, f.H, f.W, f.Co, f.Ho, f.Wo, gpr, groups);
        return check_launch();
    };
    const bool vec = vec_ok<T>(f, gy, x, nullptr);
    if (f.stride == 2)
        return vec ? launch(grad_w_1x1_kernel<2, TM, TC, true, T>) : launch(grad_w_1x1_kernel<2, TM, TC, false, T>);
    return vec ? launch(grad_w_1x1_kernel<1, TM, TC, true, T>) : launch(grad_w_1x1_kernel<1, TM, TC, false, T>);
}
template int launch_grad_w_1x1<float, float>(const float *, const float *, float *, float *, const float *, float *, int,
                                             const ConvDims &, hipStream_t);
template int launch_grad_w_1x1<bf16_t, double>(const bf16_t *, const bf16_t *, double *, double *, const float *, float *, int,
                                               const ConvDims &, hipStream_t);

}  // namespace adder

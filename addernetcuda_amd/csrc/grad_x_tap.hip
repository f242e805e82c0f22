// Input gradient of 1x1 / stride-1 layers from four input and 16 output channels on, NCHW:
//   gx[n,ci,p] = sum_co hardtanh(w[co,ci] - x[n,ci,p]) * gy[n,co,p]      (adder_cuda/adder.cu:133-272)
//
// The terms are those of grad_x.hip (two vector instructions, three above kSatMaxTerms1x1 output channels) and bound it: 90 us for
// 3.3e9 of them at 73 T lane-instructions/s.  As in fwd_tap.hip nothing is staged: a lane owns 16 input channels x 2 positions,
// reads gy of its positions four output channels ahead, the 16 weights of an output channel are one scalar load of a whole line, and
// the KSP waves of a workgroup share the output channels, so that planes of 14x14 and 7x7 and few images still fill the chip.
// Sums of sums live in LDS (once per 64 terms): 96 registers, two waves on each issue port; in registers 16 x 1 or 8 x 2 positions
// fit, 168 and 165 us where this takes 141 (512 -> 256 @28x28, 32 images).
// us, 128 positions x 64 channels with gy staged in LDS -> this: 32 images 64 -> 256 @56x56 104 -> 80, 256 -> 64 92 -> 81, 256 -> 128
// 157 -> 145, 128 -> 512 @28x28 107 -> 80, 512 -> 256 167 -> 140, 256 -> 1024 @14x14 169 -> 89, 1024 -> 256 105 -> 77, 512 -> 2048 @7x7
// 242 -> 118, 2048 -> 512 127 -> 84; one image: 256 -> 1024 @14x14 153 -> 17, 64 -> 256 @56x56 42 -> 9.
#include "wave_split.hpp"

#include <type_traits>

namespace adder {

// TM input channels x TN adjacent positions per lane, KSP waves: wave v takes the chunks v, v + KSP, ... of output channels
template <int TM_, int TN_, int KSP_>
struct GxTapCfg {
    static constexpr int TM = TM_, TN = TN_, KSP = KSP_, NT = 64 * KSP, CC = kTapChunk, FM = TM / KSP;
    static constexpr int PART = KSP * TM * TN * 64, LDS_BYTES = PART * 4 + KSP * TN * 64 * 8;
    static_assert(TM % KSP == 0, "every wave finishes the same number of channels");
};

struct GxTapDims {
    int N, Ci, Co, L;       // L = H * W positions per image
    int strips;             // of TN positions per image; the last one of an image is moved back to end at L
    int tiles, blocks;      // of 64 strips, of TM input channels
};

// SAT, FUSE, gadd, bn: as in grad_x_3x3s1_kernel (one slot of sums per tile; FUSE: float storage).
template <class C, bool SAT, class T, bool FUSE>
__global__ __launch_bounds__(C::NT, 4) void grad_x_tap_kernel(const T *__restrict__ gy, const T *__restrict__ x, const float *__restrict__ w,
                                                           T *__restrict__ gx, const GxTapDims d, const T *__restrict__ gadd,
                                                           const adder_bn_links bn) {
    constexpr int TM = C::TM, TN = C::TN, KSP = C::KSP, CQ = 4, CU = 2, NU = CQ / CU, FM = C::FM;
    extern __shared__ __align__(16) float smem[];
    int tile, blk;
    xcd_tile(blockIdx.x, d.tiles, d.blocks, tile, blk);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int sidx = tile * 64 + lane, sc = min(sidx, d.N * d.strips - 1), n = sc / d.strips, s = sc - n * d.strips;
    const int p0 = min(s * TN, d.L - TN);
    const int n_first = __builtin_amdgcn_readfirstlane(n);
    // the last group of channels is shifted down to end at Ci; channels below ci_first are not stored by it
    const int ci_first = blk * TM, ci_base = min(ci_first, d.Ci - TM);
    uniform_f32_ptr wc = as_uniform(w) + ci_base;

    float cr[TM][TN], acc[TM][TN];
    float *tot = smem + wave * (TM * TN * 64) + lane;   // sums of sums: this wave's part, [channel][position][lane]
    bool first = true;
    {
        const T *src = x + ((size_t)n * d.Ci + ci_base) * d.L + p0;
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            float xv[TN];
            ld_strip<TN>(src + (size_t)m * d.L, xv);
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                cr[m][t] = SAT ? fmaf(-0.5f, xv[t], 0.5f) : xv[t];
                acc[m][t] = 0.f;
            }
        }
    }
    const unsigned goff = (unsigned)((n - n_first) * d.Co * d.L + p0) * (unsigned)sizeof(T);
    const T *g_first = gy + (size_t)n_first * d.Co * d.L;
    float gr[2][CQ][TN], wv[2][CU][TM];
    float gs[TN];
    double gsum[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t) gs[t] = 0.f, gsum[t] = 0.0;
    auto load_g = [&](const int b, const int co) {
#pragma unroll
        for (int e = 0; e < CQ; ++e)
            ld_strip<TN>(reinterpret_cast<const T *>(reinterpret_cast<const char *>(g_first + (size_t)min(co + e, d.Co - 1) * d.L) + goff), gr[b][e]);
    };
    auto load_w = [&](const int b, const int co) {
#pragma unroll
        for (int u = 0; u < CU; ++u) {
            const int row = min(co + u, d.Co - 1) * d.Ci;
#pragma unroll
            for (int m = 0; m < TM; ++m) wv[b][u][m] = wc[row + m];
        }
    };
    int co = wave * C::CC, chunks = 0;
    if (co < d.Co) {
        load_g(0, co);
        load_w(0, co);
        auto half = [&](const int cur) -> bool {
            int next = co + CQ;
            const bool chunk_end = (next & (C::CC - 1)) == 0;
            if (chunk_end) next += (KSP - 1) * C::CC;
            const bool more = next < d.Co;
            const int cn = more ? next : co;
            if (co + CQ > d.Co) {   // channels past Co: nothing to add
#pragma unroll
                for (int e = 1; e < CQ; ++e)
                    if (co + e >= d.Co) {
#pragma unroll
                        for (int t = 0; t < TN; ++t) gr[cur][e][t] = 0.f;
                    }
            }
#pragma unroll
            for (int h = 0; h < NU; ++h) {
                const int wb = (cur * (NU & 1) + h) & 1;
#pragma unroll
                for (int idx = 0; idx < CU * TM * TN; ++idx) {
                    const int t = idx % TN, m = (idx / TN) % TM, u = idx / TN / TM, e = h * CU + u;
                    const float wgt = wv[wb][u][m];
                    const float dd = SAT ? sat01(fmaf(wgt, 0.5f, cr[m][t])) : hardtanh(wgt - cr[m][t]);
                    acc[m][t] = fmaf(dd, gr[cur][e][t], acc[m][t]);
                    if (idx == 0) {
                        __builtin_amdgcn_sched_barrier(0);
                        load_w(wb ^ 1, h + 1 < NU ? co + (h + 1) * CU : cn);
                        if (h == 0) load_g(cur ^ 1, cn);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            if constexpr (SAT) {
#pragma unroll
                for (int e = 0; e < CQ; ++e)
#pragma unroll
                    for (int t = 0; t < TN; ++t) gs[t] += gr[cur][e][t];
            }
            co = next;
            if (chunk_end || !more) {
                if constexpr (SAT) {
#pragma unroll
                    for (int t = 0; t < TN; ++t) { gsum[t] += (double)gs[t]; gs[t] = 0.f; }
                }
                if ((++chunks & 3) == 0 || !more) {   // 64-term first levels
#pragma unroll
                    for (int m = 0; m < TM; ++m)
#pragma unroll
                        for (int t = 0; t < TN; ++t) {
                            float *p = tot + (m * TN + t) * 64;
                            *p = first ? acc[m][t] : *p + acc[m][t];
                            acc[m][t] = 0.f;
                        }
                    first = false;
                }
            }
            return more;
        };
#pragma unroll 1
        while (half(0) && half(1)) {}
    }

    double *gpart = reinterpret_cast<double *>(smem + C::PART);
    if (first) {   // no channels for this wave
#pragma unroll
        for (int e = 0; e < TM * TN; ++e) tot[e * 64] = 0.f;
    }
    if constexpr (SAT) {
#pragma unroll
        for (int t = 0; t < TN; ++t) gpart[(wave * TN + t) * 64 + lane] = gsum[t];
    }
    __syncthreads();
    const int m0 = wave * FM, ci0 = ci_base + m0;
    float r[FM][TN], sg[TN];
    if constexpr (SAT) {
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            double v = gpart[t * 64 + lane];
#pragma unroll
            for (int k = 1; k < KSP; ++k) v += gpart[(k * TN + t) * 64 + lane];
            sg[t] = (float)v;
        }
    }
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            float v = smem[((m0 + f) * TN + t) * 64 + lane];
#pragma unroll
            for (int k = 1; k < KSP; ++k) v += smem[((k * TM + m0 + f) * TN + t) * 64 + lane];
            r[f][t] = SAT ? fmaf(2.f, v, -sg[t]) : v;
        }
    unsigned own = 0;   // bit t: position p0 + t is this lane's
#pragma unroll
    for (int t = 0; t < TN; ++t) own |= (sidx == sc && p0 + t >= s * TN ? 1u : 0u) << t;
    // the last group of channels is shifted down to end at Ci; channels below ci_first are not stored by it
    finish_grad_x<FM, TN, FUSE>(r, own, ci0, max(ci_first, ci0), d.Ci, d.L, (n * d.Ci + ci0) * d.L + p0, TN > 1 && d.L % TN == 0, x, gx, gadd, bn,
                                d.tiles, tile, lane);
}

static int gx_tap_tiles(const ConvDims &d, int tn) { return (int)ceil_div_l((long)d.N * ceil_div(d.H * d.W, tn), 64); }

// Which shape a layer takes: input channels and positions per lane, waves that share the output channels.  By the work a wave of 16
// channels x 2 positions would have (its output channels) and the workgroups there are of them.
//   - at most 128 workgroups: 8 x 1, eight waves (us, 16 x 2 -> 8 x 1: 56 workgroups, 128 -> 512 @28x28, one image, 15.3 -> 9.2; 100
//     workgroups 9.8 -> 8.0; 224 workgroups, 512 -> 128 @28x28, 7.2 -> 9.4)
//   - up to 128 output channels one wave does them all (1 / 4 / 8 waves: 256 -> 64 @56x56, 32 images, 84 / 96 / 141; 84 -> 48 @32x32, 64
//     images, 3072 workgroups, 21 / 24 / 35), four where there are few workgroups (512 -> 128 @28x28, 8 images, 1568 workgroups, 29 / 25 / 29)
//   - up to 512 four (64 -> 256 @56x56, 32 images, 90 / 74 / 80), above eight (256 -> 1024 @14x14, 186 / 89 / 85; 512 -> 2048 @7x7 456 / 123 / 113),
//     and eight where there are few workgroups (512 -> 128 @28x28, one image, 25 / 8.9 / 7.2)
struct GxTapShape { int tm, tn, waves; };
static GxTapShape gx_tap_shape(const ConvDims &d) {
    const long wgs = (long)gx_tap_tiles(d, 2) * ceil_div(d.Ci, 16);
    if (d.H * d.W < 2 || wgs <= 128) return {8, 1, 8};
    if (wgs < 448 || d.Co > 512) return {16, 2, 8};
    return {16, 2, d.Co <= 128 && wgs >= 2048 ? 1 : 4};
}

// Layers it takes; the distance of a wave's strips from the first one's image has to fit 32 bits.  (The launch's threads do for tensors below 2^31
// elements: eight waves share 512 output channels or a few hundred workgroups only, and four of them have 4 x 2 results a lane at least.)
static bool gx_tap_fits(const ConvDims &d) {
    const long L = (long)d.H * d.W;
    return (images_ahead(d, ceil_div_l(L, 2)) * d.Co + 1) * L <= 0x3fffffffL;
}
bool grad_x_tap_supported(const ConvDims &d) {
    if (d.kh != 1 || d.kw != 1 || d.pad != 0 || d.stride != 1 || d.Ci < 64 || d.Co < 48) return false;
    return gx_tap_fits(d);
}
// Layers of fewer channels that no BatchNorm is linked to and nothing is added to: three instructions a term, error 7e-8 to 1.4e-7 of the result where
// conv1x1.hip, which walks all output channels in one wave, has 1.4e-7 to 2.9e-7.  us, conv1x1.hip -> this: 7 -> 482 @10x10, 12 images, 91 -> 14.5, 24 -> 300 @8x8, 64
// images, 59 -> 7.4, 7 -> 227 @41x40, 26 images, bfloat16, 93 -> 13, 32 -> 200 @56x56, 64 images, 185 -> 86, 40 -> 16 @64x64, 200 images, 111 -> 61, 24 -> 48 @32x32, 64 images,
// 15.1 -> 12.6, 10 -> 23 @9x9, five, 9.5 -> 7.0, 4 -> 16 @64x64, 64 images, 7.0 -> 7.3; left there: 51 -> 15 @64x64, 23 images, bfloat16, 12.5 -> 13.4, 200 -> 24 @16x16, 64
// images, 13.9 -> 15.3.
bool grad_x_tap_narrow(const ConvDims &d) {
    if (d.kh != 1 || d.kw != 1 || d.pad != 0 || d.stride != 1 || d.Ci < 4 || d.Co < (d.Ci < 64 ? 16 : 32)) return false;
    return gx_tap_fits(d);
}
int grad_x_tap_bn_slots(const ConvDims &d) { return gx_tap_tiles(d, gx_tap_shape(d).tn); }

template <class C, bool SAT, class T, bool FUSE>
static int launch_gx_tap(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s, const T *gadd,
                         const adder_bn_links &bn) {
    const GxTapDims t{d.N, d.Ci, d.Co, d.H * d.W, ceil_div(d.H * d.W, C::TN), gx_tap_tiles(d, C::TN), ceil_div(d.Ci, C::TM)};
    if (FUSE && (!bn.in_part || bn.in_slots != t.tiles)) return ADDER_ERR_BAD_SHAPE;
    if (int rc = allow_dynamic_lds<&grad_x_tap_kernel<C, SAT, T, FUSE>>(C::LDS_BYTES)) return rc;
    hipLaunchKernelGGL((grad_x_tap_kernel<C, SAT, T, FUSE>), dim3((unsigned)t.tiles * t.blocks), dim3(C::NT), C::LDS_BYTES, s, gy, x, w, gx, t,
                       gadd, bn);
    return check_launch();
}

// The three-instruction form rounds once less (error 8.7e-8 of the result, two instructions 1.58e-7) and costs a small launch nothing
// (8 x 1: 128 -> 512 @28x28 9.5 -> 9.2 us, 64 -> 256 @56x56 8.3 -> 8.5); planes that no BatchNorm can be linked to have it with eight
// waves too (1024 -> 256 @14x14, 8 images, which can: 26.5 -> 31.9), and so have narrow layers and small ones without a link (small_unlinked).
GradXShape grad_x_tap_shape(const ConvDims &d, bool bf16) {
    const GxTapShape shape = gx_tap_shape(d);
    if (d.Ci < 8) return {4, d.H * d.W >= 2 ? 2 : 1, 4, false};   // (no link and no second gradient: grad_x_tap_narrow)
    if (d.Ci < 16) return {8, shape.tn, shape.tn == 1 ? 8 : 4, false};
    const bool exact = shape.tm == 8 || !grad_x_tap_supported(d) || (shape.waves == 8 && (d.H * d.W) % 4 != 0) ||
                       small_unlinked(d, bf16);
    return {shape.tm, shape.tn, shape.waves, !exact && d.Co <= kSatMaxTerms1x1};
}

// bn (nullable): the in_* half of adder_bn_links
template <class T>
int launch_grad_x_tap(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s, const T *gadd,
                      const adder_bn_links *bn) {
    const GradXShape shape = grad_x_tap_shape(d, sizeof(T) == 2);
    if (d.Ci < 16) {
        auto narrow = [&](auto cfg) { return launch_gx_tap<decltype(cfg), false, T, false>(gy, x, w, gx, d, s, gadd, adder_bn_links{}); };
        if (shape.tm == 4) return shape.tn == 2 ? narrow(GxTapCfg<4, 2, 4>{}) : narrow(GxTapCfg<4, 1, 4>{});
        return shape.tn == 1 ? narrow(GxTapCfg<8, 1, 8>{}) : narrow(GxTapCfg<8, 2, 4>{});
    }
    auto run = [&](auto cfg) {
        using C = decltype(cfg);
        auto form = [&](auto sat) {
            constexpr bool SAT = decltype(sat)::value;
            if constexpr (sizeof(T) == 4) {
                if (bn) return launch_gx_tap<C, SAT, T, true>(gy, x, w, gx, d, s, gadd, *bn);
            }
            return launch_gx_tap<C, SAT, T, false>(gy, x, w, gx, d, s, gadd, adder_bn_links{});
        };
        return shape.two ? form(std::true_type{}) : form(std::false_type{});
    };
    if (shape.tm == 8) return run(GxTapCfg<8, 1, 8>{});
    return shape.waves == 1 ? run(GxTapCfg<16, 2, 1>{}) : shape.waves == 4 ? run(GxTapCfg<16, 2, 4>{}) : run(GxTapCfg<16, 2, 8>{});
}
template int launch_grad_x_tap<float>(const float *, const float *, const float *, float *, const ConvDims &, hipStream_t,
                                      const float *, const adder_bn_links *);
template int launch_grad_x_tap<bf16_t>(const bf16_t *, const bf16_t *, const float *, bf16_t *, const ConvDims &, hipStream_t,
                                       const bf16_t *, const adder_bn_links *);

}  // namespace adder

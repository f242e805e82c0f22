// Input gradient of 3x3 / pad 1 and 5x5 / pad 2 layers of stride 2, NCHW:
//   gx[n,ci,h,w] = sum_{co} sum_{i,j: h+p-i, w+p-j even} hardtanh(w[co,ci,i,j] - x[n,ci,h,w]) * gy[n,co,(h+p-i)/2,(w+p-j)/2]
// Replaces the grad_i half of adder_cuda/adder.cu:194-272, adder.cu:133-192 and the fold of adder.py:32-33.
//
// A tap reaches positions of one parity only, so a block of 2 x 2 input positions meets each tap once, and the gy it needs are the 2 x 2
// (5x5: 3 x 3) outputs around its own.  A lane owns one block of TM input channels; as in grad_x_nine.hip it reads its
// window of gy straight into registers one (5x5) or three output channels ahead, the blocks of all images line up, and the waves of a
// workgroup share the output channels.  Maps of any size: ceil(H / 2) x ceil(W / 2) blocks are the outputs, what lies behind an odd edge is not stored.
// Rows of whole groups of eight keep the tiles of grad_x.hip, which carry the BatchNorm link.
//
// Three vector instructions per term (two for the layers that had them in tiles: rows of an even length, at most kSatMaxTerms terms) bound
// it, and a weight meets one position only, so that scalar loads and the reads of gy are what competes with them.  us, one position per lane from
// memory (the kernel for any layer), or tiles for rows of an even length -> this: 533 -> 113 @19x19, 28 images, 1452 -> 124; 498 -> 124 @10x9, 225 images,
// bfloat16, 2801 -> 257; 107 -> 278 @23x23, 5 images, 897 -> 25; 5x5: 6 -> 897 @41x49, 27 images, bfloat16, 8345 -> 150, 7 -> 144 @23x26, 202 images,
// 1415 -> 66, 23 -> 182 @31x39, 5 images, 1482 -> 25; even rows: 512 -> 512 @14x14, 32 images, 320 -> 247, 256 -> 256 @28x28 218 -> 212, one image
// 73 -> 18, 27 -> 968 @52x52, 16 images, 389 -> 173.  Error against float64 1.1e-7 to 1.7e-7 of the result (tiles 1.6e-7 to 2.2e-7).
// Tried on the way: 4 channels x 2 blocks per lane 256 -> 256 @28x28 239 -> 313 (four waves per SIMD instead of eight); 8 channels x one block 224
// with two instructions a term, but 512 -> 512 @14x14 271 -> 333; the weights of a block's channels asked for one channel at a time 257.
#include "wave_split.hpp"

#include <type_traits>

namespace adder {

// KS: 3 or 5; TM input channels of one block per lane; KSP waves that share the output channels in chunks of CC
template <int KS_, int TM_, int KSP_>
struct GxS2Cfg {
    static constexpr int KS = KS_, TM = TM_, KSP = KSP_, NT = 64 * KSP, CC = kNineChunk, PAD = KS / 2;
    static constexpr int ROWS = 2 * TM, FM = kFinished<ROWS, KSP>;   // rows (channel, parity) of two positions; those a wave finishes
    static constexpr int FIRST = KS == 5 ? -1 : 0, WIN = (KS + 1) / 2, RIGHT = WIN - 1;   // window of gy around block (a, b): rows a + FIRST ...
    static constexpr int AHEAD = KS == 5 ? 1 : 3;                                 // output channels that gy is asked for ahead of the arithmetic
    static constexpr int UM = KS == 3 ? 2 : 1, NU = TM / UM;                      // input channels whose weights are asked for together, a step ahead
    static constexpr int PART = KSP * ROWS * 2 * 64, SAT_BYTES = KSP * 4 * 64 * 8;   // sums in LDS: PART floats, with SAT also these
    static_assert((ROWS % KSP == 0 || KSP % ROWS == 0) && (NU == 1 || NU % 2 == 0), "a wave finishes FM rows or none; two weight buffers");
};

struct GxS2Dims {
    int N, Ci, H, W, Co, Ho, Wo;
    int tiles, blocks;      // of 64 blocks of positions, of TM input channels (the last ones are moved back to end at Ci)
};

// SAT, gadd: as in grad_x_3x3s1_kernel.
template <class C, bool SAT, class T>
__global__ __launch_bounds__(C::NT, 4) void grad_x_s2_kernel(const T *__restrict__ gy, const T *__restrict__ x, const float *__restrict__ w,
                                                             T *__restrict__ gx, const GxS2Dims d, const T *__restrict__ gadd) {
    constexpr int KS = C::KS, KK = KS * KS, PAD = C::PAD, TM = C::TM, ROWS = C::ROWS, KSP = C::KSP, FM = C::FM;
    constexpr int FIRST = C::FIRST, WIN = C::WIN, RIGHT = C::RIGHT, NB = C::AHEAD + 1, UM = C::UM, NU = C::NU;
    extern __shared__ __align__(16) float smem[];
    int tile, blk;
    xcd_tile(blockIdx.x, d.tiles, d.blocks, tile, blk);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int sidx = tile * 64 + lane, L = d.Ho * d.Wo, sc = min(sidx, d.N * L - 1), n = sc / L, rest = sc - n * L;
    const int a = rest / d.Wo, b0 = rest - a * d.Wo, ci_first = blk * TM, ci_base = min(ci_first, d.Ci - TM), plane = d.H * d.W, K = d.Ci * KK;
    const bool even = d.W % 2 == 0;   // both positions of a block row lie inside the map
    uniform_f32_ptr wc = as_uniform(w);
    float cr[ROWS][2], acc[ROWS][2];   // row 2 m + p: input row 2 a + p of channel m
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
        const T *p = x + ((size_t)n * d.Ci + ci_base + q / 2) * plane + min(2 * a + q % 2, d.H - 1) * d.W + 2 * b0;
        float xv[2];
        if (even) {
            ld_strip<2>(p, xv);
        } else {
#pragma unroll
            for (int t = 0; t < 2; ++t) xv[t] = ldf(p + min(t, d.W - 1 - 2 * b0));
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            cr[q][t] = SAT ? fmaf(-0.5f, xv[t], 0.5f) : xv[t];
            acc[q][t] = 0.f;
        }
    }
    // sums of sums in LDS: this wave's part, [row][position][lane]; and of the gy values the positions met, [parity][position][lane]
    float *tot = smem + wave * (ROWS * 2 * 64) + lane;
    double *gtot = reinterpret_cast<double *>(smem + C::PART) + wave * (2 * 2 * 64) + lane;
    bool first = true;

    // a uniform base per channel and the lane's distances from it in bytes, as in fwd_nine.hip
    const int n_first = __builtin_amdgcn_readfirstlane(n);
    const T *g_first = gy + (size_t)n_first * d.Co * L;
    const bool ok_l = b0 > 0, ok_r = b0 + 1 < d.Wo;
    bool ok[WIN];
    unsigned off[WIN], off_l[WIN], off_r[WIN];
#pragma unroll
    for (int i = 0; i < WIN; ++i) {
        const int r = a + FIRST + i;
        ok[i] = r >= 0 && r < d.Ho;
        const int o = (n - n_first) * d.Co * L + min(max(r, 0), d.Ho - 1) * d.Wo + b0;
        off[i] = (unsigned)o * (unsigned)sizeof(T);
        off_l[i] = (unsigned)(ok_l ? o - 1 : o) * (unsigned)sizeof(T);
        off_r[i] = (unsigned)(ok_r ? o + 1 : o) * (unsigned)sizeof(T);
    }
    float gr[NB][WIN][WIN], wv[2][UM][KK], gs[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) gs[0][t] = gs[1][t] = 0.f;
    auto load_g = [&](const int b, const int co) {
        const char *p = reinterpret_cast<const char *>(g_first + (size_t)co * L);
#pragma unroll
        for (int i = 0; i < WIN; ++i) {
            keep_offset(off[i]); keep_offset(off_r[i]);
            gr[b][i][-FIRST] = ldf(reinterpret_cast<const T *>(p + off[i]));
            if constexpr (FIRST != 0) {
                keep_offset(off_l[i]);
                gr[b][i][0] = ldf(reinterpret_cast<const T *>(p + off_l[i]));
            }
            gr[b][i][RIGHT] = ldf(reinterpret_cast<const T *>(p + off_r[i]));
        }
    };
    auto load_w = [&](const int b, const int hh, const int co) {   // (the channels of a block are one run of memory)
        uniform_f32_ptr wrow = wc + (co * K + ci_base * KK);
#pragma unroll
        for (int u = 0; u < UM; ++u)
#pragma unroll
            for (int e = 0; e < KK; ++e) wv[b][u][e] = wrow[(hh * UM + u) * KK + e];
    };
    auto after = [&](const int c) { return ((c + 1) & (C::CC - 1)) == 0 ? c + 1 + (KSP - 1) * C::CC : c + 1; };
    int co = wave * C::CC;
    if (co < d.Co) {
        int cl = co;   // the channel that gy is read of next (the last one again behind the end)
#pragma unroll
        for (int b = 0; b < C::AHEAD; ++b) {
            load_g(b, cl);
            const int c = after(cl);
            cl = c < d.Co ? c : cl;
        }
        load_w(0, 0, co);
        auto channel = [&](const int cur) -> bool {
            const int next = after(co);
            const bool chunk_end = ((co + 1) & (C::CC - 1)) == 0, more = next < d.Co;
            const int cn = more ? next : co;
#pragma unroll
            for (int i = 0; i < WIN; ++i) {   // positions outside gy contribute nothing
                if (i != -FIRST) gr[cur][i][-FIRST] = ok[i] ? gr[cur][i][-FIRST] : 0.f;
                if constexpr (FIRST != 0) gr[cur][i][0] = ok[i] && ok_l ? gr[cur][i][0] : 0.f;
                gr[cur][i][RIGHT] = ok[i] && ok_r ? gr[cur][i][RIGHT] : 0.f;
            }
            // tap (i, j) reaches position (p, t) of the block where p + PAD - i and t + PAD - j are even, with window element
            // ((p + PAD - i) / 2 - FIRST, (t + PAD - j) / 2 - FIRST)
            if constexpr (SAT) {
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        float v = 0.f;
#pragma unroll
                        for (int i = (p + PAD) % 2; i < KS; i += 2)
#pragma unroll
                            for (int j = (t + PAD) % 2; j < KS; j += 2) v += gr[cur][(p + PAD - i) / 2 - FIRST][(t + PAD - j) / 2 - FIRST];
                        gs[p][t] += v;
                    }
            }
#pragma unroll
            for (int hh = 0; hh < NU; ++hh) {
                const int wb = (NU == 1 ? cur : hh) & 1;
#pragma unroll
                for (int idx = 0; idx < UM * KK; ++idx) {
                    const int j = idx % KS, i = idx / KS % KS, u = idx / KK, p = (i + PAD) % 2, t = (j + PAD) % 2, q = 2 * (hh * UM + u) + p;
                    const float wgt = wv[wb][u][i * KS + j];
                    const float dd = SAT ? sat01(fmaf(wgt, 0.5f, cr[q][t])) : hardtanh(wgt - cr[q][t]);
                    acc[q][t] = fmaf(dd, gr[cur][(p + PAD - i) / 2 - FIRST][(t + PAD - j) / 2 - FIRST], acc[q][t]);
                    if (idx == 0) {
                        __builtin_amdgcn_sched_barrier(0);
                        load_w(wb ^ 1, hh + 1 < NU ? hh + 1 : 0, hh + 1 < NU ? co : cn);
                        if (hh == 0) load_g((cur + C::AHEAD) % NB, cl);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            co = next;
            {
                const int c = after(cl);
                cl = c < d.Co ? c : cl;
            }
            if (chunk_end || !more) {   // first levels of at most 32 (5x5: 72) terms
#pragma unroll
                for (int q = 0; q < ROWS; ++q)
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        float *p = tot + (q * 2 + t) * 64;
                        *p = first ? acc[q][t] : *p + acc[q][t];
                        acc[q][t] = 0.f;
                    }
                if constexpr (SAT) {
#pragma unroll
                    for (int e = 0; e < 2 * 2; ++e) {
                        double *p = gtot + e * 64;
                        float &g = gs[e / 2][e % 2];
                        *p = first ? (double)g : *p + (double)g;
                        g = 0.f;
                    }
                }
                first = false;
            }
            return more;
        };
#pragma unroll 1
        while (channel(0) && channel(1) && (NB == 2 || (channel(2) && channel(NB - 1)))) {}
        static_assert(NB == 2 || NB == 4, "the buffers take turns");
    }
    if (first) {   // no channels for this wave
#pragma unroll
        for (int e = 0; e < ROWS * 2; ++e) tot[e * 64] = 0.f;
        if constexpr (SAT) {
#pragma unroll
            for (int e = 0; e < 4; ++e) gtot[e * 64] = 0.0;
        }
    }
    __syncthreads();
    if (wave * FM >= ROWS) return;
    const int q0 = wave * FM;
    float r[FM][2], add[FM][2];
    int at[FM];      // the lane's first position of row f, from the start of the image
    bool own[FM];
#pragma unroll
    for (int f = 0; f < FM; ++f) {
        const int q = q0 + f, ci = ci_base + q / 2, h = 2 * a + q % 2;
        own[f] = sidx == sc && ci >= ci_first && h < d.H;
        at[f] = own[f] ? (ci * d.H + h) * d.W + 2 * b0 : 0;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            float v = smem[(q * 2 + t) * 64 + lane];
#pragma unroll
            for (int k = 1; k < KSP; ++k) v += smem[((k * ROWS + q) * 2 + t) * 64 + lane];
            if constexpr (SAT) {   // sum over (co, taps) of the gy values the position met
                const double *p = reinterpret_cast<const double *>(smem + C::PART) + (q % 2 * 2 + t) * 64 + lane;
                double g = p[0];
#pragma unroll
                for (int k = 1; k < KSP; ++k) g += p[k * (2 * 2 * 64)];
                v = fmaf(2.f, v, -(float)g);
            }
            r[f][t] = v;
        }
    }
    const size_t image = (size_t)n * d.Ci * plane;
    if (gadd) {   // (all loads before the first store: one counter serves both)
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int t = 0; t < 2; ++t) add[f][t] = own[f] && 2 * b0 + t < d.W ? ldf(gadd + image + at[f] + t) : 0.f;
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int t = 0; t < 2; ++t) r[f][t] += add[f][t];
    }
    #pragma unroll
    for (int f = 0; f < FM; ++f) {
        if (!own[f]) continue;
        T *dst = gx + image + at[f];
        if (2 * b0 + 1 < d.W) st_strip<2>(dst, r[f]);
        else stf(dst, r[f][0]);
    }
}

static int gx_s2_tiles(const ConvDims &d) { return (int)ceil_div_l((long)d.N * d.Ho * d.Wo, 64); }

// Input channels per lane: four where the launch fills the chip and they waste few, else two (us, four / two: 256 -> 256 @28x28, 32 images, 233 / 304,
// one image, 2048 waves of four, 19.5 / 20.5, 107 -> 278 @23x23, 5 images, 2592 waves, 31 / 28, 128 -> 128 @56x56, one image, 3328 waves, 16.5 / 19.2;
// 5x5: 36 -> 34 @38x41, 6 images, 2736 waves, 13.9 / 12.4; six channels, 6 -> 897 @41x49, 27 images, 173 / 137).
// Waves that share the output channels: one chunk each, as many as eight.  Up to 64 channels at most four, and none for less than half a chunk, where
// that still makes 2800 waves (us, 3x3 / 5x5: 64 -> 33 @29x29, 64 images, eight waves 38 / 83, four 30 / 64; -> 64 52 / 116, 46 / 105; 60 -> 33 @21x21, 32 images, 12.9 /
// 24.6, 11.2 / 21.0; 47 -> 17 @58x58, 62 images, bfloat16, four waves 55 / 108, two 43 / 86, -> 9 two 34 / 63, one 27 / 51; but 40 -> 19 @29x29, eight images, 580
// workgroups, four 5.7 / 7.8, two 6.1 / 8.4, and 60 -> 130 @21x21, 32 images, eight 27 / 65, four 29 / 67).
static GradXShape gx_s2_shape(const ConvDims &d) {
    const int most = d.Co <= 8 ? 1 : d.Co <= 16 ? 2 : d.Co <= 32 ? 4 : 8, full = full_chunks(d.Co, kNineChunk), few = full <= 2 ? full : 4;
    auto shape = [&](int waves) {
        const bool wide = d.Ci >= 4 && (long)gx_s2_tiles(d) * ceil_div(d.Ci, 4) * waves >= 3000 && 5 * ceil_div(d.Ci, 4) <= 3 * ceil_div(d.Ci, 2);
        return GradXShape{wide ? 4 : 2, 1, waves, false};
    };
    const GradXShape shared = shape(few);
    return d.Co <= 64 && (long)gx_s2_tiles(d) * ceil_div(d.Ci, shared.tm) * few >= 2800 ? shared : shape(most);
}

// Layers it takes: from two input channels on; the distance of a wave's strips from the first one's image has to fit 32 bits, and the grid 2^32 threads.
bool grad_x_s2_supported(const ConvDims &d) {
    if (d.Ci < 2 || d.kh != d.kw || (d.kh != 3 && d.kh != 5) || d.pad != d.kh / 2 || d.stride != 2) return false;
    if ((images_ahead(d, (long)d.Ho * d.Wo) * d.Co + 1) * d.Ho * d.Wo > 0x3fffffffL || (long)d.Ci * d.H * d.W > 0x7fffffffL) return false;
    return (long)gx_s2_tiles(d) * ceil_div(d.Ci, 2) <= 0x7fffffL;
}

template <class C, bool SAT, class T>
static int launch_gx_s2(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s, const T *gadd) {
    const GxS2Dims t{d.N, d.Ci, d.H, d.W, d.Co, d.Ho, d.Wo, gx_s2_tiles(d), ceil_div(d.Ci, C::TM)};
    constexpr int LDS_BYTES = C::PART * 4 + (SAT ? C::SAT_BYTES : 0);
    if (int rc = allow_dynamic_lds<&grad_x_s2_kernel<C, SAT, T>>(LDS_BYTES)) return rc;
    hipLaunchKernelGGL((grad_x_s2_kernel<C, SAT, T>), dim3((unsigned)t.tiles * t.blocks), dim3(C::NT), LDS_BYTES, s, gy, x, w, gx, t, gadd);
    return check_launch();
}

GradXShape grad_x_s2_shape(const ConvDims &d, bool sat) {
    GradXShape shape = gx_s2_shape(d);
    shape.two = shape.tm == 4 && sat && d.kh == 3;
    return shape;
}

// sat: the two-instruction form (grad_x.hip), where the launch fills the chip
template <class T>
int launch_grad_x_s2(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s, const T *gadd, bool sat) {
    const GradXShape shape = grad_x_s2_shape(d, sat);
    auto run = [&](auto ks, auto ksp) {
        constexpr int KS = decltype(ks)::value, KSP = decltype(ksp)::value;
        if (shape.tm == 2) return launch_gx_s2<GxS2Cfg<KS, 2, KSP>, false, T>(gy, x, w, gx, d, s, gadd);
        if constexpr (KS == 3) {
            if (shape.two) return launch_gx_s2<GxS2Cfg<KS, 4, KSP>, true, T>(gy, x, w, gx, d, s, gadd);
        }
        return launch_gx_s2<GxS2Cfg<KS, 4, KSP>, false, T>(gy, x, w, gx, d, s, gadd);
    };
    auto waves = [&](auto ks) {
        switch (shape.waves) {
            case 1: return run(ks, std::integral_constant<int, 1>{});
            case 2: return run(ks, std::integral_constant<int, 2>{});
            case 4: return run(ks, std::integral_constant<int, 4>{});
            default: return run(ks, std::integral_constant<int, 8>{});
        }
    };
    return d.kh == 3 ? waves(std::integral_constant<int, 3>{}) : waves(std::integral_constant<int, 5>{});
}
template int launch_grad_x_s2<float>(const float *, const float *, const float *, float *, const ConvDims &, hipStream_t, const float *, bool);
template int launch_grad_x_s2<bf16_t>(const bf16_t *, const bf16_t *, const float *, bf16_t *, const ConvDims &, hipStream_t, const bf16_t *, bool);

}  // namespace adder

// Input gradient of 3x3 / pad 1 and 5x5 / pad 2 layers of stride 1, NCHW:
//   gx[n,ci,h,w] = sum_{co,i,j} hardtanh(w[co,ci,i,j] - x[n,ci,h,w]) * gy[n,co,h+p-i,w+p-j]
// Replaces the grad_i half of adder_cuda/adder.cu:194-272, adder.cu:133-192 and the fold of adder.py:32-33.
//
// The terms are those of grad_x.hip (two vector instructions, three above kSatMaxTerms terms) and bound it.  As in fwd_nine.hip a lane
// reads the window of gy of its strip straight into registers, strips of all images line up and the waves of a workgroup share
// the output channels; sums of sums live in LDS (once per 72 terms), 10 KB a wave, so that four waves per SIMD stay.  Large maps that
// fill tiles of 16 x 16 or 8 x 32 positions are left to the tiles of grad_x.hip (see grad_x_tiles), which ask for gy once instead of nine
// times: 128 -> 128 @32x32, 128 images, 698 us there, 734 here, 256 -> 256 @16x16 902 against 921.
// us, tiles or the kernel for few positions there was -> this: 32 images 64 -> 64 @56x56 168 -> 161, 128 -> 128 @28x28 193 -> 167, 256 -> 256 @14x14 244 -> 228,
// 512 -> 512 @7x7 321 -> 281, 100 -> 100 @20x20 118 -> 64; 64 -> 64 @8x8, 256 images 29.8 -> 30.3, one image 29 -> 6.3; 128 -> 128 @28x28, 4 / 1 images 97 -> 34,
// 94 -> 16; 12 -> 48 @4x4, 64 images 8.5 -> 5.6; 256 -> 256 @14x14, one image 19.9 -> 17.6.  8 x 4 results in two instructions a term are 128 registers and five to
// seven spilled ones (24 to 32 bytes of scratch per lane).
//
// 25 taps: 4 channels x 2 positions per lane, three reads per row of the window a channel ahead; small launches 4 x 1.  Rows of an odd length and 4 x 1 take three
// instructions a term (error against float64 1.3e-7 to 1.5e-7 of the result; two instructions 2.0e-7 to 2.1e-7, tiles 2.1e-7 to 3.7e-7).  us, tiles in LDS ->
// this: 342 channels of gy -> 48 of gx @10x10, 8 images, 277 -> 56, 261 -> 10 @27x27, 5 images, bfloat16, 204 -> 42, 813 -> 551 @9x9, two images, 727 -> 252, 64 -> 64 @8x8,
// 64 images, 46 -> 27, one image 44 -> 11, 19 -> 47 @14x14, 193 images, 64 -> 51, 100 -> 100 @28x28, 32 images, bfloat16, 349 -> 285; odd rows, where tiles ran two instructions:
// 32 images, 64 -> 32 @17x17 71 -> 40, @21x21 71 -> 51, @25x25 72 -> 73, @29x29 72 -> 86, @53x53 242 -> 273; what fills tiles stays there (fills_5x5_tiles).
// Tried on the way: 4 x 4 per lane 64 -> 64 @56x56, 16 images, 471 (66 registers spilled), 4 x 2 in three instructions 295, with five waves per SIMD 327.
#include "wave_split.hpp"

#include <type_traits>

namespace adder {

// Output channels per first-level sum: 72 terms (25 taps: 50)
static constexpr int gx_nine_chunk(int ks) { return ks == 3 ? kNineChunk : 2; }

// TM input channels x TN adjacent positions per lane; KSP waves that share the output channels in chunks of CC
// KS: taps per side, 3 or 5
template <int TM_, int TN_, int KSP_, int KS_ = 3>
struct GxNineCfg {
    static constexpr int KS = KS_, KK = KS * KS, PAD = KS / 2;
    static constexpr int TM = TM_, TN = TN_, KSP = KSP_, NT = 64 * KSP, CC = gx_nine_chunk(KS), FM = kFinished<TM, KSP>, STRIP = TN + 2 * PAD;
    static constexpr int AHEAD = TN == 1 && KS == 3 ? 3 : 1;           // output channels that gy is asked for ahead of the arithmetic
    static constexpr int UM = TN == 4 || KS == 5 ? 1 : 2, NU = TM / UM;   // input channels whose weights are asked for together, a step ahead
    static constexpr int PART = KSP * TM * TN * 64, LDS_BYTES = PART * 4 + KSP * TN * 64 * 8;
    static_assert((TM % KSP == 0 || KSP % TM == 0) && (NU == 1 || NU % 2 == 0), "a wave finishes FM channels or none; two weight buffers");
    // 25 taps, two positions: the two columns on a side are both inside the map or both outside (rows of an odd length: see Strips), and one read
    static constexpr bool PAIRS = KS == 5 && TN == 2;
    static_assert(KS == 3 || (KS == 5 && TN <= 2), "nine taps, or 25 of one or two positions");
};

struct GxNineDims {
    int N, Ci, H, W, Co;
    Strips row;
    int strips;             // of TN positions per image
    int tiles, blocks;      // of 64 strips, of TM input channels
};

// SAT, FUSE, gadd, bn: as in grad_x_3x3s1_kernel (one slot of sums per tile).
template <class C, bool SAT, class T, bool FUSE>
__global__ __launch_bounds__(C::NT, 4) void grad_x_nine_kernel(const T *__restrict__ gy, const T *__restrict__ x, const float *__restrict__ w,
                                                               T *__restrict__ gx, const GxNineDims d, const T *__restrict__ gadd,
                                                               const adder_bn_links bn) {
    constexpr int TM = C::TM, TN = C::TN, KSP = C::KSP, FM = C::FM, STRIP = C::STRIP, NB = C::AHEAD + 1, UM = C::UM, NU = C::NU;
    constexpr int KS = C::KS, KK = C::KK, PAD = C::PAD;
    extern __shared__ __align__(16) float smem[];
    int tile, blk;
    xcd_tile(blockIdx.x, d.tiles, d.blocks, tile, blk);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int sidx = tile * 64 + lane, sc = min(sidx, d.N * d.strips - 1), n = sc / d.strips, rest = sc - n * d.strips;
    const int h = rest / d.row.per_row, s = rest - h * d.row.per_row, w0 = d.row.start(s, TN, d.W), ci_base = blk * TM;
    const int plane = d.H * d.W, K = d.Ci * KK;
    uniform_f32_ptr wc = as_uniform(w);
    int wofs[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) wofs[m] = min(ci_base + m, d.Ci - 1) * KK;

    float cr[TM][TN], acc[TM][TN];
#pragma unroll
    for (int m = 0; m < TM; ++m) {
        float xv[TN];
        ld_strip<TN>(x + ((size_t)n * d.Ci + min(ci_base + m, d.Ci - 1)) * plane + h * d.W + w0, xv);
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            cr[m][t] = SAT ? fmaf(-0.5f, xv[t], 0.5f) : xv[t];
            acc[m][t] = 0.f;
        }
    }
    // sums of sums in LDS: this wave's part, [channel][position][lane]; and of the gy values the positions met, [position][lane]
    float *tot = smem + wave * (TM * TN * 64) + lane;
    double *gtot = reinterpret_cast<double *>(smem + C::PART) + wave * (TN * 64) + lane;
    bool first = true;

    // a uniform base per channel and the lane's distances from it in bytes, as in fwd_nine.hip
    const int n_first = __builtin_amdgcn_readfirstlane(n);
    const T *g_first = gy + (size_t)n_first * d.Co * plane;
    constexpr int NSIDE = KS == 3 ? 3 : 1;
    const bool ok_l = w0 > 0, ok_r = w0 + TN < d.W;
    bool ok[KS];
    unsigned off[KS], off_l[NSIDE], off_r[NSIDE];
    unsigned in_row[KS], in_col[2 * PAD];   // 25 taps: bit masks and one distance per row, as in fwd_nine.hip
    int beside[2 * PAD];
#pragma unroll
    for (int k = 0; k < 2 * PAD; ++k) {
        const int c = k < PAD ? k - PAD : TN + k - PAD;   // from the strip's first column
        const bool in = w0 + c >= 0 && w0 + c < d.W;
        in_col[k] = in ? ~0u : 0u;
        beside[k] = (in ? c : 0) * (int)sizeof(T);
    }
#pragma unroll
    for (int i = 0; i < KS; ++i) {
        const int r = h + i - PAD;
        ok[i] = r >= 0 && r < d.H;
        in_row[i] = ok[i] ? ~0u : 0u;
        const int o = (n - n_first) * d.Co * plane + min(max(r, 0), d.H - 1) * d.W + w0;
        off[i] = (unsigned)o * (unsigned)sizeof(T);
        if constexpr (KS == 3) {
            off_l[i] = (unsigned)(ok_l ? o - 1 : o) * (unsigned)sizeof(T);
            off_r[i] = (unsigned)(ok_r ? o + TN : o) * (unsigned)sizeof(T);
        }
    }
    float gr[NB][KS][STRIP], wv[2][UM][KK], gs[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t) gs[t] = 0.f;
    auto load_g = [&](const int b, const int co) {
        const char *p = reinterpret_cast<const char *>(g_first + (size_t)co * plane);
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            keep_offset(off[i]);
            float u[TN];
            ld_strip<TN>(reinterpret_cast<const T *>(p + off[i]), u);
#pragma unroll
            for (int t = 0; t < TN; ++t) gr[b][i][t + PAD] = u[t];
            if constexpr (KS == 3) {
                keep_offset(off_l[i]); keep_offset(off_r[i]);
                gr[b][i][0] = ldf(reinterpret_cast<const T *>(p + off_l[i]));
                gr[b][i][TN + 1] = ldf(reinterpret_cast<const T *>(p + off_r[i]));
            } else {
#pragma unroll
                for (int k = 0; k < 4; k += 2) {
                    float q[2];
                    if constexpr (C::PAIRS) {
                        ld_strip<2>(reinterpret_cast<const T *>(p + (off[i] + (unsigned)beside[k])), q);
                    } else {
                        q[0] = ldf(reinterpret_cast<const T *>(p + (off[i] + (unsigned)beside[k])));
                        q[1] = ldf(reinterpret_cast<const T *>(p + (off[i] + (unsigned)beside[k + 1])));
                    }
                    gr[b][i][k < PAD ? k : TN + k] = q[0];
                    gr[b][i][(k < PAD ? k : TN + k) + 1] = q[1];
                }
            }
        }
    };
    auto load_w = [&](const int b, const int hh, const int co) {
#pragma unroll
        for (int u = 0; u < UM; ++u)
#pragma unroll
            for (int e = 0; e < KK; ++e) wv[b][u][e] = wc[co * K + wofs[hh * UM + u] + e];
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
            for (int i = 0; i < KS; ++i) {   // positions outside gy contribute nothing
                if constexpr (KS == 3) {
                    if (i != PAD) {
#pragma unroll
                        for (int k = 1; k <= TN; ++k) gr[cur][i][k] = ok[i] ? gr[cur][i][k] : 0.f;
                    }
                    gr[cur][i][0] = ok[i] && ok_l ? gr[cur][i][0] : 0.f;
                    gr[cur][i][TN + 1] = ok[i] && ok_r ? gr[cur][i][TN + 1] : 0.f;
                } else {
                    auto keep = [&](float &v, const unsigned m) { v = __uint_as_float(__float_as_uint(v) & m); };
                    keep_offset(in_row[i]);
                    if (i != PAD) {
#pragma unroll
                        for (int k = PAD; k < PAD + TN; ++k) keep(gr[cur][i][k], in_row[i]);
                    }
#pragma unroll
                    for (int k = 0; k < 2 * PAD; ++k) {
                        const int e = C::PAIRS ? k & ~1 : k;
                        keep_offset(in_col[e]);
                        keep(gr[cur][i][k < PAD ? k : TN + k], in_row[i] & in_col[e]);
                    }
                }
            }
            if constexpr (SAT) {
                float c[STRIP];   // sums over the window's rows
#pragma unroll
                for (int k = 0; k < STRIP; ++k) {
                    c[k] = (gr[cur][0][k] + gr[cur][1][k]) + gr[cur][2][k];
                    if constexpr (KS == 5) c[k] += gr[cur][KS - 2][k] + gr[cur][KS - 1][k];
                }
#pragma unroll
                for (int t = 0; t < TN; ++t) {
                    float v = (c[t] + c[t + 1]) + c[t + 2];
                    if constexpr (KS == 5) v += c[t + KS - 2] + c[t + KS - 1];
                    gs[t] += v;
                }
            }
#pragma unroll
            for (int hh = 0; hh < NU; ++hh) {
                const int wb = (NU == 1 ? cur : hh) & 1;
#pragma unroll
                for (int idx = 0; idx < UM * KK * TN; ++idx) {
                    const int t = idx % TN, j = idx / TN % KS, i = idx / TN / KS % KS, u = idx / TN / KK, m = hh * UM + u;
                    const float wgt = wv[wb][u][i * KS + j];
                    const float dd = SAT ? sat01(fmaf(wgt, 0.5f, cr[m][t])) : hardtanh(wgt - cr[m][t]);
                    acc[m][t] = fmaf(dd, gr[cur][2 * PAD - i][t + 2 * PAD - j], acc[m][t]);
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
            if (chunk_end || !more) {   // first levels of 72 terms (25 taps: 50)
#pragma unroll
                for (int m = 0; m < TM; ++m)
#pragma unroll
                    for (int t = 0; t < TN; ++t) {
                        float *p = tot + (m * TN + t) * 64;
                        *p = first ? acc[m][t] : *p + acc[m][t];
                        acc[m][t] = 0.f;
                    }
                if constexpr (SAT) {
#pragma unroll
                    for (int t = 0; t < TN; ++t) {
                        double *p = gtot + t * 64;
                        *p = first ? (double)gs[t] : *p + (double)gs[t];
                        gs[t] = 0.f;
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
        for (int e = 0; e < TM * TN; ++e) tot[e * 64] = 0.f;
#pragma unroll
        for (int t = 0; t < TN; ++t) gtot[t * 64] = 0.0;
    }
    __syncthreads();
    if (wave * FM >= TM) return;
    const int m0 = wave * FM, ci0 = ci_base + m0;
    float r[FM][TN], sg[TN];
    if constexpr (SAT) {   // sum over (co, taps) of the gy values a position met
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            const double *p = reinterpret_cast<const double *>(smem + C::PART) + t * 64 + lane;
            double v = p[0];
#pragma unroll
            for (int k = 1; k < KSP; ++k) v += p[k * (TN * 64)];
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
    if (ci0 >= d.Ci) return;
    unsigned own = 0;   // bit t: position w0 + t is this lane's
#pragma unroll
    for (int t = 0; t < TN; ++t) own |= (sidx == sc && w0 + t >= d.row.first(s, TN) ? 1u : 0u) << t;
    finish_grad_x<FM, TN, FUSE>(r, own, ci0, ci0, d.Ci, plane, (n * d.Ci + ci0) * plane + h * d.W + w0, TN > 1 && d.W % TN == 0, x, gx, gadd, bn,
                                d.tiles, tile, lane);
}

static int gx_nine_tiles(const ConvDims &d, int tn) { return (int)ceil_div_l((long)d.N * d.H * ceil_div(d.W, tn), 64); }

// Positions per lane (input channels: 8 x 4, 8 x 2 or 4 x 1, 25 taps 4), waves that share the output channels, and whether a term takes two instructions.
//
// Two instructions, 8 x 4 only and only where the launch fills the chip: below that they gain nothing (32 -> 32 @16x16, 32 images, 9.1 us, three 8.8; 64 -> 64
// @56x56, one, 11.9, 13.2) and round w and x once more (2.3e-7 of the result against 1.6e-7).  The line to the smaller shapes is that of fwd_nine.hip, with a
// wave's chain of 1.7, 1.15 and 0.55 us a channel and 24, 22 and 12 terms per ps (4 x 1: 7 on rows that are shorter than 8).  us, 8 x 4 / 8 x 2 / 4 x 1: 128 -> 128
// @28x28, 4 images, 29 / 31 / 36, one 29 / 20 / 14; 64 -> 64 @56x56, one, 17 / 12 / 14.
//
// Three instructions: a workgroup of 8 x 4 is long and few fill the chip, and two of them on a CU wait for each other's weights, so that the smaller shapes are
// ahead until some ten of 8 x 4 lie on each CU.  By what the busiest CU takes for a wave's channels, us per channel and workgroup of eight waves there.
// us, 8 x 4 / 8 x 2 / 4 x 1 with eight waves: 921 -> 174 (channels of gy -> of gx) @42x42, one image, 321 / 278 / 219, 713 -> 149 @42x50, one, 258 / 214 / 172, 517 -> 535
// @15x18, three, 294 / 172 / 177, 242 -> 15 @53x53, 13, 139 / 114 / 100, 144 -> 144 @28x28, eight, 82 / 88 / 89, 32, 245 / 266 / 309, 200 -> 200 @14x14, 128, 498 / 490 / 560,
// 512 -> 512 @8x8, 128, 978 / 1058 / 1293, 512 -> 512 @7x7, one, 128 / 83 / 32.
GradXShape grad_x_nine_shape(const ConvDims &d, bool bf16, bool groups) {
    const int waves = d.Co <= 8 ? 1 : d.Co <= 16 ? 2 : d.Co <= 32 ? 4 : 8;
    if (d.kh == 5) {
        // us, 4 x 2 / 4 x 1: W even, two instructions a term, 64 -> 64 @8x8, 64 images, 4096 waves of 4 x 2, 32 / 37, 48 -> 342 @10x10, 8 images, 672, 70 / 56, 64 -> 64
        // @32x32, one, 1024, 17.5 / 13.4; W odd, three, by the busiest CU's workgroups, where one of 4 x 2 takes 1.63 times as long as one of 4 x 1: 64 -> 32 @29x29, 32
        // images, 97 / 119, 16 -> 16 @17x17, 64 images, 1224 waves, 16.0 / 16.9, 32 -> 64 @21x21, 4 images, 960, 15.6 / 14.4, 821 -> 665 @9x9, two, 334 and 501 workgroups,
        // 316 / 256.  (Rows of three and five columns have no strips without a cut pair.)
        const long wide = (long)gx_nine_tiles(d, 2) * ceil_div(d.Ci, 4), narrow = (long)gx_nine_tiles(d, 1) * ceil_div(d.Ci, 4);
        const bool odd = d.W % 2 != 0, pairs = !odd || d.W >= 7;
        const int tn = pairs && wide * waves >= (odd ? 1200 : 2048) && (!odd || 163 * ceil_div_l(wide, 256) <= 100 * ceil_div_l(narrow, 256)) ? 2 : 1;
        return {4, tn, waves, tn == 2 && d.W % 2 == 0 && groups && d.Ci >= 2 && two_instructions_5x5(d.Co)};
    }
    auto wgs = [&](int n) { return (long)gx_nine_tiles(d, n) * ceil_div(d.Ci, n == 1 ? 4 : 8); };
    const int most = d.W >= 4 ? 4 : d.W >= 2 ? 2 : 1;
    const float terms = (float)d.K() * d.Co * d.N * d.H * d.W;
    const int chunks = ceil_div(ceil_div(d.Co, kNineChunk), waves), chain = min(chunks * kNineChunk, d.Co);
    if (most == 4 && groups && d.Co * 9 <= kSatMaxTerms && d.Ci >= 4 && !small_unlinked(d, bf16) && wgs(4) * waves >= 1300) {
        const float wide = fmaxf(1.7f * chain, terms / 24e6f), narrow = fmaxf(0.55f * chain, terms / (d.W < 8 ? 7e6f : 12e6f));
        // (waves that would have less than half a chunk are left out: 17 channels @28x28, 32 images, four waves 34.6 us, two 30.1, 33 channels, eight 53.6, four 48.5)
        const int full = full_chunks(d.Co, kNineChunk);
        if (narrow >= wide) return {8, 4, full <= 2 ? full : full <= 4 ? 4 : 8, true};
    }
    int tn = 1;
    float least = 0.f;
    for (int n = 1; n <= most; n *= 2) {
        const float load = (float)ceil_div_l(wgs(n), 256) * waves / 8, share = (float)d.Co / waves;
        const float per = n == 1 ? fmaxf(0.55f, (d.W < 8 ? 0.48f : 0.37f) * load) : n == 2 ? fmaxf(1.2f + 0.2f * load, 0.3f + 1.1f * load)
                                                                                         : fmaxf(2.f + 0.8f * load, 2.f * load);
        const float cost = per * (load <= 2.f ? 0.5f * (chain + share) : share);
        if (n == 1 || cost < least) { tn = n; least = cost; }
    }
    return {tn == 1 ? 4 : 8, tn, waves, false};
}

// Layers it takes; the distance of a wave's strips from the first one's image has to fit 32 bits, and so have the launch's threads.
bool grad_x_nine_supported(const ConvDims &d) {
    if (d.kh != d.kw || (d.kh != 3 && d.kh != 5) || d.pad != d.kh / 2 || d.stride != 1) return false;
    if ((images_ahead(d, (long)d.H * ceil_div(d.W, 4)) * d.Co + 1) * d.H * d.W > 0x3fffffffL) return false;
    const GradXShape shape = grad_x_nine_shape(d, false, true);
    return (long)gx_nine_tiles(d, shape.tn) * ceil_div(d.Ci, shape.tm) * 64 * shape.waves <= kMaxThreads;
}
int grad_x_nine_bn_slots(const ConvDims &d) { return gx_nine_tiles(d, grad_x_nine_shape(d, false, true).tn); }

template <class C, bool SAT, class T, bool FUSE>
static int launch_gx_nine(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s, const T *gadd,
                          const adder_bn_links &bn) {
    const int per_row = ceil_div(d.W, C::TN);
    const GxNineDims t{d.N, d.Ci, d.H, d.W, d.Co, Strips{per_row, C::PAIRS && d.W % 2 ? 2 : kNoShift}, per_row * d.H, gx_nine_tiles(d, C::TN), ceil_div(d.Ci, C::TM)};
    if (FUSE && (!bn.in_part || bn.in_slots != t.tiles)) return ADDER_ERR_BAD_SHAPE;
    if (int rc = allow_dynamic_lds<&grad_x_nine_kernel<C, SAT, T, FUSE>>(C::LDS_BYTES)) return rc;
    hipLaunchKernelGGL((grad_x_nine_kernel<C, SAT, T, FUSE>), dim3((unsigned)t.tiles * t.blocks), dim3(C::NT), C::LDS_BYTES, s, gy, x, w, gx, t,
                       gadd, bn);
    return check_launch();
}

// bn (nullable): the in_* half of adder_bn_links
template <class T>
int launch_grad_x_nine(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s, const T *gadd,
                       const adder_bn_links *bn, bool groups) {
    const GradXShape shape = grad_x_nine_shape(d, sizeof(T) == 2, groups);
    auto run = [&](auto cfg) {
        using C = decltype(cfg);
        auto form = [&](auto sat) {
            constexpr bool SAT = decltype(sat)::value;
            if constexpr (sizeof(T) == 4 && C::KS == 3) {
                if (bn) return launch_gx_nine<C, SAT, T, true>(gy, x, w, gx, d, s, gadd, *bn);
            }
            return launch_gx_nine<C, SAT, T, false>(gy, x, w, gx, d, s, gadd, adder_bn_links{});
        };
        if constexpr (C::TN == 4 || C::PAIRS) {
            if (shape.two) return form(std::true_type{});
        }
        return form(std::false_type{});
    };
    auto waves = [&](auto ksp) {
        constexpr int KSP = decltype(ksp)::value;
        if (d.kh == 5) return shape.tn == 2 ? run(GxNineCfg<4, 2, KSP, 5>{}) : run(GxNineCfg<4, 1, KSP, 5>{});
        return shape.tn == 4 ? run(GxNineCfg<8, 4, KSP>{}) : shape.tn == 2 ? run(GxNineCfg<8, 2, KSP>{}) : run(GxNineCfg<4, 1, KSP>{});
    };
    switch (shape.waves) {
        case 1: return waves(std::integral_constant<int, 1>{});
        case 2: return waves(std::integral_constant<int, 2>{});
        case 4: return waves(std::integral_constant<int, 4>{});
        default: return waves(std::integral_constant<int, 8>{});
    }
}
template int launch_grad_x_nine<float>(const float *, const float *, const float *, float *, const ConvDims &, hipStream_t,
                                       const float *, const adder_bn_links *, bool);
template int launch_grad_x_nine<bf16_t>(const bf16_t *, const bf16_t *, const float *, bf16_t *, const ConvDims &, hipStream_t,
                                        const bf16_t *, const adder_bn_links *, bool);

}  // namespace adder

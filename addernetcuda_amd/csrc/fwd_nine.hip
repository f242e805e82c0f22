// Forward of 3x3 / pad 1 and 5x5 / pad 2 layers, stride 1 or 2, NCHW in -> NCHW out:
//   y[n,co,ho,wo] = - sum_{ci,i,j} | w[co,ci,i,j] - xpad[n,ci,ho*s+i-p,wo*s+j-p] |
// Replaces adder_cuda/adder.cu:19-70 (CONV) together with the unfold + permute copies of adder.py:32-33,38-39 that feed it.
//
// Two vector instructions per term bound it: v_sub_f32 d, s_w, v_x ; v_sub_f32 acc, acc, |d| -- 73 T lane-instructions/s is what a bare
// stream of the pair reaches with two waves on each of a SIMD's two issue ports (62 T with one each).  Weights are wave-uniform and come
// through the scalar cache as scalar operands.  A lane reads the window of its strip straight into registers, one channel ahead: nine
// reads of at most 16 bytes serve 576 instructions, 4.6 KB in the 288 cycles that a CU takes for them or a quarter of the 64 bytes a cycle
// that L1 delivers, so a tile in LDS, its barriers and its halo columns had nothing to give.  Without a tile the strips of all images line up (14 columns are 4 strips, 56 are 14: 88 and 100 % of
// the lanes have work where 16 x 16 and 8 x 32 tiles left 77 and 88 %), and the waves of a workgroup can share the input channels
// instead of the positions, which is what small maps with many channels need.  Each chunk's sums meet in LDS in channel order (ChunkSums):
// any other order changes the last bits of a layer, which a deep network amplifies (ResNet-50's logits by up to 0.07 of their root
// mean square), and costs the launches below 3 to 10 % against sums that meet once at the end, small ones of 16-channel chunks up to 30 %.
// us, tiles in LDS -> this: 32 images 64 -> 64 @56x56 184 -> 158, 128 -> 128 @28x28 200 -> 169, 256 -> 256 @14x14 208 -> 191, 512 -> 512 @7x7
// 290 -> 191, 100 -> 100 @20x20 119 -> 66; 128 images 128 -> 128 @32x32 659 -> 627, 512 -> 512 @8x8 716 -> 689; 256 images 16 -> 16 @32x32 30.5 -> 31.2,
// 64 -> 64 @8x8 31.8 -> 29.5; stride 2, 32 images 128 -> 128 @56x56 225 -> 158, 512 -> 512 @14x14 376 -> 233; one image (the kernel for few
// positions there was) 64 -> 64 @8x8 7.6 -> 6.6, 256 -> 256 @14x14 19.9 -> 17.0, 512 -> 512 @7x7 30 -> 29.
// Tried on the way: 4 channels x 4 positions per lane 132 -> 179 us (64 -> 64 @56x56: reads), 8 x 2 143.
//
// 25 taps: 4 channels x 4 positions (stride 2: x 2) per lane, three or four reads per row of the window a channel ahead, 92 to 128
// registers.  (No instance of this file spills vector registers; with the inference epilogue up to 43 scalar ones live in vector lanes.)  us, tiles in LDS -> this: 64 -> 64 @56x56, 16 images, 271 -> 202, 128 -> 64 @16x16, 64 images, 137 -> 132, 32 -> 64 @16x16 40.9 -> 39.8,
// 64 -> 64 @8x8 65 -> 22, one image 61 -> 9.7, 47 -> 19 @14x14, 193 images, 111 -> 71, 9 -> 20 @53x53, 32 images, 51 -> 31, 813 -> 551 @9x9, two images, 865 -> 258,
// 32 -> 64, 32 images, @13x13 37 -> 22, @21x21 77 -> 44, @29x29 81 -> 75 (4 x 1 on such rows of whole strips and one column: 98);
// stride 2: 64 -> 64 @56x56, 32 images, 176 -> 145, 7 -> 144 @23x26, 202 images, 86 -> 60, 36 -> 34 @38x41, 6 images, 30 -> 12, 32 -> 64 @32x32, 64 images, 52 -> 55.
// On the way, 64 -> 64 @56x56: comparisons instead of bit masks for what lies outside 387 (the masks of 20 elements fill the scalar
// registers), the columns beside a strip read one by one 315, three waves per SIMD instead of four with a few spilled registers 218.
#include "wave_split.hpp"

#include <type_traits>

namespace adder {

// S: stride; TM output channels x TN adjacent positions per lane; SHARED: two to eight waves share the input channels
// EVEN (stride 2): rows of an even length, whose strips' columns and the one behind them are one read
// KS: taps per side, 3 or 5
template <int S_, int TM_, int TN_, bool SHARED_, bool EVEN_ = false, int KS_ = 3>
struct NineCfg {
    static constexpr int S = S_, TM = TM_, TN = TN_, NT = SHARED_ ? 512 : 64;
    static constexpr bool SHARED = SHARED_;
    using Sums = ChunkSums<TM, TN, SHARED>;
    static constexpr int KS = KS_, KK = KS * KS, PAD = KS / 2;
    static constexpr bool EVEN = EVEN_;
    static constexpr int AHEAD = TN == 1 && KS == 3 ? 3 : 1;   // input channels that x is asked for ahead of the arithmetic
    // Output channels whose weights are asked for together, a step ahead: a step of one channel x four positions is 72 instructions,
    // enough to hide the request behind; with fewer positions two channels (stride 2: 512 -> 512 @14x14 284 -> 203 us, 256 -> 256 @28x28
    // 181 -> 158; 512 -> 512 @7x7, one image, 32 -> 29).  Two x four positions run out of scalar registers (132 -> 180 us).
    static constexpr int UM = TN == 4 || KS == 5 ? 1 : 2, NU = TM / UM;
    static constexpr int MID = (TN - 1) * S + 1, STRIP = MID + 2 * PAD;   // columns under the strip, and with those beside it
    static_assert(NU == 1 || NU % 2 == 0, "two weight buffers");
    // 25 taps, more than one position: the two columns on a side are both inside the map or both outside -- at stride 1 (rows of whole strips and one
    // column: see Strips), at stride 2 on the left, and on the right of rows of an odd length
    static constexpr bool PAIRS = KS == 5 && TN > 1;
    static_assert(KS == 3 || KS == 5, "nine or 25 taps");
};

struct NineDims {
    int N, Ci, H, W, Co, Ho, Wo;
    Strips row;
    int strips;             // of TN positions per image
    int tiles, blocks;      // of 64 strips, of TM output channels
    int chunk, chunks;      // input channels per first-level sum (a power of two), and how many sums there are
};

// Columns c .. c + MID - 1 of a row, where c + k < W holds for every k that has a position
template <int S, int MID, class T>
__device__ __forceinline__ void load_mid(const T *p, float *v) {
    if constexpr (S == 1) {
        float u[MID];
        ld_strip<MID>(p, u);
#pragma unroll
        for (int k = 0; k < MID; ++k) v[k] = u[k];
    } else if constexpr (MID == 3) {
        float u[2];
        ld_strip<2>(p, u);
        v[0] = u[0];
        v[1] = u[1];
        v[2] = ldf(p + 2);
    } else {
        v[0] = ldf(p);
    }
}

// EVAL: the inference epilogue.
template <class C, class T, bool EVAL>
__global__ __launch_bounds__(C::NT, 4) void fwd_nine_kernel(const T *__restrict__ x, const float *__restrict__ w, T *__restrict__ y,
                                                            const NineDims d, const BnEval bn) {
    constexpr int S = C::S, TM = C::TM, TN = C::TN, MID = C::MID, STRIP = C::STRIP, NB = C::AHEAD + 1, UM = C::UM, NU = C::NU;
    constexpr int KS = C::KS, KK = C::KK, PAD = C::PAD;
    extern __shared__ __align__(16) float smem[];
    int tile, blk;
    xcd_tile(blockIdx.x, d.tiles, d.blocks, tile, blk);
    const int wave = C::SHARED ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0, waves = C::SHARED ? blockDim.x >> 6 : 1, lane = threadIdx.x & 63;
    const int sidx = tile * 64 + lane, sc = min(sidx, d.N * d.strips - 1), n = sc / d.strips, rest = sc - n * d.strips;
    const int ho = rest / d.row.per_row, s = rest - ho * d.row.per_row, wo = d.row.start(s, TN, d.Wo), co_base = blk * TM;
    const int plane = d.H * d.W, K = d.Ci * KK;
    uniform_f32_ptr wc = as_uniform(w);
    int wrow[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) wrow[m] = min(co_base + m, d.Co - 1) * K;
    // A uniform base per channel and the lane's distances from it in bytes (64 strips: far below 2^32), per row of the window: the
    // strip's own columns and the ones beside them.  What lies outside the map reads an element inside and is zeroed.
    const int n_first = __builtin_amdgcn_readfirstlane(n);
    const T *x_first = x + (size_t)n_first * d.Ci * plane;
    const int c0 = wo * S;
    // (nine taps: a distance per row and side; 25: one per row, and the side columns' distances from the strip, a further add per read)
    constexpr int NSIDE = KS == 3 ? 3 : 1;
    const bool ok_l = c0 > 0, ok_r = c0 + MID < d.W;
    bool ok[KS];
    unsigned in_row[KS], in_col[2 * PAD];   // 25 taps: all ones, or zero for what lies outside (lane masks of 20 elements are 40 scalar registers)
    unsigned off[KS], off_l[NSIDE], off_r[NSIDE];
    int beside[2 * PAD];
#pragma unroll
    for (int k = 0; k < 2 * PAD; ++k) {
        const int c = k < PAD ? k - PAD : MID + k - PAD;   // from the strip's first column
        const bool in = c0 + c >= 0 && c0 + c < d.W;
        in_col[k] = in ? ~0u : 0u;
        beside[k] = (in ? c : 0) * (int)sizeof(T);
    }
#pragma unroll
    for (int i = 0; i < KS; ++i) {
        const int h = ho * S + i - PAD;
        ok[i] = h >= 0 && h < d.H;
        in_row[i] = ok[i] ? ~0u : 0u;
        const int o = (n - n_first) * d.Ci * plane + min(max(h, 0), d.H - 1) * d.W + c0;
        off[i] = (unsigned)o * (unsigned)sizeof(T);
        if constexpr (KS == 3) {
            off_l[i] = (unsigned)(ok_l ? o - 1 : o) * (unsigned)sizeof(T);
            off_r[i] = (unsigned)(ok_r ? o + MID : o) * (unsigned)sizeof(T);
        }
    }

    typename C::Sums sums(smem, wave, lane, waves, d.chunks);
    float acc[TM][TN];
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t) acc[m][t] = 0.f;
    float xr[NB][KS][STRIP], wv[2][UM][KK];
    auto load_x = [&](const int b, const int ci) {
        const char *p = reinterpret_cast<const char *>(x_first + (size_t)ci * plane);
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            keep_offset(off[i]);
            if constexpr (KS == 5) {
                auto side = [&](const int k) { return reinterpret_cast<const T *>(p + (off[i] + (unsigned)beside[k])); };
                float *v = xr[b][i], u[4], q[2];
                if constexpr (C::PAIRS) {
                    ld_strip<2>(side(0), q);
                    v[0] = q[0]; v[1] = q[1];
                } else {
                    v[0] = ldf(side(0)); v[1] = ldf(side(1));
                }
                if constexpr (S == 2 && TN == 2 && C::EVEN) {
                    ld_strip<4>(reinterpret_cast<const T *>(p + off[i]), u);
                    v[2] = u[0]; v[3] = u[1]; v[4] = u[2]; v[5] = u[3];
                    v[6] = ldf(side(3));
                } else {
                    load_mid<S, MID>(reinterpret_cast<const T *>(p + off[i]), v + 2);
                    if constexpr (C::PAIRS) {
                        ld_strip<2>(side(2), q);
                        v[MID + 2] = q[0]; v[MID + 3] = q[1];
                    } else {
                        v[MID + 2] = ldf(side(2)); v[MID + 3] = ldf(side(3));
                    }
                }
                continue;
            }
            keep_offset(off_l[i % NSIDE]);
            if constexpr (!C::EVEN) keep_offset(off_r[i % NSIDE]);
            if constexpr (C::EVEN) {
                float u[MID + 1];
                ld_strip<MID + 1>(reinterpret_cast<const T *>(p + off[i]), u);
#pragma unroll
                for (int k = 0; k <= MID; ++k) xr[b][i][k + 1] = u[k];
            } else {
                load_mid<S, MID>(reinterpret_cast<const T *>(p + off[i]), &xr[b][i][1]);
                xr[b][i][MID + 1] = ldf(reinterpret_cast<const T *>(p + off_r[i % NSIDE]));
            }
            xr[b][i][0] = ldf(reinterpret_cast<const T *>(p + off_l[i % NSIDE]));
        }
    };
    auto load_w = [&](const int b, const int h, const int ci) {
#pragma unroll
        for (int u = 0; u < UM; ++u)
#pragma unroll
            for (int e = 0; e < KK; ++e) wv[b][u][e] = wc[wrow[h * UM + u] + ci * KK + e];
    };
    auto after = [&](const int c) { return ((c + 1) & (d.chunk - 1)) == 0 ? c + 1 + (waves - 1) * d.chunk : c + 1; };
    int ci = wave * d.chunk;   // (no more waves than chunks)
    {
        int cl = ci;   // the channel that x is read of next (the last one again behind the end)
#pragma unroll
        for (int b = 0; b < C::AHEAD; ++b) {
            load_x(b, cl);
            const int c = after(cl);
            cl = c < d.Ci ? c : cl;
        }
        load_w(0, 0, ci);
        // one input channel; weights one output channel ahead of the arithmetic
        auto channel = [&](const int cur) -> bool {
            const int next = after(ci);
            const bool chunk_end = ((ci + 1) & (d.chunk - 1)) == 0, more = next < d.Ci;
            const int cn = more ? next : ci;
#pragma unroll
            for (int i = 0; i < KS; ++i) {
                if (KS == 3 && i != PAD) {   // (the middle row is inside the map)
#pragma unroll
                    for (int k = PAD; k < PAD + MID; ++k) xr[cur][i][k] = ok[i] ? xr[cur][i][k] : 0.f;
                }
                if constexpr (KS == 5) {
                    auto keep = [&](float &v, const unsigned m) { v = __uint_as_float(__float_as_uint(v) & m); };
                    keep_offset(in_row[i]);
                    if (i != PAD) {
#pragma unroll
                        for (int k = PAD; k < PAD + MID; ++k) keep(xr[cur][i][k], in_row[i]);
                    }
#pragma unroll
                    for (int k = 0; k < 2 * PAD; ++k) {
                        const int e = C::PAIRS && !(C::EVEN && k >= PAD) ? k & ~1 : k;   // (the element of in_col that says so)
                        if (C::EVEN && k == PAD) {
                            keep(xr[cur][i][MID + k], in_row[i]);
                            continue;
                        }
                        keep_offset(in_col[e]);
                        keep(xr[cur][i][k < PAD ? k : MID + k], in_row[i] & in_col[e]);
                    }
                } else {
                    xr[cur][i][0] = ok[i] && ok_l ? xr[cur][i][0] : 0.f;
                    xr[cur][i][MID + 1] = ok[i] && (C::EVEN || ok_r) ? xr[cur][i][MID + 1] : 0.f;
                }
            }
#pragma unroll
            for (int h = 0; h < NU; ++h) {
                const int wb = (NU == 1 ? cur : h) & 1;
#pragma unroll
                for (int idx = 0; idx < UM * KK * TN; ++idx) {
                    const int t = idx % TN, j = idx / TN % KS, i = idx / TN / KS % KS, u = idx / TN / KK, m = h * UM + u;
                    const float a = wv[wb][u][i * KS + j], b = xr[cur][i][t * S + j];
                    acc[m][t] -= fabsf(a - b);
                    if (idx == 0) {
                        __builtin_amdgcn_sched_barrier(0);
                        load_w(wb ^ 1, h + 1 < NU ? h + 1 : 0, h + 1 < NU ? ci : cn);
                        if (h == 0) load_x((cur + C::AHEAD) % NB, cl);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            ci = next;
            {
                const int c = after(cl);
                cl = c < d.Ci ? c : cl;
            }
            if (chunk_end || !more) sums.add(acc);
            return more;
        };
#pragma unroll 1
        while (channel(0) && channel(1) && (NB == 2 || (channel(2) && channel(NB - 1)))) {}
        static_assert(NB == 2 || NB == 4, "the buffers take turns");
    }

    sums.finish(acc);

    unsigned own = 0;   // bit t: position wo + t is this lane's
#pragma unroll
    for (int t = 0; t < TN; ++t) own |= (sidx == sc && wo + t >= d.row.first(s, TN) ? 1u : 0u) << t;
    const int L = d.Ho * d.Wo, first = sums.first_channel();
    if (first < TM)
        finish_outputs<C::Sums::FM, TN, EVAL>(sums.tot, min(sums.per_wave, TM - first), own, co_base + first, d.Co, L, n * d.Co * L + ho * d.Wo + wo,
                                              TN > 1 && d.Wo % TN == 0, y, bn);
}

static int nine_tiles(const ConvDims &d, int tn) { return (int)ceil_div_l((long)d.N * d.Ho * ceil_div(d.Wo, tn), 64); }

// Waves that share the chunks of a launch of wgs workgroups: at most four where that makes 2800 waves, else as many as eight, or five
// where they need no more rounds: a CU holds 16 waves, three workgroups of five but two of six to eight (144 -> 144, 16 images, us: @28x28, 18 chunks, four waves 117, six 154,
// eight 116; @14x14, nine chunks, 32 images, four 74, five 66, eight 80).
static int nine_waves(const ConvDims &d, int chunk, long wgs) {
    const int chunks = ceil_div(d.Ci, chunk), full = full_chunks(d.Ci, chunk), four = full < 4 ? full : 4;
    if (wgs * four >= 2800) return four;
    return chunks >= 5 && ceil_div(chunks, 5) == ceil_div(chunks, 8) ? 5 : chunks < 8 ? chunks : 8;
}

// Output channels and positions per lane: 8 x 4 (stride 2: 8 x 2), 8 x 2, 4 x 1 or 2 x 1, the less the fewer waves there are.  A launch lasts as
// long as one wave's chain of channels -- 1.43, 0.93 and 0.46 us each -- or as the chip takes for the terms: 30, 26 and 12 per ps, 4 x 1 only
// 7 on rows that are shorter than 8 and 4 to 4.5 at stride 2, where its reads are what fills.  Between 8 x 4 and 8 x 2 the busiest CU's workgroups
// decide.  us, 8 x 4 / 8 x 2 / 4 x 1 / 2 x 1: 128 -> 128 @28x28, 4 images, 31 / 33 / 38 / 48, 256 -> 256 @14x14, 4, 54 / 37 / 41 / 50, 144 -> 144 @14x14, 128, 217 / 203;
// 86 -> 34 @29x29, 15, 42 / 28 / 33; 64 -> 64 @8x8, one, 23 / 17 / 8.4 / 6.7, 48 -> 12 @4x4, 64, 23 / 16 / 7.8 / 6.4, 64 -> 64 @8x8, 64, 23 / 17 / 14 / 17;
// stride 2: 40 -> 40 @16x16, 64 images, - / 17 / 20 / 31, 64 -> 64 @8x8, 64, - / 16 / 11.5 / 21.
LaneShape fwd_nine_shape(const ConvDims &d) {
    const int chunk = fwd_chunk(d), chunks = ceil_div(d.Ci, fwd_chunk(d));
    if (d.kh == 5) {   // 4 x 4, or 4 x 1 for few waves (one image of 64 -> 64 @32x32, 512 waves of 4 x 4, 18.6 / 10.2 us; 64 of @8x8, 2048 waves, 19.8 / 26) and
                       // rows of five, which have no strips without a cut pair; stride 2: 4 x 2 (64 -> 64 @16x16, one image, 12.7; 4 x 1 24.6)
        const int most = d.stride == 1 ? 4 : 2;
        const int tn = d.Wo >= most && (d.stride == 2 || d.W != 5) ? most : 1;
        const long wgs = (long)nine_tiles(d, tn) * ceil_div(d.Co, 4);
        const int waves = nine_waves(d, chunk, wgs);
        if (tn == 4 && wgs * waves < 1000) return {4, 1, nine_waves(d, chunk, (long)nine_tiles(d, 1) * ceil_div(d.Co, 4))};
        return {4, tn, waves};
    }
    const int most = d.stride == 1 ? 4 : 2;
    int tn = d.Wo >= most ? most : d.Wo >= 2 ? 2 : 1;
    auto wgs = [&](int n) { return (long)nine_tiles(d, n) * ceil_div(d.Co, n == 1 ? 4 : 8); };
    if (tn == 4) {   // the busiest CU's workgroups, by what one of 8 x 4 and of 8 x 2 takes; and waves enough to overlap their chains
        const int waves = nine_waves(d, chunk, wgs(4));
        if (wgs(4) * waves < (waves == 1 ? 3300 : waves <= 4 ? 1800 : 1300) || 26 * 2 * ceil_div_l(wgs(4), 256) > 30 * ceil_div_l(wgs(2), 256)) tn = 2;
    }
    const int waves = nine_waves(d, chunk, wgs(tn)), share = chunks < 8 ? chunks : 8;
    const float terms = (float)d.K() * d.Co * d.N * d.Ho * d.Wo;
    const float wide = fmaxf((tn == 4 ? 1.43f : 0.93f) * min(ceil_div(chunks, waves) * chunk, d.Ci), terms / (tn == 4 ? 30e6f : 26e6f));
    const float narrow = fmaxf(0.46f * min(ceil_div(chunks, share) * chunk, d.Ci),
                               d.stride == 2 ? 3.f + terms / (d.Wo < 8 ? 4e6f : 4.5e6f) : terms / (d.Wo < 8 ? 7e6f : 12e6f));
    if (tn > 1 && narrow >= wide) return {8, tn, waves};
    return {wgs(1) * share <= (d.stride == 2 ? 200 : chunks <= 8 ? 1024 : 600) ? 2 : 4, 1, share};
}

// Layers it takes: the distance of a wave's strips from the first one's image has to fit 32 bits, and so have the launch's threads.
bool fwd_nine_supported(const ConvDims &d) {
    if (d.kh != d.kw || (d.kh != 3 && d.kh != 5) || d.pad != d.kh / 2 || d.stride < 1 || d.stride > 2) return false;
    if ((images_ahead(d, (long)d.Ho * ceil_div(d.Wo, 4)) * d.Ci + 1) * d.H * d.W > 0x3fffffffL) return false;
    const LaneShape shape = fwd_nine_shape(d);
    return (long)nine_tiles(d, shape.tn) * ceil_div(d.Co, shape.tm) * 64 * shape.waves <= kMaxThreads;
}

template <class C, class T, bool EVAL>
static int launch_nine(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn, int waves) {
    const int per_row = ceil_div(d.Wo, C::TN);
    const NineDims t{d.N, d.Ci, d.H, d.W, d.Co, d.Ho, d.Wo, Strips{per_row, C::PAIRS && C::S == 1 && d.Wo % C::TN == 1 ? 1 : kNoShift}, per_row * d.Ho, nine_tiles(d, C::TN), ceil_div(d.Co, C::TM), fwd_chunk(d), ceil_div(d.Ci, fwd_chunk(d))};
    const int lds = waves * C::Sums::WAVE_FLOATS * 4;
    if (int rc = allow_dynamic_lds<&fwd_nine_kernel<C, T, EVAL>>(8 * C::Sums::WAVE_FLOATS * 4)) return rc;
    hipLaunchKernelGGL((fwd_nine_kernel<C, T, EVAL>), dim3((unsigned)t.tiles * t.blocks), dim3(64 * waves), lds, s, x, w, y, t, bn);
    return check_launch();
}

template <class T>
int launch_fwd_nine(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn) {
    const LaneShape shape = fwd_nine_shape(d);
    auto run = [&](auto cfg) {
        using C = decltype(cfg);
        if constexpr (sizeof(T) == 4) {
            if (bn.gamma) return launch_nine<C, T, true>(x, w, y, d, s, bn, shape.waves);
        }
        return launch_nine<C, T, false>(x, w, y, d, s, bn, shape.waves);
    };
    auto waves = [&](auto shared) {
        constexpr bool SHARED = decltype(shared)::value;
        if (d.kh == 5) {
            if (d.stride == 1) return shape.tn == 4 ? run(NineCfg<1, 4, 4, SHARED, false, 5>{}) : run(NineCfg<1, 4, 1, SHARED, false, 5>{});
            if (shape.tn == 2) return d.W % 2 ? run(NineCfg<2, 4, 2, SHARED, false, 5>{}) : run(NineCfg<2, 4, 2, SHARED, true, 5>{});
            return run(NineCfg<2, 4, 1, SHARED, false, 5>{});
        }
        if (d.stride == 1) {
            if (shape.tn == 4) return run(NineCfg<1, 8, 4, SHARED>{});
            if (shape.tn == 2) return run(NineCfg<1, 8, 2, SHARED>{});
            return shape.tm == 4 ? run(NineCfg<1, 4, 1, SHARED>{}) : run(NineCfg<1, 2, 1, SHARED>{});
        }
        if (shape.tn == 2) return d.W % 2 ? run(NineCfg<2, 8, 2, SHARED>{}) : run(NineCfg<2, 8, 2, SHARED, true>{});
        return shape.tm == 4 ? run(NineCfg<2, 4, 1, SHARED>{}) : run(NineCfg<2, 2, 1, SHARED>{});
    };
    return shape.waves == 1 ? waves(std::false_type{}) : waves(std::true_type{});
}
template int launch_fwd_nine<float>(const float *, const float *, float *, const ConvDims &, hipStream_t, const BnEval &);
template int launch_fwd_nine<bf16_t>(const bf16_t *, const float *, bf16_t *, const ConvDims &, hipStream_t, const BnEval &);

}  // namespace adder

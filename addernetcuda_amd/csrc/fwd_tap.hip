// Forward of 1x1 layers without padding, of any stride, NCHW in -> NCHW out:
//   y[n,co,p] = - sum_ci | w[co,ci] - x[n,ci,p] |        (adder_cuda/adder.cu:19-70 behind the unfold of adder.py:32)
//
// Two vector instructions per term bound it, as in fwd.hip: 73 T lane-instructions/s is what a bare stream of the pair reaches with
// two waves on each of a SIMD's two issue ports (62 T with one, 31 T with one wave per SIMD), 90 us for the 3.3e9 terms of
// 1024 -> 256 @14x14, 64 images.  A single tap shares no x between neighbouring positions, so there is nothing to stage: a wave
// reads its strips of x straight into registers, four channels ahead (one position per lane: twelve).  What that leaves to choose
// is how many waves there are, and the channels are what can be shared out without more reads per term: the waves of a
// workgroup have the same 8 x 64 * TN outputs and take the chunks of channels in turn, whose sums meet in LDS in channel order (ChunkSums;
// sums that meet once at the end would be up to 15 % faster, and other bits).
// us, 256 positions x 32 channels staged in LDS per workgroup (one wave for all channels) -> this:
//   32 images: 256 -> 64 @56x56 102 -> 93, 256 -> 128 168 -> 160, 512 -> 256 @28x28 185 -> 163, 256 -> 1024 @14x14 93 -> 87,
//   1024 -> 256 114 -> 108, 512 -> 2048 @7x7 109 -> 96, 2048 -> 512 273 -> 114; 1024 -> 256 @14x14, 64 images 185 -> 175, 8 images 106 -> 40,
//   one image (there the kernel for few positions) 33 -> 15; 300 -> 48 @8x8, 64 images 36 -> 11.
// Layers the plain kernel of conv1x1.hip had (fewer channels, or no multiple of four): 373 -> 9 @13x16, 4 images, 75 -> 7.8, 32 -> 19 @7x7, 68 images, 15.1 ->
// 4.0, 32 -> 200 @56x56, 64 images, 106 -> 70, 40 -> 16 @64x64, 200 images, 49 -> 38.  Strided ones, tiles or the kernel for few positions -> this: 239 -> 208
// @13x13, 144 images, 58 -> 32, 812 -> 226 @61x61, 2 images, 124 -> 43, 256 -> 512 @56x56, one image, 75 -> 18.
// Tried on the way: 16 channels x 2 positions per lane at stride 1 146 -> 187; the next chunk's weight lines asked for a chunk early 131 -> 140; x of eight waves
// staged in LDS 1024 -> 256 176.
#include "wave_split.hpp"

#include <type_traits>

namespace adder {

// TM output channels x TN adjacent positions per lane; SHARED: two to eight waves share the input channels.
// SUB: a stride above one.  A lane then reads positions 64 apart, so that the lanes of a read are neighbours (four adjacent positions per lane are four
// reads that each touch every line under the tile), and LDS hands each its strip at the end.
template <int TM_, int TN_, bool SHARED_, bool SUB_>
struct TapCfg {
    static constexpr int TM = TM_, TN = TN_, NT = SHARED_ ? 512 : 64;
    static constexpr bool SHARED = SHARED_, SUB = SUB_;
    using Sums = ChunkSums<TM, TN, SHARED, SUB>;
    static constexpr int AHEAD = TN == 1 ? 3 : 1;   // groups of four input channels that x is asked for ahead of the arithmetic
};

static constexpr int kTapTM = 8;
static int tap_tiles(const ConvDims &d, int tn) { return (int)ceil_div_l((long)d.N * ceil_div(d.Ho * d.Wo, tn), 64); }

struct TapDims {
    int N, Ci, Co, L;       // L = Ho * Wo positions per image
    int plane, W, Wo, stride;   // of x, whose rows and columns 0, stride, 2 stride, ... are read
    int strips;             // of TN positions per image; the last one of an image is moved back to end at L
    int tiles, blocks;      // of 64 strips, of TM output channels
    int chunk, chunks;      // input channels per first-level sum (a power of two), and how many sums there are
};

template <class C, class T, bool EVAL>
__global__ __launch_bounds__(C::NT, 4) void fwd_tap_kernel(const T *__restrict__ x, const float *__restrict__ w, T *__restrict__ y,
                                                           const TapDims d, const BnEval bn) {
    constexpr int TM = C::TM, TN = C::TN, CQ = 4, UM = TM * TN >= 32 ? 2 : (TM < 4 ? TM : 4), NU = TM / UM, NB = C::AHEAD + 1;
    constexpr bool SUB = C::SUB;
    static_assert(NU == 1 || NU % 2 == 0, "the weight buffers alternate from unit to unit");
    extern __shared__ __align__(16) float smem[];
    int tile, blk;
    xcd_tile(blockIdx.x, d.tiles, d.blocks, tile, blk);
    const int wave = C::SHARED ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0, waves = C::SHARED ? blockDim.x >> 6 : 1, lane = threadIdx.x & 63;
    const int sidx = tile * 64 + lane, sc = min(sidx, d.N * d.strips - 1), n = sc / d.strips, s = sc - n * d.strips;
    const int p0 = min(s * TN, d.L - TN), co_base = blk * TM;
    uniform_f32_ptr wc = as_uniform(w);
    int wrow[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) wrow[m] = min(co_base + m, d.Co - 1) * d.Ci;

    typename C::Sums sums(smem, wave, lane, waves, d.chunks);
    float acc[TM][TN];
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t) acc[m][t] = 0.f;
    float xr[NB][CQ][TN], wv[2][UM][CQ];
    // a uniform base per channel and the lane's distance from it in bytes (64 strips: far below 2^32): no address registers
    const int n_first = __builtin_amdgcn_readfirstlane(n);
    unsigned xoff[SUB ? TN : 1];
    if constexpr (SUB) {
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            const int q = t * 64 + lane, qs = min(tile * 64 + q / TN, d.N * d.strips - 1), qn = qs / d.strips;
            const int p = min((qs - qn * d.strips) * TN, d.L - TN) + q % TN, ho = p / d.Wo;
            xoff[t] = (unsigned)((qn - n_first) * d.Ci * d.plane + (ho * d.W + (p - ho * d.Wo)) * d.stride) * (unsigned)sizeof(T);
        }
    } else {
        xoff[0] = (unsigned)((n - n_first) * d.Ci * d.plane + p0) * (unsigned)sizeof(T);
    }
    const T *x_first = x + (size_t)n_first * d.Ci * d.plane;
    auto load_channel = [&](const int ci, float (&v)[TN]) {
        const char *p = reinterpret_cast<const char *>(x_first + (size_t)ci * d.plane);
        if constexpr (SUB) {
#pragma unroll
            for (int t = 0; t < TN; ++t) v[t] = ldf(reinterpret_cast<const T *>(p + xoff[t]));
        } else {
            ld_strip<TN>(reinterpret_cast<const T *>(p + xoff[0]), v);
        }
    };
    auto load_x = [&](const int b, const int ci) {
#pragma unroll
        for (int t = 0; t < (SUB ? TN : 1); ++t) keep_offset(xoff[t]);
#pragma unroll
        for (int e = 0; e < CQ; ++e) load_channel(ci + e, xr[b][e]);
    };
    auto load_w = [&](const int b, const int h, const int ci) {
#pragma unroll
        for (int u = 0; u < UM; ++u)
#pragma unroll
            for (int e = 0; e < CQ; ++e) wv[b][u][e] = wc[wrow[h * UM + u] + ci + e];
    };
    const int whole = d.Ci & ~(CQ - 1);   // channels in groups of CQ; the one to three behind them follow one by one, in the last chunk
    auto finish_chunk = [&]() __attribute__((always_inline)) {
        if (whole < d.Ci && sums.chunk() + 1 == d.chunks) {
#pragma unroll 1
            for (int c = whole; c < d.Ci; ++c) {
                float v[TN];
                load_channel(c, v);
#pragma unroll
                for (int m = 0; m < TM; ++m)
#pragma unroll
                    for (int t = 0; t < TN; ++t) acc[m][t] -= fabsf(wc[wrow[m] + c] - v[t]);
            }
        }
        sums.add(acc);
    };
    int ci = wave * d.chunk;   // (no more waves than chunks)
    if (ci < whole) {
        auto after = [&](const int c) { return ((c + CQ) & (d.chunk - 1)) == 0 ? c + CQ + (waves - 1) * d.chunk : c + CQ; };
        int cl = ci;   // the group that x is read of next (the last one again behind the end)
#pragma unroll
        for (int b = 0; b < C::AHEAD; ++b) {
            load_x(b, cl);
            const int c = after(cl);
            cl = c < whole ? c : cl;
        }
        load_w(0, 0, ci);
        auto group = [&](const int cur) __attribute__((always_inline)) -> bool {
            const int next = after(ci);
            const bool chunk_end = ((ci + CQ) & (d.chunk - 1)) == 0, more = next < whole;
            const int cn = more ? next : ci;
#pragma unroll
            for (int h = 0; h < NU; ++h) {
                const int wb = (cur * (NU & 1) + h) & 1;
#pragma unroll
                for (int idx = 0; idx < UM * CQ * TN; ++idx) {
                    const int t = idx % TN, u = (idx / TN) % UM, e = idx / TN / UM, m = h * UM + u;
                    acc[m][t] -= fabsf(wv[wb][u][e] - xr[cur][e][t]);
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
                cl = c < whole ? c : cl;
            }
            if (chunk_end || !more) finish_chunk();
            return more;
        };
#pragma unroll 1
        while (group(0) && group(1) && (NB == 2 || (group(2) && group(NB - 1)))) {}
        static_assert(NB == 2 || NB == 4, "the buffers take turns");
    }
    if (sums.pending()) finish_chunk();   // (a last chunk of fewer than CQ channels)
    sums.finish(acc);

    unsigned own = 0;   // bit t: position p0 + t is this lane's
#pragma unroll
    for (int t = 0; t < TN; ++t) own |= (sidx == sc && p0 + t >= s * TN ? 1u : 0u) << t;
    const int first = sums.first_channel();
    if (first < TM)
        finish_outputs<C::Sums::FM, TN, EVAL>(sums.tot, min(sums.per_wave, TM - first), own, co_base + first, d.Co, d.L, n * d.Co * d.L + p0,
                                              TN > 1 && d.L % TN == 0, y, bn);
}

// Chunks of a layer: one to three channels behind the groups of four join the last chunk, or are one where a chunk ends with the groups
// (strides that the plain kernel of conv1x1.hip does not have; that one folds in front of a group only).
static int tap_chunks(const ConvDims &d) {
    const int chunk = fwd_chunk(d);
    return conv1x1_supported(d, nullptr, nullptr) ? max(1, ceil_div(d.Ci & ~3, chunk)) : ceil_div(d.Ci, chunk);
}

// Output channels and positions per lane, and waves.  8 x 4, unless the launch is then about one workgroup per CU or less: 8 x 2 (us, 8 x 4 / 8 x 2:
// 1024 -> 256 @14x14, 4 images 42 / 34; 512 -> 128 @28x28, 4 images, 22.7 / 24.3), and one position where that leaves half the chip idle or costs no
// more tiles (64 strips of two on a plane of 49; 2048 -> 512 @7x7, 4 images, 78 / 55 / 45); 4 x 1 up to 1400 waves of 8 x 1, whose weights are what
// a wave waits for (8 x 1 / 4 x 1: 300 -> 48 @8x8, one image, 9.4 / 6.9, 64 images, 1920 waves, 13.9 / 13.2, 11.9 with 8 x 2).
LaneShape fwd_tap_shape(const ConvDims &d) {
    const int L = d.Ho * d.Wo, blocks = ceil_div(d.Co, kTapTM), chunks = tap_chunks(d), waves = waves_for(chunks, 8);
    int tn = L >= 4 ? 4 : L >= 2 ? 2 : 1;
    if (tn == 4 && (long)tap_tiles(d, 4) * blocks < 256 + 256 / waves) tn = 2;
    if (tn == 2 && ((long)tap_tiles(d, 2) * blocks < 128 || tap_tiles(d, 1) == tap_tiles(d, 2))) tn = 1;
    const long wgs = (long)tap_tiles(d, tn) * blocks;
    if (tn == 1 && wgs * waves <= 1400) return {4, 1, waves};
    // With a stride it is 16 channels x 2 positions instead of 8 x 4: what a line holds beside the sampled positions comes with it, and half as many
    // blocks ask for it.  us, 8 x 4 / 16 x 2: 105 -> 620 @58x57, 44 images, 220 / 138; 256 -> 512 @56x56, 4 images, 55 / 47, 512 -> 1024 @28x28 64 / 53.
    if (tn == 4 && d.stride > 1 && d.Ci > 16) return {16, 2, waves};
    if (tn < 4) return {kTapTM, tn, waves};
    // (large launches: us with 1 / 2 / 4 / 8 waves, 64 -> 256 @56x56, 32 images, 81 / 85 / 91 / 91, 80 -> 128 @28x28, 64 images, 37 / 38 / 40 / 48, 128 -> 512 @28x28, 32, 85 / 83 / 84 / 96,
    // 256 -> 64 @56x56 100 / 93 / 87 / 98, 512 -> 128 @28x28 114 / 104 / 92 / 100)
    const int full = full_chunks(d.Ci, fwd_chunk(d)), large = full <= 5 ? 1 : full <= 8 ? 2 : 4;
    if (wgs * large >= 3000) return {kTapTM, 4, large};
    return {kTapTM, 4, wgs * 4 >= 3000 && chunks >= 4 ? 4 : waves};
}

// Layers it takes: all but large strided ones of 8-channel chunks (fwd_strided_tile_supported) and wide maps of few channels, which memory bounds and conv1x1.hip reads in rows (24 -> 48 @32x32, 64 images, 9.6 us there, 10.1
// here; 8 -> 64 @64x64 of stride 2 10.1, 10.5; 7 -> 227 @41x40, 26 images, bfloat16, 11.1, 11.5; 32 -> 200 @56x56 106, 70).  The distance of a wave's
// strips from the first one's image has to fit 32 bits, and so have the launch's threads.
bool fwd_tap_supported(const ConvDims &d) {
    if (d.kh != 1 || d.kw != 1 || d.pad != 0) return false;
    if (d.Ci <= 24 && d.stride <= 2 && (long)d.N * d.Ho * d.Wo >= 16384) return false;
    if ((images_ahead(d, ceil_div_l((long)d.Ho * d.Wo, 4)) * d.Ci + 1) * d.H * d.W > 0x3fffffffL) return false;
    const LaneShape shape = fwd_tap_shape(d);
    return (long)tap_tiles(d, shape.tn) * ceil_div(d.Co, shape.tm) * 64 * shape.waves <= kMaxThreads;
}

template <class C, class T, bool EVAL>
static int launch_tap(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn, int waves) {
    const TapDims t{d.N, d.Ci, d.Co, d.Ho * d.Wo, d.H * d.W, d.W, d.Wo, d.stride, ceil_div(d.Ho * d.Wo, C::TN), tap_tiles(d, C::TN), ceil_div(d.Co, C::TM),
                    fwd_chunk(d), tap_chunks(d)};
    const int lds = waves * C::Sums::WAVE_FLOATS * 4;
    if (int rc = allow_dynamic_lds<&fwd_tap_kernel<C, T, EVAL>>(8 * C::Sums::WAVE_FLOATS * 4)) return rc;
    hipLaunchKernelGGL((fwd_tap_kernel<C, T, EVAL>), dim3((unsigned)t.tiles * t.blocks), dim3(64 * waves), lds, s, x, w, y, t, bn);
    return check_launch();
}

template <class T>
int launch_fwd_tap(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn) {
    const LaneShape shape = fwd_tap_shape(d);
    auto run = [&](auto cfg) {
        using C = decltype(cfg);
        if constexpr (sizeof(T) == 4) {
            if (bn.gamma) return launch_tap<C, T, true>(x, w, y, d, s, bn, shape.waves);
        }
        return launch_tap<C, T, false>(x, w, y, d, s, bn, shape.waves);
    };
    auto per_lane = [&](auto shared, auto sub) {
        constexpr bool SHARED = decltype(shared)::value, SUB = decltype(sub)::value;
        if constexpr (SUB) {
            if (shape.tm == 16) return run(TapCfg<16, 2, SHARED, SUB>{});
        }
        if constexpr (!SUB || !SHARED) {   // (a shared strided layer of four positions is the former)
            if (shape.tn == 4) return run(TapCfg<kTapTM, 4, SHARED, SUB>{});
        }
        if (shape.tn == 2) return run(TapCfg<kTapTM, 2, SHARED, SUB>{});
        return shape.tm == 4 ? run(TapCfg<4, 1, SHARED, SUB>{}) : run(TapCfg<kTapTM, 1, SHARED, SUB>{});
    };
    if (d.stride == 1) return shape.waves == 1 ? per_lane(std::false_type{}, std::false_type{}) : per_lane(std::true_type{}, std::false_type{});
    return shape.waves == 1 ? per_lane(std::false_type{}, std::true_type{}) : per_lane(std::true_type{}, std::true_type{});
}
template int launch_fwd_tap<float>(const float *, const float *, float *, const ConvDims &, hipStream_t, const BnEval &);
template int launch_fwd_tap<bf16_t>(const bf16_t *, const float *, bf16_t *, const ConvDims &, hipStream_t, const BnEval &);

}  // namespace adder

// Forward of 1x1 layers without padding, of any stride, NCHW in -> NCHW out:
//   y[n,co,p] = - sum_ci | w[co,ci] - x[n,ci,p] |        (adder_cuda/adder.cu:19-70 behind the unfold of adder.py:32)
//
// Two vector instructions per term bound it, as in fwd.hip: 73 T lane-instructions/s is what a bare stream of the pair reaches with
// two waves on each of a SIMD's two issue ports (62 T with one, 31 T with one wave per SIMD), 90 us for the 3.3e9 terms of
// 1024 -> 256 @14x14, 64 images.  A single tap shares no x between neighbouring positions, so there is nothing to stage: a wave
// reads its strips of x straight into registers, four channels ahead, and runs without a barrier.  What that leaves to choose
// is how many waves there are, and the channels are what can be shared out without more reads per term: the KSP waves of a
// workgroup have the same 8 x 64 * TN outputs and take 16-channel chunks in turn; their sums meet in LDS at the end.
// us, 256 positions x 32 channels staged in LDS per workgroup (one wave for all channels) -> this:
//   32 images: 256 -> 64 @56x56 89 -> 72, 256 -> 128 151 -> 130, 512 -> 256 @28x28 171 -> 133, 256 -> 1024 @14x14 86 -> 71,
//   1024 -> 256 109 -> 82, 512 -> 2048 @7x7 104 -> 84, 2048 -> 512 273 -> 97; 1024 -> 256 @14x14, 64 images 178 -> 140, 8 images 106 -> 31,
//   one image (there the kernel for few positions) 34 -> 18; 300 -> 48 @8x8, 64 images 36 -> 8.
// Layers the plain kernel of conv1x1.hip had (fewer channels, or no multiple of four): 373 -> 9 @13x16, 4 images, 75 -> 8, 32 -> 19 @7x7, 68 images, 15.5 ->
// 5.5, 32 -> 200 @56x56, 64 images, 101 -> 75, 40 -> 16 @64x64, 200 images, 45 -> 34.  Strided ones, tiles or the kernel for few positions -> this: 239 -> 208
// @13x13, 144 images, 56 -> 28, 812 -> 226 @61x61, 2 images, 123 -> 37, 256 -> 512 @56x56, one image, 75 -> 14; 32 images: tap_tall.
// Tried on the way: sums of sums in LDS instead of registers (116 -> 84 registers) 131 -> 141 us; 16 channels x 2 positions per lane
// 146 -> 187; the next chunk's weight lines asked for a chunk early 131 -> 140; x of eight waves staged in LDS 1024 -> 256 176.
#include "wave_split.hpp"

#include <type_traits>

namespace adder {

// TM output channels x TN adjacent positions per lane; wave v of the KSP of a workgroup takes the chunks v, v + KSP, ... of input
// channels.  Two-level sums in registers (a chunk, a wave's chunks), the waves' sums are added in the order of the waves.
template <int TM_, int TN_, int KSP_>
struct TapCfg {
    static constexpr int TM = TM_, TN = TN_, KSP = KSP_, NT = 64 * KSP, CC = kTapChunk, FM = kFinished<TM, KSP>;
    static constexpr int LDS_BYTES = KSP * TM * TN * 64 * 4;
};

static constexpr int kTapTM = 8;
static int tap_tiles(const ConvDims &d, int tn) { return (int)ceil_div_l((long)d.N * ceil_div(d.Ho * d.Wo, tn), 64); }

struct TapDims {
    int N, Ci, Co, L;       // L = Ho * Wo positions per image
    int plane, W, Wo, stride;   // of x, whose rows and columns 0, stride, 2 stride, ... are read
    int strips;             // of TN positions per image; the last one of an image is moved back to end at L
    int tiles, blocks;      // of 64 strips, of TM output channels
};

// SUB: a stride above one.  A lane then reads positions 64 apart, so that the lanes of a read are neighbours (four adjacent positions per lane are four
// reads that each touch every line under the tile), and LDS hands each its strip at the end.
template <class C, class T, bool EVAL, bool SUB>
__global__ __launch_bounds__(C::NT) void fwd_tap_kernel(const T *__restrict__ x, const float *__restrict__ w, T *__restrict__ y,
                                                        double *__restrict__ stats, const TapDims d, const BnEval bn) {
    constexpr int TM = C::TM, TN = C::TN, KSP = C::KSP, CQ = 4, UM = TM * TN >= 32 ? 2 : (TM < 4 ? TM : 4), NU = TM / UM, FM = C::FM;
    static_assert(NU == 1 || NU % 2 == 0, "the weight buffers alternate from unit to unit");
    extern __shared__ __align__(16) float smem[];
    int tile, blk;
    xcd_tile(blockIdx.x, d.tiles, d.blocks, tile, blk);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int sidx = tile * 64 + lane, sc = min(sidx, d.N * d.strips - 1), n = sc / d.strips, s = sc - n * d.strips;
    const int p0 = min(s * TN, d.L - TN), co_base = blk * TM;
    uniform_f32_ptr wc = as_uniform(w);
    int wrow[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) wrow[m] = min(co_base + m, d.Co - 1) * d.Ci;

    float acc[TM][TN], tot[TM][TN];
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t) acc[m][t] = tot[m][t] = 0.f;
    float xr[2][CQ][TN], wv[2][UM][CQ];
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
    const int whole = d.Ci & ~(CQ - 1);   // channels in groups of CQ; the one to three behind them follow one by one
    int ci = wave * C::CC;
    if (ci < whole) {
        load_x(0, ci);
        load_w(0, 0, ci);
        auto half = [&](const int cur) -> bool {
            int next = ci + CQ;
            const bool chunk_end = (next & (C::CC - 1)) == 0;
            if (chunk_end) next += (KSP - 1) * C::CC;
            const bool more = next < whole;
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
                        if (h == 0) load_x(cur ^ 1, cn);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            ci = next;
            if (chunk_end || !more) {
#pragma unroll
                for (int m = 0; m < TM; ++m)
#pragma unroll
                    for (int t = 0; t < TN; ++t) { tot[m][t] += acc[m][t]; acc[m][t] = 0.f; }
            }
            return more;
        };
#pragma unroll 1
        while (half(0) && half(1)) {}
    }
    if (whole < d.Ci && wave == whole / C::CC % KSP) {
#pragma unroll 1
        for (int c = whole; c < d.Ci; ++c) {
            float v[TN];
            load_channel(c, v);
#pragma unroll
            for (int m = 0; m < TM; ++m)
#pragma unroll
                for (int t = 0; t < TN; ++t) tot[m][t] -= fabsf(wc[wrow[m] + c] - v[t]);
        }
    }

    float r[FM][TN];
    add_waves<TM, TN, KSP, SUB>(smem, wave, lane, tot, r);
    unsigned own = 0;   // bit t: position p0 + t is this lane's
#pragma unroll
    for (int t = 0; t < TN; ++t) own |= (sidx == sc && p0 + t >= s * TN ? 1u : 0u) << t;
    finish_outputs<FM, TN, EVAL>(r, own, co_base + wave * FM, d.Co, d.L, n * d.Co * d.L + p0, TN > 1 && d.L % TN == 0, y, stats, d.tiles,
                                 tile, lane, bn);
}

template <class C, class T>
static int launch_tap(const T *x, const float *w, T *y, double *stats, const ConvDims &d, hipStream_t s, const BnEval &bn) {
    const TapDims t{d.N, d.Ci, d.Co, d.Ho * d.Wo, d.H * d.W, d.W, d.Wo, d.stride, ceil_div(d.Ho * d.Wo, C::TN), tap_tiles(d, C::TN), ceil_div(d.Co, C::TM)};
    const long grid = (long)t.tiles * t.blocks;
    if (grid > 0x7fffffL) return ADDER_ERR_TOO_LARGE;   // (2^32 threads; tensors below 2^31 elements stay far from it)
    auto launch = [&](auto eval, auto sub) {
        constexpr bool EVAL = decltype(eval)::value, SUB = decltype(sub)::value;
        if (int rc = allow_dynamic_lds<&fwd_tap_kernel<C, T, EVAL, SUB>>(C::LDS_BYTES)) return rc;
        hipLaunchKernelGGL((fwd_tap_kernel<C, T, EVAL, SUB>), dim3((unsigned)grid), dim3(C::NT), C::LDS_BYTES, s, x, w, y, stats, t, bn);
        return check_launch();
    };
    if constexpr (sizeof(T) == 4) {
        if (bn.gamma) return d.stride == 1 ? launch(std::true_type{}, std::false_type{}) : launch(std::true_type{}, std::true_type{});
    }
    return d.stride == 1 ? launch(std::false_type{}, std::false_type{}) : launch(std::false_type{}, std::true_type{});
}

// Waves that share the channels: as many as have two chunks each (but one up to 16 channels, two from 17 on), by the channels alone, so that a layer's results have the same
// bits whatever the batch.  us with 2 / 4 / 8 of them, 32 images: 64 -> 256 @56x56 76 / 82 / 114, 128 -> 512 @28x28 71 / 74 / 80,
// 256 -> 128 @56x56 132 / 130 / 137, 512 -> 256 @28x28 147 / 133 / 133, 1024 -> 256 @14x14 105 / 87 / 82, 2048 -> 512 @7x7 247 / 145 / 97.
static int tap_waves(int Ci) { return Ci <= kTapChunk ? 1 : Ci <= 128 ? 2 : Ci <= 256 ? 4 : 8; }

// Positions per lane.  Four, unless the launch is then about one workgroup per CU or less: two (us, four -> two: 1024 -> 256 @14x14, 8
// images, 224 workgroups, 34 -> 31, 4 images 27 -> 23; 512 -> 128 @28x28, 8 images, 400 workgroups, 25 -> 28), and one where that
// leaves half the chip idle or costs no more tiles (64 strips of two on a plane of 49): 512 -> 128 @28x28, one image, 11.4 -> 10.0,
// 512 -> 2048 @7x7 11.5 -> 10.0; 256 -> 64 @56x56, 200 workgroups, 7.0 -> 8.5.
static int tap_positions(const ConvDims &d) {
    const int L = d.Ho * d.Wo, blocks = ceil_div(d.Co, kTapTM);
    int tn = L >= 4 ? 4 : L >= 2 ? 2 : 1;
    if (tn == 4 && (long)tap_tiles(d, 4) * blocks < 256 + 256 / tap_waves(d.Ci)) tn = 2;
    if (tn == 2 && ((long)tap_tiles(d, 2) * blocks < 128 || tap_tiles(d, 1) == tap_tiles(d, 2))) tn = 1;
    return tn;
}

// With a stride it is 16 channels x 2 positions instead of 8 x 4: what a line holds beside the sampled positions comes with it, and half as many
// blocks ask for it.  us, 8 x 4 / 16 x 2 (tiles in LDS there were): 32 images 256 -> 512 @56x56 269 / 162 (198), 512 -> 1024 @28x28 238 / 221 (198),
// 1024 -> 2048 @14x14 633 / 267 (274), 4 images 512 -> 1024 @28x28 44 / 41 (113).
static bool tap_tall(const ConvDims &d) { return d.stride > 1 && d.Ci > kTapChunk && tap_positions(d) == 4; }

// Layers it takes: all but wide maps of few channels, which memory bounds and conv1x1.hip reads in rows (24 -> 48 @32x32, 64 images, 9.6 us there, 10.1
// here; 8 -> 64 @64x64 of stride 2 10.1, 10.5; 7 -> 227 @41x40, 26 images, bfloat16, 11.1, 11.5; 32 -> 200 @56x56 101, 75).  The distance of a wave's
// strips from the first one's image has to fit 32 bits.
bool fwd_tap_supported(const ConvDims &d) {
    if (d.kh != 1 || d.kw != 1 || d.pad != 0) return false;
    if (d.Ci <= 24 && d.stride <= 2 && (long)d.N * d.Ho * d.Wo >= 16384) return false;
    const long images = 63 / ceil_div_l((long)d.Ho * d.Wo, 4) + 1;
    return (images * d.Ci + 1) * d.H * d.W <= 0x3fffffffL;
}
int fwd_tap_stats_slots(const ConvDims &d) { return tap_tiles(d, tap_tall(d) ? 2 : tap_positions(d)); }

template <class T>
int launch_fwd_tap(const T *x, const float *w, T *y, double *stats, const ConvDims &d, hipStream_t s, const BnEval &bn) {
    auto run = [&](auto tn, auto ksp) {
        if constexpr (decltype(tn)::value == 4 && decltype(ksp)::value > 1)
            if (tap_tall(d)) return launch_tap<TapCfg<16, 2, decltype(ksp)::value>, T>(x, w, y, stats, d, s, bn);
        return launch_tap<TapCfg<kTapTM, decltype(tn)::value, decltype(ksp)::value>, T>(x, w, y, stats, d, s, bn);
    };
    auto waves = [&](auto tn) {
        switch (tap_waves(d.Ci)) {
            case 1: return run(tn, std::integral_constant<int, 1>{});
            case 2: return run(tn, std::integral_constant<int, 2>{});
            case 4: return run(tn, std::integral_constant<int, 4>{});
            default: return run(tn, std::integral_constant<int, 8>{});
        }
    };
    switch (tap_positions(d)) {
        case 4: return waves(std::integral_constant<int, 4>{});
        case 2: return waves(std::integral_constant<int, 2>{});
        default: return waves(std::integral_constant<int, 1>{});
    }
}
template int launch_fwd_tap<float>(const float *, const float *, float *, double *, const ConvDims &, hipStream_t, const BnEval &);
template int launch_fwd_tap<bf16_t>(const bf16_t *, const float *, bf16_t *, double *, const ConvDims &, hipStream_t, const BnEval &);

}  // namespace adder

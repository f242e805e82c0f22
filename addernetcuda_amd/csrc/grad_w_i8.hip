// Weight gradient of large 3x3 / pad 1, 5x5 / pad 2 and 1x1 layers of stride 1 in bfloat16 storage, on the 8-bit matrix cores.  (First the kernel
// of the 3x3 and 5x5 layers, then that of the single taps.)
//
//   gw[co,ci,i,j] = sum_pos x[ci, pos + (i,j)] * gy[co,pos]  -  w[co,ci,i,j] * sum_pos gy[co,pos]
//
// The sum over positions needs more than fp32 (see grad_w_mfma.hip), and v_mfma_f64_16x16x4_f64 gives it at 16 multiply-adds a
// cycle and SIMD.  v_mfma_i32_16x16x64_i8 does 1000, exactly, so the operands are written in fixed point, four signed 8-bit digits
// each, and thirteen digit products (of the sixteen: the three left out lie below the last digit) stand for one fp64 product:
//   x = 2^ex * sum_d X_d 2^-8d,   gy = 2^eg * sum_d G_d 2^-8d,   x * gy = 2^(ex+eg) * sum_{s<5} 2^-8s sum_{d+e=s} X_d G_e.
// The scales 2^ex, 2^eg belong to one channel of one staged tile (256 positions of gy, those and the halo of x), so the fixed point is
// relative to the largest of these values: 32 bits, which hold the eight bits of every value down to 2^-22 of it.  The digit sums of a tile are
// exact in 32 bits (at most four products of 2^14, 256 positions) and go into fp64 sums with their scales; gy is added up in fp64 as it is.  Where values
// were rounded that matter, and where one is infinite or not a number, the workgroup goes through its tiles again with the values
// and fp64 products ("whether the digits will do", below).  Error of the raw gradient against float64 on the tensors of a ResNet-20 training
// step, 2-norm, worst layer: 2.591e-8, all of it the rounding to float, where the fp64 kernels have 2.591e-8; no layer is gone through again.
// (Not for float storage: its 24 bits are exact down to 2^-6 of the largest only, and half of a training step's gradients lie below 2^-10.  Without
// a rule the same layers' error was 2.89e-8 for 2.59e-8, and wrong altogether where large values met zeros; with a rule that holds it, ordinary
// steps were gone through again: VGG-small 8.0 -> 11 ms, with the fp64 kernels 9.8.)
//
// Layout: a tile is four images x 64 positions.  Its LDS cells are dwords of one digit of four images, so that a
// lane's sixteen 8-bit operands -- four adjacent columns x four images -- are four cells of a row, and a tap's shift moves whole
// cells: j shifts by register, i by row.  MFMA rows are output channels, columns are input channels; a wave owns one tap
// row of a 16 x 16 channel block, i.e. KS accumulator tiles x five digit weights.
//
// Half of a workgroup's waves multiply, the other half load, find the largest values and write digits, a tile ahead: the conversion is
// eight vector instructions a value, as much time as the matrix instructions it feeds, and on other waves it runs beside them.
// What bounds it: the issue of both kinds' instructions, which hardly overlap (per tile and SIMD, 128 -> 128 @32x32: 3700 cycles of matrix
// instructions and 6600 of vector ones, 10 200 measured).  128 -> 128 @32x32, 128 images: fp64 737 us, this 253 (the passes again with values: 1110 in all);
// 64 -> 64 @56x56, 32 images 170 -> 70; 512 -> 512 @8x8, 128 images 830 -> 283.
#include "common.hpp"

#include <type_traits>

namespace adder {

typedef int int4v __attribute__((ext_vector_type(4)));

template <int KS_, int TH_, int TW_, int MB_, int NB_, int PW_, int LWAVES_, int MINWAVES_>
struct GwI8Cfg {
    static constexpr int KS = KS_, KK = KS_ * KS_, PAD = KS_ / 2, TH = TH_, TW = TW_, MB = MB_, NB = NB_, MINWAVES = MINWAVES_;
    static constexpr int COB = 16 * MB, CIB = 16 * NB;
    // A tile's rows fall into strips of eight columns; a step of the multiplying waves takes four strips, one per 16 lanes.
    static constexpr int STRIPS = TW / 8, PW = PW_, STEPS = TH * STRIPS / 4 / PW;   // PW waves share a tile's steps
    static constexpr int MWAVES = KS * MB * NB * PW, LWAVES = LWAVES_;      // multiplying and loading waves
    static constexpr int NTHREADS = 64 * (MWAVES + LWAVES), LTHREADS = 64 * LWAVES;
    static constexpr int QW = TW / 4;                          // groups of four columns per row
    // x cells: [channel][digit][row][column] with the halo columns of the rows behind them, [row][2 PAD]; gy cells alike.  Channels start
    // four banks apart (16-byte reads of eight channels meet 32 banks).
    static constexpr int XR = TH + KS - 1, HC = 2 * PAD, XH = XR * TW, XDIG = XH + XR * HC, XPLANE = round_up(4 * XDIG, 32) + 4;
    static constexpr int GDIG = TH * TW, GPLANE = 4 * GDIG + 4;
    static constexpr int XUNITS = CIB * XR * QW, HUNITS = CIB * XR * HC, GUNITS = COB * TH * QW;
    static constexpr int XITER = ceil_div(XUNITS, LTHREADS), HITER = ceil_div(HUNITS, LTHREADS), GITER = ceil_div(GUNITS, LTHREADS);
    static constexpr int G0 = CIB * XPLANE;                    // a tile's x cells, then its gy cells
    static constexpr int TILE_WORDS = G0 + COB * GPLANE;
    static constexpr int OUT = COB * CIB * KK;                 // results, folded and reordered through LDS at the end (fp64)
    static constexpr int CH = COB + CIB;                       // largest-value slots: gy channels, then x channels
    static constexpr int MX0 = 2 * TILE_WORDS, SM0 = MX0 + 4 * CH, FLAG0 = SM0 + 4 * CH;
    // the error sums of the multiplying waves' results lie in LDS: beside the accumulators they would not stay in registers
    static constexpr int ERR0 = FLAG0 + 4, COEF0 = ERR0 + 64 * MWAVES * 8;
    static constexpr int LDS_BYTES = COEF0 * 4;
    static_assert(TW % 8 == 0 && 4 % STRIPS == 0 && TH * STRIPS % (4 * PW) == 0 && KS % 2 == 1, "whole steps of four strips");
    static_assert((XR * QW) % 4 == 0 && (XR * HC) % 4 == 0 && (TH * QW) % 4 == 0, "four units in a row share a channel");
    static_assert(LDS_BYTES <= 160 * 1024 && NTHREADS <= 1024, "workgroup limits");
    static_assert(2 * (OUT + GUNITS) <= 2 * TILE_WORDS, "the results fit the cells' place");
    static_assert(XDIG % 4 == 0 && XH % 4 == 0 && GPLANE % 4 == 0 && COEF0 % 4 == 0, "16-byte alignment of the cells");
};

// Four images of a tensor as a buffer: loads from beyond its end (images that do not exist) or at kNowhere give zeros, so they need no
// branch -- with loads under way in two register sets, a wait has to know how many are newer.
typedef unsigned uint4v __attribute__((ext_vector_type(4)));
typedef unsigned uint2v __attribute__((ext_vector_type(2)));
static constexpr unsigned kNowhere = 0x80000000u;
static constexpr int kBufferImage = 1 << 27;   // elements per image: four fill 2^30 bytes, and kNowhere + three does not wrap
__device__ __forceinline__ __amdgpu_buffer_rsrc_t i8_images(const bf16_t *base, int image, int n0, int N) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(base + (size_t)n0 * image), 0, min(4, N - n0) * image * (int)sizeof(bf16_t), 0x00020000);
}
__device__ __forceinline__ float i8_load1(__amdgpu_buffer_rsrc_t r, unsigned off) { return bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0)); }
// four consecutive elements of a row, `left` elements before its end (VEC: rows are whole groups of four)
template <bool VEC>
__device__ __forceinline__ float4 i8_load4(__amdgpu_buffer_rsrc_t r, unsigned off, int left) {
    if constexpr (!VEC) {
        constexpr unsigned E = sizeof(bf16_t);
        return make_float4(i8_load1(r, off), i8_load1(r, left > 1 ? off + E : kNowhere), i8_load1(r, left > 2 ? off + 2 * E : kNowhere),
                           i8_load1(r, left > 3 ? off + 3 * E : kNowhere));
    } else {
        const uint2v u = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
        return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                           __uint_as_float(u.y & 0xffff0000u));
    }
}

// the larger magnitude, as bits (NaN and infinity come out above every number)
__device__ __forceinline__ float i8_absmax(float m, float a, float b) {
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(a), fabsf(b)), m);
}
__device__ __forceinline__ float i8_absmax4(float m, const float4 &v) { return i8_absmax(i8_absmax(m, v.x, v.y), v.z, v.w); }

// A channel's exponent from the bits of its largest magnitude: magnitudes from 1.96875 up count as the next power of two,
// so that |v| 2^(30-e) < 2^31 - 2^24 and the first digit stays within +-127 (the last three carry into it).  255: not finite (or within
// 1.6 % of the largest float).  Below 2^-97 the last digit stays at 2^-127, which 2^127 still reaches.
__device__ __forceinline__ int i8_exponent(unsigned m) { return max((int)((m + 0x40000u) >> 23), 30); }
__device__ __forceinline__ double i8_unit(int e) { return __hiloint2double((e - 127 - 30 + 1023) << 20, 0); }   // 2^(e - 127 - 30): the last digit's
__device__ __forceinline__ float i8_scale(int e) { return __uint_as_float((unsigned)(30 + 127 + 127 - e) << 23); }   // its reciprocal, 2^(30 - (e - 127))

// largest magnitude of the four lanes of a quad into its channel's slot
__device__ __forceinline__ void i8_note_max(float m, unsigned *slot, int *flag, bool ok) {
    unsigned u = __float_as_uint(m) & 0x7fffffffu;
    u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
    u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
    if (ok && (threadIdx.x & 3) == 0) {
        atomicMax(slot, u);
        if (i8_exponent(u) >= 255) *flag = 1;
    }
}
// sum over the four lanes of a quad into its channel's slot
__device__ __forceinline__ void i8_note_sum(int u, int *slot) {
    if (__builtin_amdgcn_ballot_w64(u) == 0) return;
    u += __builtin_amdgcn_update_dpp(0, u, 0xB1, 0xF, 0xF, true);
    u += __builtin_amdgcn_update_dpp(0, u, 0x4E, 0xF, 0xF, true);
    if ((threadIdx.x & 3) == 0 && u) atomicAdd(slot, u);
}

// v times a power of two, to the nearest integer; off: the largest distance from it so far.  (v_cvt_rpi_i32_f32 would do both steps, but rounds odd
// results above 2^23 away.)
__device__ __forceinline__ unsigned i8_round(float v, float scale, float &off) {
    const float t = v * scale, r = rintf(t);
    off = fmaxf(off, fabsf(t - r));
    return (unsigned)(int)r;
}
// how many of four values were rounded
__device__ __forceinline__ int i8_count(float a, float b, float c, float d, float scale) {
    auto one = [&](const float v) { return v * scale != rintf(v * scale) ? 1 : 0; };
    return (one(a) + one(b)) + (one(c) + one(d));
}
// four values (one column of four images) as four cells, one per digit.  Adding 0x808080 turns the lower three digits into unsigned
// ones with carries, the exclusive-or makes them signed again.
__device__ __forceinline__ void i8_digits(float a, float b, float c, float d, float scale, int (&cell)[4], float &off) {
    const unsigned u0 = i8_round(a, scale, off) + 0x808080u, u1 = i8_round(b, scale, off) + 0x808080u,
                   u2 = i8_round(c, scale, off) + 0x808080u, u3 = i8_round(d, scale, off) + 0x808080u;
    const unsigned lo01 = __builtin_amdgcn_perm(u1, u0, 0x05010400u), hi01 = __builtin_amdgcn_perm(u1, u0, 0x07030602u);
    const unsigned lo23 = __builtin_amdgcn_perm(u3, u2, 0x05010400u), hi23 = __builtin_amdgcn_perm(u3, u2, 0x07030602u);
    cell[0] = (int)__builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
    cell[1] = (int)(__builtin_amdgcn_perm(hi23, hi01, 0x05040100u) ^ 0x80808080u);
    cell[2] = (int)(__builtin_amdgcn_perm(lo23, lo01, 0x07060302u) ^ 0x80808080u);
    cell[3] = (int)(__builtin_amdgcn_perm(lo23, lo01, 0x05040100u) ^ 0x80808080u);
}

// a unit of four columns x four images into the cells at p (p + digit * pitch); RAW: the values themselves, image k in the
// place of digit k.  Gives how many were rounded.
template <bool RAW>
__device__ __forceinline__ int i8_put4(const float4 (&v)[4], float scale, int *p, int pitch) {
    int rounded = 0;
    if constexpr (!RAW) {
        float off = 0.f;
        int c0[4], c1[4], c2[4], c3[4];
        i8_digits(v[0].x, v[1].x, v[2].x, v[3].x, scale, c0, off);
        i8_digits(v[0].y, v[1].y, v[2].y, v[3].y, scale, c1, off);
        i8_digits(v[0].z, v[1].z, v[2].z, v[3].z, scale, c2, off);
        i8_digits(v[0].w, v[1].w, v[2].w, v[3].w, scale, c3, off);
#pragma unroll
        for (int k = 0; k < 4; ++k) *reinterpret_cast<int4v *>(p + k * pitch) = int4v{c0[k], c1[k], c2[k], c3[k]};
        if (__builtin_amdgcn_ballot_w64(off > 0.f))   // (seldom)
            rounded = (i8_count(v[0].x, v[1].x, v[2].x, v[3].x, scale) + i8_count(v[0].y, v[1].y, v[2].y, v[3].y, scale)) +
                      (i8_count(v[0].z, v[1].z, v[2].z, v[3].z, scale) + i8_count(v[0].w, v[1].w, v[2].w, v[3].w, scale));
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) *reinterpret_cast<float4 *>(p + k * pitch) = v[k];
    }
    return rounded;
}

// The digit sums of one result (a[s]: digit weights 2^-8s) in units of the third, in fp64: first digits lie within +-127, the others
// within +-128, a tile has at most 256 positions, so the sums stay within 2^24 and the first two fit one 32-bit number.
__device__ __forceinline__ double i8_product(int a0, int a1, int a2, int a3, int a4) {
    return fma((double)(((a3 & 255) << 8) + a4), 0x1p-16, fma((double)((a0 << 8) + a1), 256.0, (double)(a2 + (a3 >> 8))));
}

// ---- whether the digits will do ----
// A bfloat16 value has eight significant bits, so the fixed point holds it exactly down to 2^-22 of its channel's largest in the tile; the products left
// out are those of two digits below 2^-16.  What can go wrong is a tile whose largest values meet nothing but zeros, so that the sum consists of
// values far below them.  In units of the two channels' first digits (X = |x| / 2^(ex-6) < 126, G alike) the square of a tile's error is, on the average
// over roundings, at most 2^-50 / 3 of  126^2 * the number of values that were rounded  (+ kLeftOut for the products left out).  A lane adds that up over all
// tiles for its results, and at the end the block's rows and columns are looked at one by one: where the errors' sum of squares is above 2^-48 of the
// results', the workgroup works its block out again in fp64.  (126 is the most a partner can have; it has a quarter of that on the average.)
static constexpr int kRounded = 126 * 126, kLeftOut = 42;
static constexpr double kFine = 3 * 0x1p-30;   // 3 * 2^50 * 2^-48, and scales count in the third digit, 2^16 a product less
__device__ __forceinline__ bool i8_fine(double errors, double results) { return errors <= kFine * results; }

// sum over the sixteen lanes of a row of a wave (in registers: forty sums through LDS would be 3 us of a small layer's 16)
__device__ __forceinline__ double i8_row_sum(double v) {
    auto from = [&](auto ctrl) __attribute__((always_inline)) {
        return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), decltype(ctrl)::value, 0xF, 0xF, true),
                                __builtin_amdgcn_update_dpp(0, __double2loint(v), decltype(ctrl)::value, 0xF, 0xF, true));
    };
    v += from(std::integral_constant<int, 0xB1>{});    // quad_perm [1,0,3,2]
    v += from(std::integral_constant<int, 0x4E>{});    // quad_perm [2,3,0,1]
    v += from(std::integral_constant<int, 0x141>{});   // row_half_mirror
    v += from(std::integral_constant<int, 0x140>{});   // row_mirror
    return v;
}

typedef double double4v __attribute__((ext_vector_type(4)));
// The row of 16 that lane l of a wave gives v_mfma_f64_16x16x4_f64, so that the results, rows 4 e + l / 16 there, lie like those of the 8-bit
// ones, rows 4 (l / 16) + e.
__device__ __forceinline__ int i8_fp64_row(int l16) { return 4 * (l16 & 3) + (l16 >> 2); }

template <class G, bool VEC>
__global__ __launch_bounds__(G::NTHREADS, G::MINWAVES) void grad_w_i8_kernel(const bf16_t *__restrict__ gy, const bf16_t *__restrict__ x,
                                                                double *__restrict__ part, double *__restrict__ sgpart, int N,
                                                                int Ci, int H, int W, int Co, int tilesH, int tilesW, int ntiles) {
    constexpr int KS = G::KS, PAD = G::PAD, QW = G::QW, SQ = 2;   // SQ: groups of four columns in a strip
    extern __shared__ __align__(16) int cells[];   // two tiles: x cells, gy cells
    unsigned *const mx = reinterpret_cast<unsigned *>(cells + G::MX0);   // the channels' largest magnitudes in four tiles,
    int *const sm = cells + G::SM0;   // how many of their values were rounded
    int *const flag = cells + G::FLAG0;   // the digits will not do

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, lk = lane >> 4;
    const bool loader = wave >= G::MWAVES;
    const int lt = tid - 64 * G::MWAVES;   // loader thread
    // a multiplying wave's accumulators (tap row, block of 16 output channels, of 16 input channels) and its share of a tile's steps
    const int ti = wave % KS, pw = wave / KS % G::PW, mb = wave / KS / G::PW % G::MB, nb = wave / KS / G::PW / G::MB;
    const int co_blk = blockIdx.y * G::COB, ci_blk = blockIdx.z * G::CIB;
    // the workgroup's tiles lie side by side: the lines that neighbouring tiles share stay in one L2
    const int each = (ntiles + (int)gridDim.x - 1) / (int)gridDim.x, mine = min(each, ntiles - (int)blockIdx.x * each);
    int tile0 = blockIdx.x * each;

    for (int e = tid; e < G::FLAG0 + 1 - G::MX0; e += G::NTHREADS) mx[e] = 0;
    __syncthreads();

    // ---- the loading waves ----
    // A thread's units: channel, row and column within the tile, offset from the tile's first position, place among the cells.
    const int ximg = Ci * H * W, gimg = Co * H * W;
    int gch[G::GITER], grow[G::GITER], gcol[G::GITER], xch[G::XITER], xrow[G::XITER], xcol[G::XITER], hch[G::HITER], hrow[G::HITER], hcol[G::HITER];
#pragma unroll
    for (int it = 0; it < G::GITER; ++it) {
        const int u = lt + it * G::LTHREADS;
        gcol[it] = u % QW * 4; grow[it] = u / QW % G::TH; gch[it] = u / QW / G::TH;
    }
#pragma unroll
    for (int it = 0; it < G::XITER; ++it) {
        const int u = lt + it * G::LTHREADS;
        xcol[it] = u % QW * 4; xrow[it] = u / QW % G::XR; xch[it] = u / QW / G::XR;
    }
#pragma unroll
    for (int it = 0; it < G::HITER; ++it) {
        const int u = lt + it * G::LTHREADS;
        hcol[it] = u % G::HC; hrow[it] = u / G::HC % G::XR; hch[it] = u / G::HC / G::XR;
    }
    // Two tiles under way in registers; one, where a thread has two gy units: the multiplying waves last longer than a load there, and
    // a second set would spill (and a wait for a spilled address is a wait for all loads: 48 -> 48 5x5 @28x28, 8 images, 33 us with two, 26 with one).
    constexpr int SETS = G::GITER > 1 ? 1 : 2;
    float4 xv[SETS][G::XITER][4], gv[SETS][G::GITER][4];
    float hv[SETS][G::HITER][4];
    double sgt[G::GITER];   // sums of the gy units' values
    auto place = [&](const int i, int &n0, int &h0, int &w0) {
        int t = tile0 + i;
        const int tw = t % tilesW; t /= tilesW;
        const int th = t % tilesH; t /= tilesH;
        n0 = t * 4; h0 = th * G::TH; w0 = tw * G::TW;
    };
    // (Always inlined: a call would put the registers it captures into memory.)
    // tile i of the workgroup (nothing, if it has none) into register set b
    auto fetch = [&](const int i, auto set) __attribute__((always_inline)) {
        constexpr int b = decltype(set)::value;
        constexpr unsigned E = sizeof(bf16_t);
        int n0, h0, w0;
        place(min(i, mine - 1), n0, h0, w0);
        const auto gbuf = i8_images(gy, gimg, n0, N), xbuf = i8_images(x, ximg, n0, N);
#pragma unroll
        for (int it = 0; it < G::GITER; ++it) {
            const int ch = co_blk + gch[it], ho = h0 + grow[it], wo = w0 + gcol[it];
            const bool ok = i < mine && (G::GUNITS % G::LTHREADS == 0 || gch[it] < G::COB) && ch < Co && ho < H && wo < W;
            const unsigned off = ok ? ((ch * H + ho) * W + wo) * E : kNowhere;
#pragma unroll
            for (int k = 0; k < 4; ++k) gv[b][it][k] = i8_load4<VEC>(gbuf, off + k * gimg * E, W - wo);
        }
#pragma unroll
        for (int it = 0; it < G::XITER; ++it) {
            const int ch = ci_blk + xch[it], hi = h0 - PAD + xrow[it], wi = w0 + xcol[it];
            const bool ok = i < mine && (G::XUNITS % G::LTHREADS == 0 || xch[it] < G::CIB) && ch < Ci && hi >= 0 && hi < H && wi < W;
            const unsigned off = ok ? ((ch * H + hi) * W + wi) * E : kNowhere;
#pragma unroll
            for (int k = 0; k < 4; ++k) xv[b][it][k] = i8_load4<VEC>(xbuf, off + k * ximg * E, W - wi);
        }
#pragma unroll
        for (int it = 0; it < G::HITER; ++it) {
            const int ch = ci_blk + hch[it], hi = h0 - PAD + hrow[it], wi = w0 + (hcol[it] < PAD ? hcol[it] - PAD : G::TW + hcol[it] - PAD);
            const bool ok = i < mine && (G::HUNITS % G::LTHREADS == 0 || hch[it] < G::CIB) && ch < Ci && hi >= 0 && hi < H && wi >= 0 && wi < W;
            const unsigned off = ok ? ((ch * H + hi) * W + wi) * E : kNowhere;
#pragma unroll
            for (int k = 0; k < 4; ++k) hv[b][it][k] = i8_load1(xbuf, off + k * ximg * E);
        }
    };
    // the largest magnitudes of the channels of tile i, which is in set b
    auto note = [&](const int i, auto set) __attribute__((always_inline)) {
        constexpr int b = decltype(set)::value;
        unsigned *const mxs = mx + (i & 3) * G::CH;
        if (blockIdx.z == 0) {
#pragma unroll
            for (int it = 0; it < G::GITER; ++it)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    sgt[it] += ((double)gv[b][it][k].x + (double)gv[b][it][k].y) + ((double)gv[b][it][k].z + (double)gv[b][it][k].w);
        }
#pragma unroll
        for (int it = 0; it < G::GITER; ++it) {
            const bool ok = G::GUNITS % G::LTHREADS == 0 || gch[it] < G::COB;
            float m = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) m = i8_absmax4(m, gv[b][it][k]);
            i8_note_max(m, mxs + (ok ? gch[it] : 0), flag, ok);
        }
#pragma unroll
        for (int it = 0; it < G::XITER; ++it) {
            const bool ok = G::XUNITS % G::LTHREADS == 0 || xch[it] < G::CIB;
            float m = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) m = i8_absmax4(m, xv[b][it][k]);
            i8_note_max(m, mxs + G::COB + (ok ? xch[it] : 0), flag, ok);
        }
#pragma unroll
        for (int it = 0; it < G::HITER; ++it) {
            const bool ok = G::HUNITS % G::LTHREADS == 0 || hch[it] < G::CIB;
            const float m = i8_absmax(i8_absmax(0.f, hv[b][it][0], hv[b][it][1]), hv[b][it][2], hv[b][it][3]);
            i8_note_max(m, mxs + G::COB + (ok ? hch[it] : 0), flag, ok);
        }
    };
    // set b into the cells of tile i
    auto commit = [&](const int i, auto set, auto with_values) __attribute__((always_inline)) {
        constexpr int b = decltype(set)::value;
        constexpr bool RAW = decltype(with_values)::value;
        int *const tile = cells + (i & 1) * G::TILE_WORDS;
        const unsigned *const mxs = mx + (i & 3) * G::CH;
        int *const sms = sm + (i & 3) * G::CH;
#pragma unroll
        for (int it = 0; it < G::GITER; ++it)
            if (G::GUNITS % G::LTHREADS == 0 || gch[it] < G::COB) {
                const int rounded = i8_put4<RAW>(gv[b][it], i8_scale(i8_exponent(mxs[gch[it]])),
                                                 tile + G::G0 + gch[it] * G::GPLANE + grow[it] * G::TW + gcol[it], G::GDIG);
                if constexpr (!RAW) i8_note_sum(rounded, sms + gch[it]);
            }
#pragma unroll
        for (int it = 0; it < G::XITER; ++it)
            if (G::XUNITS % G::LTHREADS == 0 || xch[it] < G::CIB) {
                const int rounded = i8_put4<RAW>(xv[b][it], i8_scale(i8_exponent(mxs[G::COB + xch[it]])),
                                                 tile + xch[it] * G::XPLANE + xrow[it] * G::TW + xcol[it], G::XDIG);
                if constexpr (!RAW) i8_note_sum(rounded, sms + G::COB + xch[it]);
            }
#pragma unroll
        for (int it = 0; it < G::HITER; ++it)
            if (G::HUNITS % G::LTHREADS == 0 || hch[it] < G::CIB) {
                int cell[4];
                if constexpr (!RAW) {
                    const float (&v)[4] = hv[b][it], scale = i8_scale(i8_exponent(mxs[G::COB + hch[it]]));
                    float off = 0.f;
                    i8_digits(v[0], v[1], v[2], v[3], scale, cell, off);
                    i8_note_sum(i8_count(v[0], v[1], v[2], v[3], scale), sms + G::COB + hch[it]);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) cell[k] = __float_as_int(hv[b][it][k]);
                }
                int *p = tile + hch[it] * G::XPLANE + G::XH + hrow[it] * G::HC + hcol[it];
#pragma unroll
                for (int k = 0; k < 4; ++k) p[k * G::XDIG] = cell[k];
            }
    };

    // ---- the multiplying waves ----
    // tot[j][e]: row 4 * lk + e (output channel), column l16 (input channel), tap (ti, j)
    // The wave's operands: lane group lk takes strip lk of a step's four.  The cells before and after a strip are its neighbours' or,
    // at the ends of a row, the halo's.  (Steps are whole rows apart, 4 / STRIPS of them.)
    constexpr int ROWS = 4 / G::STRIPS;
    const int strip = lk % G::STRIPS, lrow = pw * G::STEPS * ROWS + lk / G::STRIPS;
    const int goff = G::G0 + (mb * 16 + l16) * G::GPLANE + lrow * G::TW + 8 * strip;
    const int xch0 = (nb * 16 + l16) * G::XPLANE, xoff = xch0 + (lrow + ti) * G::TW + 8 * strip, xhalo = xch0 + G::XH + (lrow + ti) * G::HC;
    const bool first = strip == 0, last = strip == G::STRIPS - 1;
    const int loff = first ? xhalo : xoff - PAD, roff = last ? xhalo + PAD : xoff + 8;
    const int lstep = ROWS * (first ? G::HC : G::TW), rstep = ROWS * (last ? G::HC : G::TW);
    double2 *const errs = reinterpret_cast<double2 *>(cells + G::ERR0) + wave * 128 + lane;   // of rows e = 0, 1 and 64 further on of 2, 3
    // tile i at row h0: into tot, and the squares of the errors into errs
    auto multiply = [&](const int i, const int h0, double4v (&tot)[KS]) __attribute__((always_inline)) {
        const int *const tile = cells + (i & 1) * G::TILE_WORDS, *const sms = sm + (i & 3) * G::CH;
        const unsigned *const mxs = mx + (i & 3) * G::CH;
        int4v acc[KS][5];
#pragma unroll
        for (int j = 0; j < KS; ++j)
#pragma unroll
            for (int s = 0; s < 5; ++s) acc[j][s] = int4v{0, 0, 0, 0};
        // The x cells of one digit and step are a phase: KS matrix instructions per digit of gy that goes with it.  The next phase's cells
        // are asked for before a phase's instructions, a step's last gy digits (which the last phase does not need) with them.
        int4v a[SQ][4], mid[2][SQ];
        int edge[2][2 * PAD];
        auto ask_a = [&](const int rs, const int d) {
#pragma unroll
            for (int q = 0; q < SQ; ++q) a[q][d] = *reinterpret_cast<const int4v *>(tile + goff + rs * ROWS * G::TW + d * G::GDIG + 4 * q);
        };
        auto ask_x = [&](const int p) {
            const int rs = p / 4, dx = p % 4;
#pragma unroll
            for (int q = 0; q < SQ; ++q) mid[p & 1][q] = *reinterpret_cast<const int4v *>(tile + xoff + rs * ROWS * G::TW + dx * G::XDIG + 4 * q);
#pragma unroll
            for (int e = 0; e < PAD; ++e) {
                edge[p & 1][e] = tile[loff + rs * lstep + dx * G::XDIG + e];
                edge[p & 1][PAD + e] = tile[roff + rs * rstep + dx * G::XDIG + e];
            }
        };
        ask_x(0);
        ask_a(0, 3);
        ask_a(0, 2);
#pragma unroll
        for (int p = 0; p < 4 * G::STEPS; ++p) {
            const int dx = p % 4;
            if (dx == 0) { ask_a(p / 4, 1); ask_a(p / 4, 0); }
            int win[8 + 2 * PAD];   // tap j of column c of the strip meets cell c + j
#pragma unroll
            for (int e = 0; e < PAD; ++e) { win[e] = edge[p & 1][e]; win[PAD + 8 + e] = edge[p & 1][PAD + e]; }
#pragma unroll
            for (int q = 0; q < SQ; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) win[PAD + 4 * q + e] = mid[p & 1][q][e];
            if (p + 1 < 4 * G::STEPS) ask_x(p + 1);
            if (dx == 3 && p + 1 < 4 * G::STEPS) { ask_a(p / 4 + 1, 3); ask_a(p / 4 + 1, 2); }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < SQ; ++q) {
                int4v b[KS];
#pragma unroll
                for (int j = 0; j < KS; ++j) b[j] = int4v{win[4 * q + j], win[4 * q + j + 1], win[4 * q + j + 2], win[4 * q + j + 3]};
#pragma unroll
                for (int dg = dx == 0 ? 3 : 4 - dx; dg >= 0; --dg)
#pragma unroll
                    for (int j = 0; j < KS; ++j)
                        acc[j][dx + dg] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[q][dg], b[j], acc[j][dx + dg], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const unsigned xm = mxs[G::COB + nb * 16 + l16];
        const int xs = kRounded * sms[G::COB + nb * 16 + l16] + kLeftOut;
        const uint4v gm = *reinterpret_cast<const uint4v *>(mxs + mb * 16 + 4 * lk);
        const int4v gs = *reinterpret_cast<const int4v *>(sms + mb * 16 + 4 * lk);
        const double sx = xm ? i8_unit(i8_exponent(xm)) * 4294967296.0 : 0.0;   // (i8_product counts in 2^32)
        double err[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const double sc = gm[e] ? sx * i8_unit(i8_exponent(gm[e])) : 0.0;
            err[e] = (sc * sc) * (double)(kRounded * gs[e] + xs);
#pragma unroll
            for (int j = 0; j < KS; ++j)
                tot[j][e] = fma(i8_product(acc[j][0][e], acc[j][1][e], acc[j][2][e], acc[j][3][e], acc[j][4][e]), sc, tot[j][e]);
        }
        // (a tap row that lies outside the image throughout the tile has no products)
        if (max(h0, PAD - ti) < min(h0 + G::TH, min(H, H + PAD - ti))) {
            const double2 a = errs[0], b = errs[64];
            errs[0] = make_double2(a.x + err[0], a.y + err[1]);
            errs[64] = make_double2(b.x + err[2], b.y + err[3]);
        }
    };
    // a tile's values instead of digits: fp64, four images at a time; positions outside the tensor do not count (zero times infinity)
    auto multiply_raw = [&](const int i, double4v (&tot)[KS]) __attribute__((always_inline)) {
        int n0, h0, w0;
        place(i, n0, h0, w0);
        const int *const tile = cells + (i & 1) * G::TILE_WORDS;
        constexpr int RROWS = G::TH / G::PW;
        const int gch0 = G::G0 + (mb * 16 + i8_fp64_row(l16)) * G::GPLANE + lk * G::GDIG;
#pragma unroll 1
        for (int r = pw * RROWS; r < min((pw + 1) * RROWS, H - h0); ++r) {
            const int xr = xch0 + lk * G::XDIG + (r + ti) * G::TW, hr = xch0 + lk * G::XDIG + G::XH + (r + ti) * G::HC;   // the row's cells and its halo's
#pragma unroll 1
            for (int c = 0; c < min(G::TW, W - w0); c += 4) {
                const float4 g = *reinterpret_cast<const float4 *>(tile + gch0 + r * G::TW + c);
                const float4 x = *reinterpret_cast<const float4 *>(tile + xr + c);
                float win[4 + 2 * PAD];
#pragma unroll
                for (int e = 0; e < PAD; ++e) {
                    win[e] = __int_as_float(tile[(c ? xr + c - PAD : hr) + e]);
                    win[PAD + 4 + e] = __int_as_float(tile[(c + 4 < G::TW ? xr + c + 4 : hr + PAD) + e]);
                }
                win[PAD] = x.x; win[PAD + 1] = x.y; win[PAD + 2] = x.z; win[PAD + 3] = x.w;
                const float gs[4] = {g.x, g.y, g.z, g.w};
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (w0 + c + u < W) {
#pragma unroll
                        for (int j = 0; j < KS; ++j) tot[j] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)gs[u], (double)win[u + j], tot[j], 0, 0, 0);
                    }
            }
        }
    };

    // While the multiplying waves work on tile i, the loading ones write the cells of tile i + 1, ask for tile i + 3 and note the
    // largest values of tile i + 2, which has arrived meanwhile: one barrier a tile.  (Each kind of wave runs a loop of its own,
    // with the same barriers, so that neither kind's registers are kept for the other's.)  Should the digits not do, both go through the tiles once more.
    double *const out = reinterpret_cast<double *>(cells), *const sgs = out + G::OUT;
    auto again = [&]() __attribute__((always_inline)) {
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(*flag) == 0) return false;
        __syncthreads();
        for (int e = tid; e < G::FLAG0 - G::MX0; e += G::NTHREADS) mx[e] = 0;
        __syncthreads();
        return true;
    };
    if (loader) {
        constexpr std::integral_constant<int, 0> even{};
        constexpr std::integral_constant<int, SETS - 1> odd{};
        auto pass = [&](auto with_values) __attribute__((always_inline)) {
            asm volatile("" : "+s"(tile0));   // (no offset of the first pass is kept in a register for the second)
#pragma unroll
            for (int it = 0; it < G::GITER; ++it) sgt[it] = 0.0;
            fetch(0, even);
            if (SETS == 2) fetch(1, odd);
            note(0, even);
            __syncthreads();
            commit(0, even, with_values);
            fetch(SETS, even);
            note(1, odd);
            __syncthreads();
            auto turn = [&](const int i, auto next, auto after) __attribute__((always_inline)) {   // the sets that hold tiles i + 1 and i + 2
                // (addresses in LDS are made from these in every turn: kept, they would not all stay in registers, and a wait for one from memory
                // is a wait for the loads under way)
#pragma unroll
                for (int it = 0; it < G::GITER; ++it) asm volatile("" : "+v"(gch[it]));
#pragma unroll
                for (int it = 0; it < G::XITER; ++it) asm volatile("" : "+v"(xch[it]));
#pragma unroll
                for (int it = 0; it < G::HITER; ++it) asm volatile("" : "+v"(hch[it]));
                if (i + 1 < mine) commit(i + 1, next, with_values);
                for (int e = lt; e < G::CH; e += G::LTHREADS) mx[((i + 3) & 3) * G::CH + e] = sm[((i + 3) & 3) * G::CH + e] = 0;
                fetch(i + 1 + SETS, next);
                if (i + 2 < mine) note(i + 2, after);
                __syncthreads();
            };
            for (int i = 0; i < mine; i += 2) {   // (always both: a wait for one set must not have to allow for the turn left out)
                turn(i, odd, even);
                turn(i + 1, even, odd);
            }
        };
        pass(std::false_type{});
        if (again()) {
            pass(std::true_type{});
            __syncthreads();
        }
        if (blockIdx.z == 0) {
#pragma unroll
            for (int it = 0; it < G::GITER; ++it)
                if (G::GUNITS % G::LTHREADS == 0 || gch[it] < G::COB) sgs[lt + it * G::LTHREADS] = sgt[it];
        }
        for (int p = 0; p < G::PW; ++p) __syncthreads();
    } else {
        double4v tot[KS];
#pragma unroll
        for (int j = 0; j < KS; ++j) tot[j] = double4v{0.0, 0.0, 0.0, 0.0};
        errs[0] = errs[64] = make_double2(0.0, 0.0);
        __syncthreads();
        __syncthreads();
        int n0, h0, w0;
        place(0, n0, h0, w0);
        for (int i = 0; i < mine; ++i) {
            multiply(i, h0, tot);
            if ((w0 += G::TW) >= tilesW * G::TW) {
                w0 = 0;
                if ((h0 += G::TH) >= tilesH * G::TH) h0 = 0;
            }
            __syncthreads();
        }
        if (mine & 1) __syncthreads();
        // a wave's rows and columns of KS taps
        const double err[4] = {errs[0].x, errs[0].y, errs[64].x, errs[64].y};
        double col_err = 0.0, col_res = 0.0;
        bool fine = true;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const double row_err = KS * err[e];
            double row_res = 0.0;
#pragma unroll
            for (int j = 0; j < KS; ++j) row_res = fma(tot[j][e], tot[j][e], row_res);
            col_err += row_err;
            col_res += row_res;
            fine = fine && i8_fine(i8_row_sum(row_err), i8_row_sum(row_res));
        }
#pragma unroll
        for (int d = 16; d < 64; d <<= 1) {
            col_err += __shfl_xor(col_err, d, 64);
            col_res += __shfl_xor(col_res, d, 64);
        }
        if (!fine || !i8_fine(col_err, col_res)) *flag = 1;
        if (again()) {
#pragma unroll
            for (int j = 0; j < KS; ++j) tot[j] = double4v{0.0, 0.0, 0.0, 0.0};
            __syncthreads();
            __syncthreads();
            for (int i = 0; i < mine; ++i) {
                multiply_raw(i, tot);
                __syncthreads();
            }
            if (mine & 1) __syncthreads();
            __syncthreads();
        }
        // ---- fold the waves that shared a tile's steps and put the block in the order of the slab, through LDS ----
        for (int p = 0; p < G::PW; ++p) {
            if (pw == p) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    double *o = out + ((mb * 16 + 4 * lk + e) * G::CIB + nb * 16 + l16) * G::KK + ti * KS;
#pragma unroll
                    for (int j = 0; j < KS; ++j) o[j] = p == 0 ? tot[j][e] : o[j] + tot[j][e];
                }
            }
            __syncthreads();
        }
    }
    if (blockIdx.z == 0 && tid < min(G::COB, Co - co_blk)) {   // a channel's sums of gy are those of TH * QW units in a row
        double sum = 0.0;
        for (int u = 0; u < G::TH * QW; ++u) sum += sgs[tid * (G::TH * QW) + u];
        sgpart[(size_t)blockIdx.x * Co + co_blk + tid] = sum;
    }
    const int K = Ci * G::KK, kcols = min(G::CIB, Ci - ci_blk) * G::KK;
    double *dst = part + ((size_t)blockIdx.x * Co + co_blk) * K + (size_t)ci_blk * G::KK;
    for (int c = 0; c < min(G::COB, Co - co_blk); ++c)
        for (int k = tid; k < kcols; k += G::NTHREADS) dst[(size_t)c * K + k] = out[c * (G::CIB * G::KK) + k];
}

// ---------------------------------------------------------------------------
// Single taps: gw[co,ci] = sum_pos x[ci,pos] gy[co,pos] over the positions of all planes in a row (so planes of any size fill the
// tiles).  The same fixed point and digits.  A tile is 128 positions; the four digits that share a cell are 32 positions apart, so that
// a thread's four loads are each part of a line that eight threads read, and those eight threads hold a channel's tile: its largest
// value needs no exchange with other waves, and a thread converts a unit as soon as it has arrived and asks for the same unit of
// the next tile.  Each multiplying wave owns 16 MT x 16 NT results.
// ---------------------------------------------------------------------------
template <int MT_, int NT_, int MB_, int NB_, int LWAVES_, int MINWAVES_>
struct GwI8RowCfg {
    static constexpr int MT = MT_, NT = NT_, MB = MB_, NB = NB_, LWAVES = LWAVES_, MINWAVES = MINWAVES_, TP = 128;
    static constexpr int COB = 16 * MT * MB, CIB = 16 * NT * NB, ROWS = COB + CIB;
    static constexpr int MWAVES = MB * NB, NTHREADS = 64 * (MWAVES + LWAVES), LTHREADS = 64 * LWAVES;
    static constexpr int CELLS = TP / 4, PLANE = 4 * CELLS + 4;      // cells per digit, per channel (channels start four banks apart)
    static constexpr int UNITS = ROWS * 8, ITER = ceil_div(UNITS, LTHREADS), STEPS = TP / 64;
    static constexpr int TILE_WORDS = ROWS * PLANE, EX0 = 2 * TILE_WORDS;
    static constexpr int SM0 = EX0 + 2 * ROWS, FLAG0 = SM0 + 2 * ROWS;
    static constexpr int ERR0 = round_up(FLAG0 + 1, 4), LDS_BYTES = (ERR0 + 64 * MWAVES * NT * 8) * 4;   // (a wave's first row of tiles has its error sums in LDS)
    static_assert(LDS_BYTES <= 160 * 1024 && NTHREADS <= 1024 && LTHREADS % 8 == 0, "workgroup limits");
};

// P = N * L positions of N images with planes of L; VEC: planes are whole groups of four.  x and gy: (N, Ci, L) and (N, Co, L).
template <class G, bool VEC>
__global__ __launch_bounds__(G::NTHREADS, G::MINWAVES) void grad_w_i8_row_kernel(const bf16_t *__restrict__ gy, const bf16_t *__restrict__ x,
                                                                    double *__restrict__ part, double *__restrict__ sgpart, int N,
                                                                    int Ci, int Co, int L, int ntiles) {
    constexpr int MT = G::MT, NT = G::NT;
    constexpr unsigned E = sizeof(bf16_t);
    extern __shared__ __align__(16) int cells[];
    // the channels' exponents in two tiles (0: nothing but zeros), how many of their values were rounded; whether the digits will not do
    int *const ex = cells + G::EX0, *const sm = cells + G::SM0, *const flag = cells + G::FLAG0;

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, lk = lane >> 4;
    const int co_blk = blockIdx.y * G::COB, ci_blk = blockIdx.z * G::CIB;
    const long P = (long)N * L;
    const int each = (ntiles + (int)gridDim.x - 1) / (int)gridDim.x, mine = min(each, ntiles - (int)blockIdx.x * each);
    int tile0 = blockIdx.x * each;
    const double rL = 1.0 / L;
    // image and place in its plane of position p
    auto place = [&](const long p, int &n, int &l) __attribute__((always_inline)) {
        n = (int)((double)p * rL);
        l = (int)(p - (long)n * L);
        if (l < 0) { l += L; --n; }
        if (l >= L) { l -= L; ++n; }
    };
    if (tid == 0) *flag = 0;
    __syncthreads();

    const int mb = wave % G::MB, nb = wave / G::MB % G::NB;
    auto again = [&]() __attribute__((always_inline)) {
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(*flag) == 0) return false;
        __syncthreads();
        return true;
    };
    if (wave >= G::MWAVES) {
        // ---- the loading waves: unit u = thread's channel row0 + it * (LTHREADS / 8), columns 4 * (u % 8) .. + 3 of each 32 ----
        const int lt = tid - 64 * G::MWAVES, col = 4 * (lt & 7), row0 = lt >> 3;
        float4 v[G::ITER][4];
        constexpr int GITER = ceil_div(G::COB, G::LTHREADS / 8);   // its units from here on are of x
        double sgt[GITER];   // sums of the gy rows' values
        // Offsets (bytes) of the thread's four groups from the first image of the tile that is being asked for, and of its channels; those
        // that do not exist push the sum beyond every buffer, which ends below 2^31.
        constexpr unsigned NO_GROUP = 0x80000000u, NO_ROW = 0x7fffffffu;
        unsigned xoff[4], goff[4], rowoff[G::ITER];
        int l[4], left[4], nlo = 0;
        const int wrow0 = __builtin_amdgcn_readfirstlane(row0 & ~7);   // (a wave's eight rows are of one tensor)
#pragma unroll
        for (int it = 0; it < G::ITER; ++it) {
            const int row = row0 + it * (G::LTHREADS / 8);
            const bool is_x = row >= G::COB, ok = row < G::ROWS && (is_x ? ci_blk + row - G::COB < Ci : co_blk + row < Co);
            rowoff[it] = ok ? (unsigned)((is_x ? ci_blk + row - G::COB : co_blk + row) * L) * E : NO_ROW;
        }
        auto aim = [&](const int i) __attribute__((always_inline)) {
            const long base = (long)(tile0 + i) * G::TP;
            int n, l0;
            place(min(base, P - 1), nlo, l0);
            nlo = __builtin_amdgcn_readfirstlane(nlo);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const long p = base + col + 32 * k;
                place(p, n, l[k]);
                left[k] = i < mine ? (int)max(min(P - p, 4L), 0L) : 0;
                xoff[k] = left[k] ? (unsigned)((n - nlo) * Ci * L + l[k]) * E : NO_GROUP;
                goff[k] = left[k] ? (unsigned)((n - nlo) * Co * L + l[k]) * E : NO_GROUP;
            }
        };
        auto ask = [&](const int it) __attribute__((always_inline)) {
            const bool is_x = wrow0 + it * (G::LTHREADS / 8) >= G::COB;
            const int C = is_x ? Ci : Co;
            auto one = [&](const bf16_t *t, float4 (&dst)[4]) __attribute__((always_inline)) {
                const long rest = ((long)N - nlo) * C * L * (long)E;
                const auto buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(t + (size_t)nlo * C * L), 0,
                                                                   (int)(rest < 0x7fffffffL ? rest : 0x7fffffffL), 0x00020000);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const unsigned off = (is_x ? xoff[k] : goff[k]) + rowoff[it];
                    if constexpr (VEC) {
                        dst[k] = i8_load4<true>(buf, off, 4);
                    } else {   // a group may run on into the next image's plane
                        float q[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            q[e] = i8_load1(buf, e < left[k] ? off + e * E + (l[k] + e >= L ? (unsigned)(C - 1) * L * E : 0u) : kNowhere);
                        dst[k] = make_float4(q[0], q[1], q[2], q[3]);
                    }
                }
            };
            one(is_x ? x : gy, v[it]);
        };
        static_assert(G::COB % 8 == 0, "eight rows of a wave are of one tensor");
        auto turn = [&](const int i, auto with_values) __attribute__((always_inline)) {   // writes tile i, asks for tile i + 1
            int *const tile = cells + (i & 1) * G::TILE_WORDS;
            aim(i + 1);
#pragma unroll
            for (int it = 0; it < G::ITER; ++it) {
                const int row = row0 + it * (G::LTHREADS / 8);
                const bool ok = G::UNITS % G::LTHREADS == 0 || row < G::ROWS;
                float m = 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k) m = i8_absmax4(m, v[it][k]);
                unsigned u = __float_as_uint(m) & 0x7fffffffu;   // over the eight lanes of the channel
                u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
                u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x4E, 0xF, 0xF, true));    // quad_perm [2,3,0,1]
                u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x141, 0xF, 0xF, true));   // row_half_mirror
                const int e = i8_exponent(u);
                if (it < GITER && blockIdx.z == 0 && wrow0 + it * (G::LTHREADS / 8) < G::COB) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) sgt[it] += ((double)v[it][k].x + (double)v[it][k].y) + ((double)v[it][k].z + (double)v[it][k].w);
                }
                if (ok) {
                    int rounded = i8_put4<decltype(with_values)::value>(v[it], i8_scale(min(e, 254)), tile + row * G::PLANE + col, G::CELLS);
                    if (__builtin_amdgcn_ballot_w64(rounded)) {   // over the eight lanes of the channel
                        rounded += __builtin_amdgcn_update_dpp(0, rounded, 0xB1, 0xF, 0xF, true);
                        rounded += __builtin_amdgcn_update_dpp(0, rounded, 0x4E, 0xF, 0xF, true);
                        rounded += __builtin_amdgcn_update_dpp(0, rounded, 0x141, 0xF, 0xF, true);
                    }
                    if ((lt & 7) == 0) {
                        ex[(i & 1) * G::ROWS + row] = u ? e : 0;
                        sm[(i & 1) * G::ROWS + row] = rounded;
                        if (e >= 255) *flag = 1;
                    }
                }
                ask(it);
            }
        };
        auto pass = [&](auto with_values) __attribute__((always_inline)) {
            asm volatile("" : "+s"(tile0));   // (no offset of the first pass is kept in a register for the second)
#pragma unroll
            for (int it = 0; it < GITER; ++it) sgt[it] = 0.0;
            aim(0);
#pragma unroll
            for (int it = 0; it < G::ITER; ++it) ask(it);
            turn(0, with_values);
            __syncthreads();
            for (int i = 0; i < mine; ++i) {
                if (i + 1 < mine) turn(i + 1, with_values);
                __syncthreads();
            }
        };
        pass(std::false_type{});
        if (again()) {
            pass(std::true_type{});
            __syncthreads();
        }
        if (blockIdx.z == 0) {
#pragma unroll
            for (int it = 0; it < GITER; ++it) {
                const int row = row0 + it * (G::LTHREADS / 8);
                double sum = sgt[it];   // over the eight lanes of the channel
#pragma unroll
                for (int d = 1; d < 8; d <<= 1) sum += __shfl_xor(sum, d, 64);
                if ((lt & 7) == 0 && row < G::COB && co_blk + row < Co) sgpart[(size_t)blockIdx.x * Co + co_blk + row] = sum;
            }
        }
    } else {
        // ---- the multiplying waves ----
        const int goff = (mb * MT * 16 + l16) * G::PLANE + 4 * lk, xoff = (G::COB + nb * NT * 16 + l16) * G::PLANE + 4 * lk;
        double4v tot[MT][NT], err[MT][NT];   // results and the squares of their errors (as in the kernel above; those of m = 0 in LDS)
        double2 *const errs = reinterpret_cast<double2 *>(cells + G::ERR0) + wave * (128 * NT) + lane;
        auto multiply = [&](const int i) __attribute__((always_inline)) {
            const int *const tile = cells + (i & 1) * G::TILE_WORDS, *const exs = ex + (i & 1) * G::ROWS, *const sms = sm + (i & 1) * G::ROWS;
            int4v acc[MT][NT][5], a[MT][4], b[2][NT];
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int s = 0; s < 5; ++s) acc[m][n][s] = int4v{0, 0, 0, 0};
            auto ask_a = [&](const int st, const int d) {
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    a[m][d] = *reinterpret_cast<const int4v *>(tile + goff + m * 16 * G::PLANE + d * G::CELLS + 16 * st);
            };
            auto ask_b = [&](const int p) {
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    b[p & 1][n] = *reinterpret_cast<const int4v *>(tile + xoff + n * 16 * G::PLANE + p % 4 * G::CELLS + 16 * (p / 4));
            };
            ask_b(0);
            ask_a(0, 3);
            ask_a(0, 2);
#pragma unroll
            for (int p = 0; p < 4 * G::STEPS; ++p) {   // (phases as in the kernel above)
                const int dx = p % 4;
                if (dx == 0) { ask_a(p / 4, 1); ask_a(p / 4, 0); }
                if (p + 1 < 4 * G::STEPS) ask_b(p + 1);
                if (dx == 3 && p + 1 < 4 * G::STEPS) { ask_a(p / 4 + 1, 3); ask_a(p / 4 + 1, 2); }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int dg = dx == 0 ? 3 : 4 - dx; dg >= 0; --dg)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
#pragma unroll
                        for (int n = 0; n < NT; ++n)
                            acc[m][n][dx + dg] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[m][dg], b[p & 1][n], acc[m][n][dx + dg], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            double sx[NT];
            int xs[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const int xe = exs[G::COB + (nb * NT + n) * 16 + l16];
                sx[n] = xe ? i8_unit(xe) * 4294967296.0 : 0.0;
                xs[n] = kRounded * sms[G::COB + (nb * NT + n) * 16 + l16] + kLeftOut;
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int4v ge = *reinterpret_cast<const int4v *>(exs + (mb * MT + m) * 16 + 4 * lk),
                            gs = *reinterpret_cast<const int4v *>(sms + (mb * MT + m) * 16 + 4 * lk);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const double sg = ge[e] ? i8_unit(ge[e]) : 0.0;
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
                        const double sc = sx[n] * sg;
                        tot[m][n][e] = fma(i8_product(acc[m][n][0][e], acc[m][n][1][e], acc[m][n][2][e], acc[m][n][3][e], acc[m][n][4][e]),
                                           sc, tot[m][n][e]);
                        const double more = (sc * sc) * (double)(kRounded * gs[e] + xs[n]);
                        if (m == 0) {
                            double *const at = reinterpret_cast<double *>(errs + 64 * (2 * n + e / 2)) + e % 2;
                            *at += more;
                        } else {
                            err[m][n][e] += more;
                        }
                    }
                }
            }
        };
        auto multiply_raw = [&](const int i) __attribute__((always_inline)) {   // a tile's values instead of digits: fp64, positions 32 apart four at a time
            const int *const tile = cells + (i & 1) * G::TILE_WORDS + lk * G::CELLS;
            const int goff = (mb * MT * 16 + i8_fp64_row(l16)) * G::PLANE, xoff = (G::COB + nb * NT * 16 + l16) * G::PLANE;
#pragma unroll 1
            for (int c = 0; c < G::CELLS; c += 4) {
                float4 g[MT];
#pragma unroll
                for (int m = 0; m < MT; ++m) g[m] = *reinterpret_cast<const float4 *>(tile + goff + m * 16 * G::PLANE + c);
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    const float4 x = *reinterpret_cast<const float4 *>(tile + xoff + n * 16 * G::PLANE + c);
                    const float xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                    for (int m = 0; m < MT; ++m) {
                        const float gs[4] = {g[m].x, g[m].y, g[m].z, g[m].w};
#pragma unroll
                        for (int u = 0; u < 4; ++u) tot[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)gs[u], (double)xs[u], tot[m][n], 0, 0, 0);
                    }
                }
            }
        };
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                tot[m][n] = err[m][n] = double4v{0.0, 0.0, 0.0, 0.0};
                if (m == 0) errs[128 * n] = errs[128 * n + 64] = make_double2(0.0, 0.0);
            }
        __syncthreads();
        for (int i = 0; i < mine; ++i) {
            multiply(i);
            __syncthreads();
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const double2 a = errs[128 * n], b = errs[128 * n + 64];
            err[0][n] = double4v{a.x, a.y, b.x, b.y};
        }
        bool fine = true;
        double col_err[NT] = {}, col_res[NT] = {};
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                double row_err = 0.0, row_res = 0.0;
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    const double r2 = tot[m][n][e] * tot[m][n][e];
                    row_err += err[m][n][e];
                    row_res += r2;
                    col_err[n] += err[m][n][e];
                    col_res[n] += r2;
                }
                fine = fine && i8_fine(i8_row_sum(row_err), i8_row_sum(row_res));
            }
#pragma unroll
        for (int n = 0; n < NT; ++n) {
#pragma unroll
            for (int d = 16; d < 64; d <<= 1) {
                col_err[n] += __shfl_xor(col_err[n], d, 64);
                col_res[n] += __shfl_xor(col_res[n], d, 64);
            }
            fine = fine && i8_fine(col_err[n], col_res[n]);
        }
        if (!fine) *flag = 1;
        if (again()) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n) tot[m][n] = double4v{0.0, 0.0, 0.0, 0.0};
            __syncthreads();
            for (int i = 0; i < mine; ++i) {
                multiply_raw(i);
                __syncthreads();
            }
            __syncthreads();
        }
        // ---- straight to the slab: sixteen lanes hold sixteen columns in a row ----
        double *dst = part + (size_t)blockIdx.x * Co * Ci;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int co = co_blk + (mb * MT + m) * 16 + 4 * lk + e;
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    const int ci = ci_blk + (nb * NT + n) * 16 + l16;
                    if (co < Co && ci < Ci) dst[(size_t)co * Ci + ci] = tot[m][n][e];
                }
            }
        }
    }
}

// ---- host side ------------------------------------------------------------------
// Channel blocks of 16 x 16 (two waves per tap row) and 32 x 16, tiles of 2 x 32, 4 x 16 and 8 x 8 positions of four images.
//                       KS TH TW MB NB PW loading waves, waves per SIMD
using Gi3a32 = GwI8Cfg<3, 2, 32, 1, 1, 2, 6, 3>;
using Gi3a16 = GwI8Cfg<3, 4, 16, 1, 1, 2, 6, 3>;
using Gi3a8  = GwI8Cfg<3, 8, 8, 1, 1, 2, 6, 3>;
using Gi3b16 = GwI8Cfg<3, 4, 16, 2, 1, 1, 6, 3>;
using Gi3b8  = GwI8Cfg<3, 8, 8, 2, 1, 1, 6, 3>;
using Gi5w32 = GwI8Cfg<5, 2, 32, 1, 1, 1, 3, 2>;
using Gi5w16 = GwI8Cfg<5, 4, 16, 1, 1, 1, 3, 2>;
using Gi5w8  = GwI8Cfg<5, 8, 8, 1, 1, 1, 3, 2>;

// Single taps: 64 x 64 and, for few output channels, 32 x 96, each of 16 (14) waves on a CU of its own.  Whole calls with their
// finalizing and scaling kernels, fp64 matrix cores -> this: 128 -> 512 @28x28, 32 images 98 -> 55 us, 128 -> 128 @28x28, 16 images 33 -> 18.
// Bound by the issue of both kinds of waves together (1024 -> 256 @14x14, 64 images, of 82 us the multiplying waves alone took 59, the loading
// waves alone 60, and without their loads both 80).
//                           MT NT MB NB loading waves, waves per SIMD
using GiRow  = GwI8RowCfg<2, 1, 2, 4, 8, 4>;
using GiRowN = GwI8RowCfg<2, 1, 1, 6, 8, 4>;

template <class G, bool VEC>
static int launch_i8_row_v(const bf16_t *gy, const bf16_t *x, double *part, double *sgpart, const ConvDims &d, const GradWMfmaPlan &p, hipStream_t s) {
    if (int rc = allow_dynamic_lds<&grad_w_i8_row_kernel<G, VEC>>(G::LDS_BYTES)) return rc;
    hipLaunchKernelGGL((grad_w_i8_row_kernel<G, VEC>), dim3(p.slots, p.gy, p.gz), dim3(G::NTHREADS), G::LDS_BYTES, s, gy, x, part, sgpart, d.N, d.Ci, d.Co,
                       d.H * d.W, p.ntiles);
    return check_launch();
}

template <class G>
static int launch_i8_row(const bf16_t *gy, const bf16_t *x, double *part, double *sgpart, const ConvDims &d, const GradWMfmaPlan &p, hipStream_t s) {
    return d.H * d.W % 4 == 0 && aligned_groups(x) && aligned_groups(gy) ? launch_i8_row_v<G, true>(gy, x, part, sgpart, d, p, s)
                                                                        : launch_i8_row_v<G, false>(gy, x, part, sgpart, d, p, s);
}

template <class G>
static void plan_i8_row(int N, int Ci, int Co, int L, GradWMfmaPlan &p) {
    p.ntiles = (int)ceil_div_l((long)N * L, G::TP);
    p.gy = ceil_div(Co, G::COB);
    p.gz = ceil_div(Ci, G::CIB);
    p.slots = plan_grad_w_slots(p.gy * p.gz, p.ntiles, sizeof(double) * ((size_t)Co * Ci + Co));
}

template <class G, bool VEC>
static int launch_i8_v(const bf16_t *gy, const bf16_t *x, double *part, double *sgpart, const ConvDims &d, const GradWMfmaPlan &p, hipStream_t s) {
    if (int rc = allow_dynamic_lds<&grad_w_i8_kernel<G, VEC>>(G::LDS_BYTES)) return rc;
    hipLaunchKernelGGL((grad_w_i8_kernel<G, VEC>), dim3(p.slots, p.gy, p.gz), dim3(G::NTHREADS), G::LDS_BYTES, s, gy, x, part, sgpart, d.N, d.Ci, d.H, d.W,
                       d.Co, p.tilesH, p.tilesW, p.ntiles);
    return check_launch();
}

template <class G>
static int launch_i8(const bf16_t *gy, const bf16_t *x, double *part, double *sgpart, const ConvDims &d, const GradWMfmaPlan &p, hipStream_t s) {
    return d.W % 4 == 0 ? launch_i8_v<G, true>(gy, x, part, sgpart, d, p, s) : launch_i8_v<G, false>(gy, x, part, sgpart, d, p, s);
}

template <class G>
static void plan_i8(const ConvDims &d, GradWMfmaPlan &p) {
    p.tilesH = ceil_div(d.H, G::TH);
    p.tilesW = ceil_div(d.W, G::TW);
    p.ntiles = ceil_div(d.N, 4) * p.tilesH * p.tilesW;
    p.gy = ceil_div(d.Co, G::COB);
    p.gz = ceil_div(d.Ci, G::CIB);
    p.slots = plan_grad_w_slots(p.gy * p.gz, p.ntiles, sizeof(double) * ((size_t)d.Co * d.Ci * G::KK + d.Co));
}

static bool plan_i8_rows(const ConvDims &d, GradWMfmaPlan &p) {
    const long L = (long)d.H * d.W;
    if (L < 4 || (128 + 2 * L) * (d.Ci > d.Co ? d.Ci : d.Co) > 2L * kBufferImage || d.N * L > 1L << 30) return false;   // 32-bit offsets from a tile's first image
    p.variant = d.Co > 32 ? 32 : 33;
    if (p.variant == 32) plan_i8_row<GiRow>(d.N, d.Ci, d.Co, (int)L, p);
    else plan_i8_row<GiRowN>(d.N, d.Ci, d.Co, (int)L, p);
    return true;
}

// Whether it takes a layer.  Against the fp64 matrix kernel it has some more to set up (half a workgroup's waves load, digits, four
// images at a time), 2-3 us, and a fifth to a half of the matrix time; us, other kernel -> this, bfloat16:
//   3x3, multiply-adds with the channels filled up to 16: 2.26e8 (6 images) 20.1 -> 20.8, 2.39e8 (5 images) 31.1 -> 23.4 and 25.4 -> 21.5, 2.6e8 (9 images)
//   25.6 -> 22.3, 2.65e8 (7, 8 images) 20.7 -> 20.8 and 21.7 -> 22.5, 2.7e8 38.1 -> 28.5, 3e8 21.8 -> 20.3, 5.8e8 (5 images) 36.6 -> 31.2;
//   5x5: maps wider than 8, 4e6 24.9 -> 21.0 to 2.6e9 147 -> 59 (the fp64 kernel's 25-tap blocks start late); 8x8, 1.5e8 and up;
//   1x1, from 64 channels on both sides: 64 -> 64 @2x2, 64 images 14.5 -> 11.1, @8x8, 16 images 14.4 -> 11.4, 2048 -> 512 @14x14, 1 image 34.9 -> 25.4;
//   fewer channels, planes of whole groups of four: 160 -> 48 @28x28, 64 images (3.9e8) 32.5 -> 26.5; other planes, which the plain kernel reads element by
//   element: 8 -> 8 @15x15, 64 images 27.8 -> 15.1, 16 -> 64 25.7 -> 15.1, 24 -> 512 @25x25, 16 images 34.9 -> 25.3, 1024 -> 16 @15x15, 64 images 86 -> 33.
// Three channels on wide maps have a block of 32 columns there (stem).  Fewer than four images would leave digits empty.
bool plan_grad_w_i8(const ConvDims &d, GradWMfmaPlan &p) {
    if (d.stride != 1 || d.kh != d.kw || d.pad != d.kh / 2) return false;
    if (d.kh == 1) {
        // (the layers below 64 channels have a plain kernel beside this one, which reads planes that are not whole groups of four
        // element by element; a block of fewer than 32 channels wastes more than the digits give)
        const long L = (long)d.H * d.W;
        const double macs = (double)round_up(d.Ci, 16) * round_up(d.Co, 16) * d.N * L;
        if (!(d.Ci >= 64 && d.Co >= 64) && !(L % 4 && d.N * L >= 3000) && !(d.Ci >= 32 && d.Co >= 32 && macs >= 2.2e8)) return false;
        return plan_i8_rows(d, p);
    }
    if (d.N < 4 || (d.kh != 3 && d.kh != 5)) return false;
    if ((long)d.Ci * d.H * d.W > kBufferImage || (long)d.Co * d.H * d.W > kBufferImage) return false;
    if (d.kh == 3 && d.Ci * 9 <= 32 && d.W > 16) return false;
    const double macs = (double)round_up(d.Ci, 16) * round_up(d.Co, 16) * d.kh * d.kw * d.N * d.H * d.W;
    if (macs < (d.kh == 3 ? 2.3e8 : d.W > 8 ? 0.0 : 1.5e8)) return false;
    // the tile that needs fewest; rows in one piece load whole lines and no halo columns, which is worth a seventh
    const int n32 = ceil_div(d.H, 2) * ceil_div(d.W, 32), n16 = ceil_div(d.H, 4) * ceil_div(d.W, 16), n8 = ceil_div(d.H, 8) * ceil_div(d.W, 8);
    const int shape = 7 * n32 <= 7 * n16 && 7 * n32 <= 8 * n8 ? 0 : 7 * n16 <= 8 * n8 ? 1 : 2;
    if (d.kh == 3) {
        p.variant = (d.Co > 16 ? 24 : 20) + shape;
        switch (p.variant) {
            case 20: plan_i8<Gi3a32>(d, p); break;
            case 21: plan_i8<Gi3a16>(d, p); break;
            case 22: plan_i8<Gi3a8>(d, p); break;
            case 24: case 25: plan_i8<Gi3b16>(d, p); break;
            default: plan_i8<Gi3b8>(d, p); break;
        }
        return true;
    }
    p.variant = 28 + shape;
    if (shape == 0) plan_i8<Gi5w32>(d, p);
    else if (shape == 1) plan_i8<Gi5w16>(d, p);
    else plan_i8<Gi5w8>(d, p);
    return true;
}

int launch_grad_w_i8(const bf16_t *gy, const bf16_t *x, double *part, double *sgpart, const ConvDims &d, const GradWMfmaPlan &p, hipStream_t s) {
    switch (p.variant) {
        case 20: return launch_i8<Gi3a32>(gy, x, part, sgpart, d, p, s);
        case 21: return launch_i8<Gi3a16>(gy, x, part, sgpart, d, p, s);
        case 22: return launch_i8<Gi3a8>(gy, x, part, sgpart, d, p, s);
        case 24: case 25: return launch_i8<Gi3b16>(gy, x, part, sgpart, d, p, s);
        case 26: return launch_i8<Gi3b8>(gy, x, part, sgpart, d, p, s);
        case 28: return launch_i8<Gi5w32>(gy, x, part, sgpart, d, p, s);
        case 29: return launch_i8<Gi5w16>(gy, x, part, sgpart, d, p, s);
        case 30: return launch_i8<Gi5w8>(gy, x, part, sgpart, d, p, s);
        case 32: return launch_i8_row<GiRow>(gy, x, part, sgpart, d, p, s);
        case 33: return launch_i8_row<GiRowN>(gy, x, part, sgpart, d, p, s);
        default: return ADDER_ERR_BAD_SHAPE;
    }
}

}  // namespace adder

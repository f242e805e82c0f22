// Shared device/host helpers for the gfx950 AdderNet kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/addernet_hip.h"

namespace adder {

// Wave-uniform read-only data (weights) is fetched through the scalar cache:
// a load from the constant address space with a uniform address becomes
// s_load_dword*, and the value is then used directly as the SGPR operand of the
// vector subtract, so weights cost neither VGPRs nor LDS bandwidth.
typedef const __attribute__((address_space(4))) float *uniform_f32_ptr;

__device__ __forceinline__ uniform_f32_ptr as_uniform(const float *p) {
    return (uniform_f32_ptr)p;
}

// Touch `rows` runs of `len` floats, `pitch` floats apart, with one vector load per 128-byte line, so that
// the scalar weight loads of a kernel's main loop -- which run only one unit ahead and would otherwise wait
// for HBM on every new line, all workgroups at the same place -- find their lines in L2.
__device__ __forceinline__ void l2_warm(const float *p, int rows, int pitch, int len) {
    const int lines = (len + 31) / 32;
    for (int i = threadIdx.x; i < rows * lines; i += blockDim.x) {
        const int r = i / lines, l = i - r * lines;
        const float v = p[(size_t)r * pitch + min(l * 32, len - 1)];
        asm volatile("" ::"v"(v));
    }
}

// Storage types of activations: float, or bfloat16 (the upper half of a float, round to nearest even on the way
// out) for the optional reduced-storage mode; arithmetic is fp32 (fp64 for the weight gradient) either way.
typedef uint16_t bf16_t;
__device__ __forceinline__ float bf16_to_f32(bf16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);   // round to nearest, ties to even (NaN payloads are not preserved)
    return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float ldf(const float *p) { return *p; }
__device__ __forceinline__ float ldf(const bf16_t *p) { return bf16_to_f32(*p); }
__device__ __forceinline__ void stf(float *p, float v) { *p = v; }
__device__ __forceinline__ void stf(bf16_t *p, float v) { *p = f32_to_bf16(v); }
// four / two consecutive elements at an address aligned to their total size
__device__ __forceinline__ float4 ldf4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ float4 ldf4(const bf16_t *p) {
    const uint2 u = *reinterpret_cast<const uint2 *>(p);
    return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                       __uint_as_float(u.y & 0xffff0000u));
}
__device__ __forceinline__ void stf4(float *p, float4 v) { *reinterpret_cast<float4 *>(p) = v; }
__device__ __forceinline__ void stf4(bf16_t *p, float4 v) {
    uint2 u;
    u.x = (uint32_t)f32_to_bf16(v.x) | ((uint32_t)f32_to_bf16(v.y) << 16);
    u.y = (uint32_t)f32_to_bf16(v.z) | ((uint32_t)f32_to_bf16(v.w) << 16);
    *reinterpret_cast<uint2 *>(p) = u;
}
__device__ __forceinline__ float2 ldf2(const float *p) { return *reinterpret_cast<const float2 *>(p); }
__device__ __forceinline__ float2 ldf2(const bf16_t *p) {
    const uint32_t u = *reinterpret_cast<const uint32_t *>(p);
    return make_float2(__uint_as_float(u << 16), __uint_as_float(u & 0xffff0000u));
}
__device__ __forceinline__ void stf2(float *p, float2 v) { *reinterpret_cast<float2 *>(p) = v; }
__device__ __forceinline__ void stf2(bf16_t *p, float2 v) {
    *reinterpret_cast<uint32_t *>(p) = (uint32_t)f32_to_bf16(v.x) | ((uint32_t)f32_to_bf16(v.y) << 16);
}

// CNT consecutive elements at an address aligned to one element only (global memory takes loads and stores of any alignment).
typedef float f32x2_any __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t u16x2_any __attribute__((ext_vector_type(2), aligned(2)));
typedef uint16_t u16x4_any __attribute__((ext_vector_type(4), aligned(2)));
template <int CNT>
__device__ __forceinline__ void ld_strip(const float *p, float (&v)[CNT]) {
    static_assert(CNT == 1 || CNT == 2 || CNT == 4, "one, two or four elements");
    if constexpr (CNT == 4) {
        const f32x4_any u = *reinterpret_cast<const f32x4_any *>(p);
        v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
    } else if constexpr (CNT == 2) {
        const f32x2_any u = *reinterpret_cast<const f32x2_any *>(p);
        v[0] = u.x; v[1] = u.y;
    } else {
        v[0] = *p;
    }
}
template <int CNT>
__device__ __forceinline__ void ld_strip(const bf16_t *p, float (&v)[CNT]) {
    static_assert(CNT == 1 || CNT == 2 || CNT == 4, "one, two or four elements");
    if constexpr (CNT == 4) {
        const u16x4_any u = *reinterpret_cast<const u16x4_any *>(p);
        v[0] = bf16_to_f32(u.x); v[1] = bf16_to_f32(u.y); v[2] = bf16_to_f32(u.z); v[3] = bf16_to_f32(u.w);
    } else if constexpr (CNT == 2) {
        const u16x2_any u = *reinterpret_cast<const u16x2_any *>(p);
        v[0] = bf16_to_f32(u.x); v[1] = bf16_to_f32(u.y);
    } else {
        v[0] = ldf(p);
    }
}
template <int CNT>
__device__ __forceinline__ void st_strip(float *p, const float (&v)[CNT]) {
    static_assert(CNT == 2 || CNT == 4, "two or four elements");
    if constexpr (CNT == 4) *reinterpret_cast<f32x4_any *>(p) = f32x4_any{v[0], v[1], v[2], v[3]};
    else *reinterpret_cast<f32x2_any *>(p) = f32x2_any{v[0], v[1]};
}
template <int CNT>
__device__ __forceinline__ void st_strip(bf16_t *p, const float (&v)[CNT]) {
    static_assert(CNT == 2 || CNT == 4, "two or four elements");
    if constexpr (CNT == 4)
        *reinterpret_cast<u16x4_any *>(p) = u16x4_any{f32_to_bf16(v[0]), f32_to_bf16(v[1]), f32_to_bf16(v[2]), f32_to_bf16(v[3])};
    else
        *reinterpret_cast<u16x2_any *>(p) = u16x2_any{f32_to_bf16(v[0]), f32_to_bf16(v[1])};
}

// A lane's 32-bit byte offset from a uniform base, used in a loop: without this the compiler widens it to 64 bits in front of the loop and
// adds base and offset in vector registers at every load; with it the load takes both as they are.
__device__ __forceinline__ void keep_offset(unsigned &off) { asm volatile("" : "+v"(off)); }

static constexpr int kTapChunk = 16;   // output channels that a wave of grad_x_tap.hip takes at a time
static constexpr int kNineChunk = 8;   // ... of grad_x_nine.hip and grad_x_s2.hip: at most 72 terms

// Workgroup number -> (tile, block) of a launch whose blocks read the same tile of x.  Workgroups go to the eight dies in turn, each
// with its own L2: the blocks of one tile follow each other on one die, so that x crosses to it once.
__device__ __forceinline__ void xcd_tile(unsigned id, int tiles, int blocks, int &tile, int &blk) {
    const unsigned whole = (unsigned)(tiles & ~7);
    if (id < whole * blocks) {
        const unsigned j = id >> 3;
        tile = (int)(j / blocks * 8 + (id & 7));
        blk = (int)(j % blocks);
    } else {
        const unsigned r = id - whole * blocks, rem = (unsigned)tiles - whole;
        tile = (int)(whole + r % rem);
        blk = (int)(r / rem);
    }
}

// Most workgroups along a grid's y (hipDeviceProp_t::maxGridSize: 65536).  Kernels with few channels per workgroup leave layers
// with more channels than that to those with many.
static constexpr int kMaxGridY = 65535;

// Whether a tensor's base lets four consecutive elements be moved as one group (NULL: no tensor).
template <class T>
inline bool aligned_groups(const T *p) { return (reinterpret_cast<uintptr_t>(p) & (4 * sizeof(T) - 1)) == 0; }

// Clamp to [0, 1]: the compiler folds it into the clamp output modifier of the instruction that
// produces v, so it costs no instruction of its own.
__device__ __forceinline__ float sat01(float v) { return __builtin_amdgcn_fmed3f(v, 0.f, 1.f); }

// hardtanh of adder.cu:17 (x<-1 -> -1, x<=1 -> x, else 1) is one v_med3_f32.
__device__ __forceinline__ float hardtanh(float v) {
    return __builtin_amdgcn_fmed3f(v, -1.0f, 1.0f);
}

// Kernels with more than 48 KB of dynamic LDS need hipFuncAttributeMaxDynamicSharedMemorySize, once per device
// (the attribute belongs to the device's copy of the function).  One flag word per kernel instantiation.
int record_hip_error(hipError_t e);
template <auto Kernel>
inline int allow_dynamic_lds(int bytes) {
    static unsigned long long done = 0;   // bit d: set on device d (benign race: setting it twice is harmless)
    if (bytes <= 48 * 1024) return 0;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return record_hip_error(e);
    if (dev >= 0 && dev < 64 && ((done >> dev) & 1ull)) return 0;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return record_hip_error(e);
    if (dev >= 0 && dev < 64) done |= 1ull << dev;
    return 0;
}

__host__ __device__ constexpr int ceil_div(int a, int b) { return (a + b - 1) / b; }
__host__ __device__ constexpr long ceil_div_l(long a, long b) { return (a + b - 1) / b; }
__host__ __device__ constexpr int round_up(int a, int b) { return ceil_div(a, b) * b; }

// Read `CNT` consecutive floats from LDS, `ALIGN` (1, 2 or 4 floats) being the
// alignment the caller guarantees for `p`; widest ds_read that alignment allows.
template <int CNT, int ALIGN>
__device__ __forceinline__ void lds_read_strip(const float *p, float (&dst)[CNT]) {
    int e = 0;
    if constexpr (ALIGN >= 4) {
#pragma unroll
        for (; e + 4 <= CNT; e += 4) {
            const float4 v = *reinterpret_cast<const float4 *>(p + e);
            dst[e] = v.x; dst[e + 1] = v.y; dst[e + 2] = v.z; dst[e + 3] = v.w;
        }
    }
    if constexpr (ALIGN >= 2) {
#pragma unroll
        for (; e + 2 <= CNT; e += 2) {
            const float2 v = *reinterpret_cast<const float2 *>(p + e);
            dst[e] = v.x; dst[e + 1] = v.y;
        }
    }
#pragma unroll
    for (; e < CNT; ++e) dst[e] = p[e];
}

// The same for `CNT` consecutive floats in global memory at an address aligned to `ALIGN` floats.
template <int CNT, int ALIGN>
__device__ __forceinline__ void global_read_strip(const float *__restrict__ p, float (&dst)[CNT]) {
    lds_read_strip<CNT, ALIGN>(p, dst);
}

// Sum over the 64 lanes of a wave; every lane receives the total.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Sum over the 64 lanes without LDS traffic: four DPP steps inside each row of 16 lanes, then the four row
// sums are read back as scalars.  The result is wave-uniform.
__device__ __forceinline__ float wave_sum_dpp(float v) {
    int t;
    t = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true);    // quad_perm [1,0,3,2]
    v += __int_as_float(t);
    t = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true);    // quad_perm [2,3,0,1]
    v += __int_as_float(t);
    t = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true);   // row_half_mirror
    v += __int_as_float(t);
    t = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, true);   // row_mirror
    v += __int_as_float(t);
    const float r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    const float r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    const float r2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    const float r3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
    return (r0 + r1) + (r2 + r3);
}

// K sums over the 64 lanes at once (K = 4, 8 or 16) for a caller that needs each of them in one lane only: a
// reduce-scatter.  In each of the first log2(K) steps a lane keeps half of its values, hands the other half to its
// partner and adds what the partner hands over, so that the values halve while the lanes per sum double (partners: lane
// ^ 1, lane ^ 2, then the lanes 4 and 8 further round the row of 16, which pairs the quads just as well); what is left
// of the four in-row steps are plain sums, and the four rows are added lane by lane through the LDS crossbar (two
// ds_bpermute; the row broadcasts of DPP hand on lane 15 only).  K + K/2 + ... additions instead of 6 K.
// Returns, in every lane, the sum of v[j] over the wave with j = wave_sum_scatter_index<K>(lane); v is used up.
template <int CTRL>
__device__ __forceinline__ float dpp_row_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int K>
__device__ __forceinline__ int wave_sum_scatter_index(int lane) {
    constexpr int BITS = K == 16 ? 4 : (K == 8 ? 3 : 2);
    return (int)(__brev((unsigned)lane) >> (32 - BITS));   // step s splits on bit s of the lane and on bit BITS-1-s of j
}
template <int K, int S, int CTRL>
__device__ __forceinline__ void wave_sum_scatter_step(float (&v)[K], int lane) {
    constexpr int n = (K >> S) > 1 ? (K >> S) : 1;   // values still held before this step
    if constexpr (n > 1) {
        constexpr int h = n / 2;
        const bool up = (lane >> S) & 1;
#pragma unroll
        for (int i = 0; i < h; ++i) {
            const float keep = up ? v[i + h] : v[i], send = up ? v[i] : v[i + h];
            v[i] = keep + dpp_row_move<CTRL>(send);
        }
    } else {
        v[0] += dpp_row_move<CTRL>(v[0]);
    }
}
template <int K>
__device__ __forceinline__ float wave_sum_scatter(float (&v)[K], int lane) {
    static_assert(K == 4 || K == 8 || K == 16, "4, 8 or 16 sums");
    wave_sum_scatter_step<K, 0, 0xB1>(v, lane);    // quad_perm [1,0,3,2]
    wave_sum_scatter_step<K, 1, 0x4E>(v, lane);    // quad_perm [2,3,0,1]
    wave_sum_scatter_step<K, 2, 0x124>(v, lane);   // row_ror:4
    wave_sum_scatter_step<K, 3, 0x128>(v, lane);   // row_ror:8
    float r = v[0];
    r += __shfl_xor(r, 16, 64);
    r += __shfl_xor(r, 32, 64);
    return r;
}

// BatchNorm with fixed statistics (inference), applied to a finished value of channel c:
// act((v - mean) / sqrt(var + eps) * gamma + beta [+ residual]).  gamma == null: not used.  The roundings -- reciprocal square
// root in one instruction, normalised value, multiply-add, shortcut -- are those of the BatchNorm that torch runs, so that a
// network gives the same bits whichever of the two it goes through (deep untrained ones amplify the last bit to 1e-3).
struct BnEval {
    const float *gamma, *beta, *mean, *var, *res;   // res (nullable): shaped like the output
    float eps;
    int relu;
};
static constexpr BnEval kNoBnEval{nullptr, nullptr, nullptr, nullptr, nullptr, 0.f, 0};
struct BnEvalChannel {
    float mean, rstd, gamma, beta;
    __device__ __forceinline__ BnEvalChannel(const BnEval &b, int c)
        : mean(b.mean[c]), rstd(rsqrtf(b.var[c] + b.eps)), gamma(b.gamma[c]), beta(b.beta[c]) {}
    __device__ __forceinline__ float operator()(float v) const { return fmaf(gamma, (v - mean) * rstd, beta); }
};
__device__ __forceinline__ float relu_keep_nan(float v) { return v < 0.f ? 0.f : v; }

struct ConvDims {
    int N, Ci, H, W, Co, kh, kw, stride, pad, Ho, Wo;
    __host__ __device__ int K() const { return Ci * kh * kw; }
};

// A wave's strips of `strips` per image lie in the image of the first and so many behind it
static inline long images_ahead(const ConvDims &d, long strips) {
    const long most = 63 / strips + 1;
    return most < d.N - 1 ? most : d.N - 1;
}
static constexpr long kMaxThreads = 0xffffffffL;   // of a launch

// ---- host-side launch plumbing -------------------------------------------------
int record_hip_error(hipError_t e);  // stores the message, returns ADDER_ERR_HIP
int check_launch();                  // hipGetLastError -> status

// Launchers implemented in the kernel translation units.
// T: storage type of the activations and their gradients, float or bf16_t (the optional reduced-storage mode).
// Forward without statistics (fwd.hip): which kernel, then those for 1x1 / pad 0 of any stride (fwd_tap.hip) and for 3x3 / pad 1 and
// 5x5 / pad 2 of stride 1 or 2 (fwd_nine.hip)
enum class FwdKernel { general = 0, plain_1x1 = 1, strided_tile = 2, tap = 3, nine = 4 };
struct LaneShape { int tm, tn, waves; };        // channels and positions per lane, waves that share the channels that are summed over
template <class T>
int launch_fwd(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn = kNoBnEval);
int fwd_kernel(const ConvDims &d);              // as in adder_conv2d_fwd_kernel
LaneShape fwd_tap_shape(const ConvDims &d);
LaneShape fwd_nine_shape(const ConvDims &d);
template <class T>
int launch_fwd_tap(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn);
bool fwd_tap_supported(const ConvDims &d);
template <class T>
int launch_fwd_nine(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn);
bool fwd_nine_supported(const ConvDims &d);
// ... large strided 1x1 layers in tiles (y aligned to groups where planes are whole groups); with statistics, and the ordinary convolution (fwd_tile.hip)
template <class T>
int launch_fwd_strided_tile(const T *x, const float *w, T *y, const ConvDims &d, hipStream_t s, const BnEval &bn);
bool fwd_strided_tile_supported(const ConvDims &d);
int launch_fwd_stats(const float *x, const float *w, float *y, double *stats, const ConvDims &d, hipStream_t s);
int fwd_stats_slots(const ConvDims &d);        // 0: no statistics epilogue for these dimensions
int fwd_stats_kernel(const ConvDims &d);       // as in adder_conv2d_fwd_stats_kernel
int fwd_chunk(const ConvDims &d);              // input channels per first-level sum of every forward of these dimensions: 8, 16 or 64
bool fwd_pair_supported(const ConvDims &d);
int launch_fwd_pair(const float *x, const float *w, const float *w_side, float *y, float *y_side, double *stats, double *stats_side,
                    const ConvDims &d, hipStream_t s);
int launch_mulconv_fwd(const float *x, const float *w, float *y, double *stats, const ConvDims &d, hipStream_t s);
template <class T>
int launch_grad_x(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s, const T *gadd = nullptr);
int grad_x_kernel(const ConvDims &d, bool bf16);   // as in adder_conv2d_grad_x_kernel
struct GradXShape { int tm, tn, waves; bool two; };   // of the kernels without tiles; two: two instructions a term, not three
GradXShape grad_x_tap_shape(const ConvDims &d, bool bf16);
GradXShape grad_x_nine_shape(const ConvDims &d, bool bf16, bool groups);
GradXShape grad_x_s2_shape(const ConvDims &d, bool sat);
// Whether the input gradient of a 3x3 or 1x1 layer of stride 1 is small and has no kernel that a BatchNorm is linked to: bfloat16, or rows (1x1: planes)
// that are no whole groups of four.  Those take three instructions a term: the doubled sum minus the sum of gy that two need rounds once more (3x3 of 60
// to 100 output channels: 2.4e-7 of the result against 1.7e-7, the largest element 1.5 times as far) and makes an infinite gy NaN.  Small: a launch that a
// kernel of one position per lane finishes (0.45 us of nine taps or 0.15 of one a channel of a wave's share, then 9 or 6.5 terms per ps) before one of 16
// results per lane (small maps: eight) has walked all output channels (5.5 or 9.5 ns a term and result).
static inline bool small_unlinked(const ConvDims &d, bool bf16) {
    const bool nine = d.kh == 3;
    const int row = nine ? d.W : d.H * d.W;
    if (!bf16 && row % 4 == 0) return false;
    if (!nine && row <= 64 && (long)ceil_div(d.N, 4) * ceil_div(d.Ci, 64) > 256) return false;
    const int results = row > (nine ? 8 : 64) ? 16 : 8, eighth = round_up(ceil_div(d.Co, 8), 8), chunk = nine ? 8 : eighth < 16 ? 16 : eighth > 64 ? 64 : eighth;
    const float terms = (float)d.K() * d.Co * d.N * d.H * d.W, share = (float)(ceil_div(ceil_div(d.Co, chunk), 8) * chunk);
    const float all = nine ? 2.f + 0.0055f * 9 * results * d.Co : 3.f + 0.0095f * results * d.Co;
    return (nine ? 2.f + 0.45f * share + terms / 9e6f : 3.f + 0.15f * share + terms / 6.5e6f) < 0.9f * all;
}
// 1x1 / stride 1 (grad_x_tap.hip); bn (nullable): the in_* half of adder_bn_links, slots of sums per channel
template <class T>
int launch_grad_x_tap(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s, const T *gadd,
                      const adder_bn_links *bn);
bool grad_x_tap_supported(const ConvDims &d);
bool grad_x_tap_narrow(const ConvDims &d);      // layers it takes beside those, without links and second gradients
int grad_x_tap_bn_slots(const ConvDims &d);
// 3x3 / pad 1 and 5x5 / pad 2 / stride 1 (grad_x_nine.hip), likewise; groups: rows are no whole groups of four, or the bases are aligned to
// groups (elsewhere three instructions a term)
template <class T>
int launch_grad_x_nine(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s, const T *gadd,
                       const adder_bn_links *bn, bool groups = true);
bool grad_x_nine_supported(const ConvDims &d);
int grad_x_nine_bn_slots(const ConvDims &d);
// 3x3 / pad 1 and 5x5 / pad 2 / stride 2 (grad_x_s2.hip); sat: two instructions a term
template <class T>
int launch_grad_x_s2(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s, const T *gadd, bool sat);
bool grad_x_s2_supported(const ConvDims &d);
static constexpr int kSatMaxTerms = 1152;      // terms up to which a 3x3 layer's input gradient takes two instructions a term (grad_x.hip)
static constexpr bool two_instructions_5x5(int Co) { return Co >= 10 && Co * 25 <= 2500; }   // ... and those of 5x5 layers (grad_x.hip)
static constexpr int kSatMaxTerms1x1 = 1024;   // output channels up to which a single tap's input gradient takes two instructions a term (grad_x.hip)
size_t grad_w_workspace_bytes(const ConvDims &d, bool bf16 = false, size_t limit = SIZE_MAX);   // of the storage type's kernels
int grad_w_kernel(const ConvDims &d, bool bf16);                                                // which of them, as in adder_conv2d_grad_w_kernel
// The sums of the backward of the BatchNorm behind a layer, as the consumer's input-gradient kernel left them
// ((C, slots, 2) floats -- a wave's fp32 totals: sum dz, sum dz * xhat), with what turns them into the four coefficients per channel.
// A weight-gradient kernel that is given these instead of ready coefficients adds the slots itself (every
// workgroup its own channels, all in the same order) and writes dgamma / dbeta on the way.  part == null: not used.
struct BnSums {
    const float *part;
    int slots;
    double count;            // N * Ho * Wo: values per channel of the BatchNorm
    const float *gamma, *mean, *rstd;
    float *dgamma, *dbeta;
};
static constexpr BnSums kNoBnSums{nullptr, 0, 0.0, nullptr, nullptr, nullptr, nullptr, nullptr};
template <class T>
int launch_grad_w(const T *gy, const T *x, const float *w, float *gw, float eta,
                  void *ws, size_t ws_bytes, const ConvDims &d, hipStream_t s, const float *bn_y = nullptr,
                  const float *bn_coef = nullptr, float *gy_out = nullptr, const BnSums &sums = kNoBnSums,
                  size_t limit = SIZE_MAX);   // limit, as given to grad_w_workspace_bytes: fewer slabs where they are too many for it
// launch_grad_w without slabs (any layer): `ws` holds the norm partials only, kGradWGeneralWs bytes
static constexpr size_t kGradWGeneralWs = 128 * 1024;
template <class T>
int launch_grad_w_general(const T *gy, const T *x, const float *w, float *gw, float eta, void *ws, const ConvDims &d,
                          hipStream_t s);
// the BatchNorm backward passes of a layer's neighbours inside the layer's backward kernels (adder_bn_links)
int grad_x_bn_slots(const ConvDims &d);
int launch_grad_x_bn(const float *gy, const float *x, const float *w, float *gx, const ConvDims &d, hipStream_t s,
                     const float *gadd, const adder_bn_links &bn);
bool grad_w_bn_supported(const ConvDims &d, const void *gy, const void *x, const void *bn_y, const void *bn_coef);
int launch_bn_bwd_coef(const float *part, int slots, const float *gamma, const float *mean, const float *rstd,
                       double count, float *coef, float *dgamma, float *dbeta, int C, hipStream_t s);

// matrix-core weight gradient of the 3x3 / pad-1, 5x5 / pad-2 and wide 1x1 layers (grad_w_mfma.hip); variant 0 = not applicable
struct GradWMfmaPlan { int variant, slots, gy, gz, tilesH, tilesW, ntiles; };
GradWMfmaPlan plan_grad_w_mfma(const ConvDims &d);
template <class T>
int launch_grad_w_mfma(const T *gy, const T *x, double *part, double *sgpart, const ConvDims &d, const GradWMfmaPlan &p,
                       hipStream_t s);
int launch_grad_w_mfma_bn(const float *gy, const float *x, double *part, double *sgpart, const ConvDims &d,
                          const GradWMfmaPlan &p, const float *bn_y, const float *bn_coef, float *gy_out, hipStream_t s,
                          const BnSums &sums = kNoBnSums);
int plan_grad_w_slots(int blocks, int ntiles, size_t slab_bytes);
// large layers in bfloat16 storage, on the 8-bit matrix cores (grad_w_i8.hip): variants from 20 on
bool plan_grad_w_i8(const ConvDims &d, GradWMfmaPlan &p);
int launch_grad_w_i8(const bf16_t *gy, const bf16_t *x, double *part, double *sgpart, const ConvDims &d, const GradWMfmaPlan &p, hipStream_t s);

// 1x1 / pad 0 / stride 1-2 kernels (conv1x1.hip)
bool conv1x1_supported(const ConvDims &d, const void *a, const void *b);
int fwd_1x1_stats_slots(const ConvDims &d);
template <class T>
int launch_fwd_1x1(const T *x, const float *w, T *y, double *stats, const ConvDims &d, hipStream_t s, const BnEval &bn = kNoBnEval);
static constexpr int kGx1x1TM = 4;   // input channels per workgroup; latency-bound at ResNet sizes: more workgroups beat more reuse per lane
template <class T>
int launch_grad_x_1x1(const T *gy, const T *x, const float *w, T *gx, const ConvDims &d, hipStream_t s);
int grad_w_1x1_slots(const ConvDims &d);
// P: float slabs for float storage, double ones for bfloat16; with gw (bfloat16 only, slots = 1) the finished gradient and no slabs
template <class T, class P>
int launch_grad_w_1x1(const T *gy, const T *x, P *part, P *sgpart, const float *w, float *gw, int slots, const ConvDims &d,
                      hipStream_t s);

// fused BatchNorm + residual + ReLU (bn_act.hip)
size_t bn_workspace_bytes(int N, int C, int HW);
size_t bn_mask_words(int N, int C, int HW);
int launch_bn_act_fwd(const float *x, const float *res, const float *gamma, const float *beta, float *y,
                      unsigned *mask, float *mean, float *rstd, float *running_mean, float *running_var,
                      long long *num_batches, float momentum, float eps, int relu, int N, int C, int HW, void *ws,
                      const double *stats, int stats_slots, hipStream_t s);
int launch_bn_eval(const float *x, float *y, const BnEval &bn, int N, int C, int HW, hipStream_t s);
int launch_bn_act_bwd(const float *dy, const float *y, const unsigned *mask, const float *x, const float *gamma,
                      const float *mean, const float *rstd, float *dx, float *dres, float *dgamma, float *dbeta,
                      int relu, int N, int C, int HW, void *ws, hipStream_t s);

// average pool over the whole map -> matrix product -> BatchNorm of the ResNet classifier head (head.hip)
bool head_supported(int N, int C, int HW, int J);
int launch_head_fwd(const float *x, const float *w, const float *gamma, const float *beta, float *pooled, float *z,
                    float *y, float *mean, float *rstd, float *running_mean, float *running_var, long long *num_batches,
                    float momentum, float eps, int N, int C, int HW, int J, hipStream_t s);
int launch_head_bwd(const float *dy, const float *z, const float *pooled, const float *w, const float *gamma,
                    const float *mean, const float *rstd, float *dz, float *dx, float *dw, float *dgamma, float *dbeta,
                    int N, int C, int HW, int J, hipStream_t s);

int launch_ce_fwd(const float *y, const long long *target, float *loss, float *lse, int N, int J, hipStream_t s);
int launch_ce_bwd(const float *y, const long long *target, const float *lse, const float *grad_loss, float *gy, int N,
                  int J, hipStream_t s);

size_t norm_scale_workspace_bytes(long n);
int launch_norm_scale(float *g, long n, float eta, float eps, void *ws, hipStream_t s);
static constexpr int kNormBatchMax = ADDER_NORM_BATCH_MAX;
static constexpr int kSgdBatchMax = ADDER_SGD_BATCH_MAX;
int launch_sgd_momentum(int count, float *const *p, const float *const *g, float *const *buf, const long *n,
                        const float *lr_ptr, float lr, float momentum, float weight_decay, hipStream_t s);
static constexpr int kGwFinishMax = ADDER_GRAD_W_FINISH_MAX;
int launch_grad_w_staged(const float *gy, const float *x, const float *w, float *gw, float eta, void *ws,
                         size_t ws_bytes, const ConvDims &d, adder_grad_w_stage *stage, hipStream_t s,
                         const float *bn_y = nullptr, const float *bn_coef = nullptr, float *gy_out = nullptr,
                         const BnSums &sums = kNoBnSums);
size_t grad_w_finish_workspace_bytes(int count, const adder_grad_w_stage *st);
int launch_grad_w_finish(int count, const adder_grad_w_stage *st, void *ws, hipStream_t s);
size_t norm_scale_batched_workspace_bytes(int count);
int launch_norm_scale_batched(int count, float *const *g, const long *n, const float *eta, float eps, void *ws,
                              hipStream_t s);

int launch_grad_w_slab_finalize(const double *part, const double *sgpart, const float *w, float *gw, int slots, int Co,
                                int K, bool accumulate, hipStream_t s);
int launch_col_fwd(const float *X, const float *W, float *out, int K, long NL, int Co, hipStream_t s);
size_t col_grad_w_workspace_bytes(int K, long NL, int Co);
int launch_col_grad_w(const float *gy, const float *X, const float *W, float *gW, int K, long NL,
                      int Co, void *ws, hipStream_t s, bool add = true);
int launch_col_grad_x(const float *gy, const float *X, const float *W, float *gX, int K, long NL,
                      int Co, hipStream_t s, bool add = true);
int launch_col_bwd_small(const float *gy, const float *X, const float *W, float *gW, float *gX, int K, long NL, int Co,
                         hipStream_t s, bool add = true);
int launch_col_bwd_fused(const float *gy, const float *X, const float *W, float *gW, float *gX, int K, long NL, int Co,
                         void *ws, hipStream_t s, bool add = true);

}  // namespace adder

// What the kernels whose waves share the channels of one set of results have in common: sums that meet in LDS, the inference
// epilogue, the stores.  A lane holds TM channels x TN adjacent positions.
#pragma once
#include "common.hpp"

namespace adder {

// TN adjacent floats of LDS, aligned to as many
template <int TN>
__device__ __forceinline__ void lds_ld(const float *p, float (&v)[TN]) {
    static_assert(TN == 1 || TN == 2 || TN == 4, "one, two or four positions");
    if constexpr (TN == 4) {
        const float4 u = *reinterpret_cast<const float4 *>(p);
        v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
    } else if constexpr (TN == 2) {
        const float2 u = *reinterpret_cast<const float2 *>(p);
        v[0] = u.x; v[1] = u.y;
    } else {
        v[0] = *p;
    }
}
template <int TN>
__device__ __forceinline__ void lds_st(float *p, const float (&v)[TN]) {
    if constexpr (TN == 4) *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
    else if constexpr (TN == 2) *reinterpret_cast<float2 *>(p) = make_float2(v[0], v[1]);
    else *p = v[0];
}

// Forward sums: chunks of input channels, added in channel order (fwd_chunk), so that a layer's results have the same bits in
// every kernel and however many waves share its chunks -- wave v takes the chunks v, v + waves, ...
// SHARED: after each round the waves' chunk sums meet in LDS and a wave adds those of its FM channels, from v * per_wave on, to what
// it holds.  Otherwise one wave has all chunks and keeps the sums of sums in LDS, a place of its own per lane, which frees TM * TN
// registers.
// TURN: a lane's sums are those of positions lane, 64 + lane, ... of the tile; what it has at the end is those of TN adjacent ones.
template <int TM_, int TN_, bool SHARED_, bool TURN_ = false>
struct ChunkSums {
    static constexpr int TM = TM_, TN = TN_;
    static constexpr bool SHARED = SHARED_, TURN = TURN_;
    static constexpr int FM = SHARED ? TM / 2 : TM;      // most channels a wave finishes
    static constexpr int WAVE_FLOATS = TM * TN * 64;     // of LDS
    static_assert(TM % 2 == 0, "two waves finish half of the channels each");
    float *smem;
    int wave, lane, waves, chunks, per_wave, round = 0;
    float tot[FM][TN];

    __device__ __forceinline__ ChunkSums(float *smem_, int wave_, int lane_, int waves_, int chunks_)
        : smem(smem_), wave(wave_), lane(lane_), waves(waves_), chunks(chunks_), per_wave(SHARED ? (TM + waves_ - 1) / waves_ : TM) {
        if constexpr (SHARED) {
#pragma unroll
            for (int f = 0; f < FM; ++f)
#pragma unroll
                for (int t = 0; t < TN; ++t) tot[f][t] = 0.f;
        }
    }
    __device__ __forceinline__ int chunk() const { return SHARED ? round * waves + wave : round; }   // that this wave is at
    __device__ __forceinline__ bool pending() const { return chunk() < chunks; }
    __device__ __forceinline__ int first_channel() const { return SHARED ? wave * per_wave : 0; }

    // A chunk of this wave ends (mine), or it has none in this round: acc -> the sums of sums, and zero.
    __device__ __forceinline__ void add(float (&acc)[TM][TN], const bool mine = true) {
        if constexpr (SHARED) {
            if (round > 0) __syncthreads();   // the sums of the round before have been read
            if (mine) {
#pragma unroll
                for (int m = 0; m < TM; ++m) lds_st<TN>(smem + wave * WAVE_FLOATS + (m * 64 + lane) * TN, acc[m]);
            }
            __syncthreads();
            if (first_channel() < TM) {
                const int here = min(waves, chunks - round * waves);
                if (per_wave == 1) gather<1>(here);
                else if (per_wave == 2) gather<(FM < 2 ? FM : 2)>(here);
                else if (FM <= 4 || per_wave <= 4) gather<(FM < 4 ? FM : 4)>(here);
                else gather<FM>(here);
            }
        } else if (round == 0) {
#pragma unroll
            for (int m = 0; m < TM; ++m) lds_st<TN>(smem + (m * 64 + lane) * TN, acc[m]);
        } else {
            constexpr int R = TM < 4 ? TM : 4;   // rows at a time
#pragma unroll
            for (int m0 = 0; m0 < TM; m0 += R) {
                float u[R][TN];
#pragma unroll
                for (int m = 0; m < R; ++m) lds_ld<TN>(smem + ((m0 + m) * 64 + lane) * TN, u[m]);
#pragma unroll
                for (int m = 0; m < R; ++m) {
#pragma unroll
                    for (int t = 0; t < TN; ++t) u[m][t] += acc[m0 + m][t];
                    lds_st<TN>(smem + ((m0 + m) * 64 + lane) * TN, u[m]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        ++round;
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int t = 0; t < TN; ++t) acc[m][t] = 0.f;
    }
    // this round's sums of the first F of this wave's channels (and of others, which nobody asks for, where it has fewer)
    template <int F>
    __device__ __forceinline__ void gather(const int here) {
        const float *p = smem + (first_channel() * 64 + lane) * TN;
        const int last = TM - 1 - first_channel();
        constexpr int B = 8 / F;   // waves whose sums are asked for together
        for (int v0 = 0; v0 < here; v0 += B) {
            float u[B][F][TN];
#pragma unroll
            for (int b = 0; b < B; ++b)
#pragma unroll
                for (int f = 0; f < F; ++f) lds_ld<TN>(p + min(v0 + b, here - 1) * WAVE_FLOATS + min(f, last) * (64 * TN), u[b][f]);
#pragma unroll
            for (int b = 0; b < B; ++b) {
                if (v0 + b >= here) break;
#pragma unroll
                for (int f = 0; f < F; ++f)
#pragma unroll
                    for (int t = 0; t < TN; ++t) tot[f][t] += u[b][f][t];
            }
        }
    }
    // Behind the last chunk: a wave that had none in the last round meets the others there; tot holds this wave's results
    __device__ __forceinline__ void finish(float (&acc)[TM][TN]) {
        if constexpr (SHARED) {
            if (round * waves < chunks) add(acc, false);
        } else {
#pragma unroll
            for (int m = 0; m < TM; ++m) lds_ld<TN>(smem + (m * 64 + lane) * TN, tot[m]);
        }
        if constexpr (TURN) {
            __syncthreads();   // the last sums have been read
            float *p = smem + first_channel() * (64 * TN);
#pragma unroll
            for (int f = 0; f < FM; ++f)
                if (first_channel() + f < TM && f < per_wave) {
#pragma unroll
                    for (int t = 0; t < TN; ++t) p[(f * TN + t) * 64 + lane] = tot[f][t];
                }
            __syncthreads();
#pragma unroll
            for (int f = 0; f < FM; ++f)
                if (first_channel() + f < TM && f < per_wave) lds_ld<TN>(p + (f * 64 + lane) * TN, tot[f]);
        }
    }
};

// Strips of TN columns per row: strip s starts at column s * TN, the last one is moved back to end with the row.  Where the columns beside a strip are read in
// pairs (25 taps) no pair may be half inside the row, so rows that would cut one take the strips from number `from` on a column earlier.
// start, first: a strip's first column, and the first that is its own and not the strip's before it.
struct Strips {
    int per_row, from;
    __device__ __forceinline__ int start(int s, int tn, int row) const { return min(s * tn - (s >= from ? 1 : 0), row - tn); }
    __device__ __forceinline__ int first(int s, int tn) const { return s * tn - (s > from ? 1 : 0); }
};
static constexpr int kNoShift = 0x7fffffff;

// Waves that share `chunks` chunks, at most `most`: as few as finish them in the same number of rounds
static inline int waves_for(int chunks, int most) { return ceil_div(chunks, ceil_div(chunks, most)); }

// Chunks of `channels` input channels, one less where less than half of the last one is filled: what counts where waves share them
static inline int full_chunks(int channels, int chunk) {
    const int chunks = ceil_div(channels, chunk);
    return chunks > 1 && 2 * (channels - (chunks - 1) * chunk) < chunk ? chunks - 1 : chunks;
}

// The waves' results on their way out, count of the FM channels from co0 on.  own: bit t of the positions that are this lane's; off: its
// first one in channel 0 of its image; L: positions per plane.  EVAL: bn is applied (float storage).  whole: TN positions are always
// this lane's own.
template <int FM, int TN, bool EVAL, class T>
__device__ __forceinline__ void finish_outputs(float (&r)[FM][TN], int count, unsigned own, int co0, int Co, int L, int off, bool whole,
                                               T *__restrict__ y, const BnEval &bn) {
    if constexpr (EVAL) {
        float a[FM][TN];
#pragma unroll
        for (int f = 0; f < FM; ++f) {   // (all loads before the first store: one counter serves both)
#pragma unroll
            for (int t = 0; t < TN; ++t) a[f][t] = 0.f;
            if (bn.res) ld_strip<TN>(bn.res + (size_t)min(co0 + f, Co - 1) * L + off, a[f]);
        }
#pragma unroll
        for (int f = 0; f < FM; ++f) {
            const BnEvalChannel ch(bn, min(co0 + f, Co - 1));
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                r[f][t] = ch(r[f][t]) + a[f][t];
                if (bn.relu) r[f][t] = relu_keep_nan(r[f][t]);
            }
        }
    }
#pragma unroll
    for (int f = 0; f < FM; ++f) {
        if (f >= count || co0 + f >= Co) break;
        T *dst = y + (size_t)(co0 + f) * L + off;
        if (whole && own) {
            if constexpr (TN == 4 || TN == 2) st_strip<TN>(dst, r[f]);
        } else {
#pragma unroll
            for (int t = 0; t < TN; ++t)
                if (own >> t & 1) stf(dst + t, r[f][t]);
        }
    }
}

// Of the rows of results of an input gradient, those that one of KSP waves finishes: all share them, or one each
template <int TM, int KSP>
static constexpr int kFinished = TM >= KSP ? TM / KSP : 1;

// Input gradients likewise: a second gradient (gadd, nullable) is added, the first pass of the BatchNorm in front of the layer is
// made where FUSE (the in_* fields of adder_bn_links: one slot of sums per tile; float storage), channels first <= c < Ci of the
// FM from ci0 on are stored.  off: the lane's first position in channel ci0.
template <int FM, int TN, bool FUSE, class T>
__device__ __forceinline__ void finish_grad_x(float (&r)[FM][TN], unsigned own, int ci0, int first, int Ci, int L, int off, bool whole,
                                              const T *__restrict__ x, T *__restrict__ gx, const T *__restrict__ gadd,
                                              const adder_bn_links &bn, int tiles, int tile, int lane) {
    // (all loads before the first store: one counter serves both; channels past Ci read the last one)
    float a[FM][TN];
    if (gadd) {
#pragma unroll
        for (int f = 0; f < FM; ++f) ld_strip<TN>(gadd + off + (size_t)min(f, Ci - 1 - ci0) * L, a[f]);
    }
    if constexpr (FUSE) {
        // x = relu(bn(in_x) [+ residual]): dz = (gx + gadd) * [x > 0] and per channel the sums of dz and dz * xhat.  xhat comes from x
        // where nothing but the ReLU followed the BatchNorm and |gamma| is large enough for the division, else from in_x.
        float xv[FM][TN];
#pragma unroll
        for (int f = 0; f < FM; ++f) ld_strip<TN>(x + off + (size_t)min(f, Ci - 1 - ci0) * L, xv[f]);
#pragma unroll
        for (int f = 0; f < FM; ++f) {
            const int c = min(ci0 + f, Ci - 1);
            const float g = bn.in_gamma ? as_uniform(bn.in_gamma)[c] : 0.f, be = bn.in_gamma ? as_uniform(bn.in_beta)[c] : 0.f;
            const bool from_x = bn.in_gamma && fabsf(g) >= 0x1p-6f * fmaxf(1.f, fabsf(be));
            float bx[TN];
#pragma unroll
            for (int t = 0; t < TN; ++t) bx[t] = xv[f][t];
            if (!from_x) ld_strip<TN>(bn.in_x + off + (size_t)(c - ci0) * L, bx);
            const float centre = from_x ? be : as_uniform(bn.in_mean)[c];
            const float scale = from_x ? __builtin_amdgcn_rcpf(g) : as_uniform(bn.in_rstd)[c];
            float a1 = 0.f, a2 = 0.f;
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                if (gadd) r[f][t] += a[f][t];
                const bool keep = (own >> t & 1) && !(bn.in_relu && !(xv[f][t] > 0.f));
                const float v = keep ? r[f][t] : 0.f;
                r[f][t] = v;
                a1 += v;
                a2 = fmaf(v, bx[t] - centre, a2);
            }
            const float s1 = wave_sum_dpp(a1), s2 = wave_sum_dpp(a2) * scale;
            if (lane == 0 && ci0 + f >= first && ci0 + f < Ci) {
                float *dst = bn.in_part + ((size_t)(ci0 + f) * tiles + tile) * 2;
                dst[0] = s1;
                dst[1] = s2;
            }
        }
    } else if (gadd) {
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int t = 0; t < TN; ++t) r[f][t] += a[f][t];
    }
#pragma unroll
    for (int f = 0; f < FM; ++f) {
        if (ci0 + f < first || ci0 + f >= Ci) continue;
        T *dst = gx + off + (size_t)f * L;
        if (whole && own) {
            if constexpr (TN == 2 || TN == 4) st_strip<TN>(dst, r[f]);
        } else {
#pragma unroll
            for (int t = 0; t < TN; ++t)
                if (own >> t & 1) stf(dst + t, r[f][t]);
        }
    }
}

}  // namespace adder

// The channel filter branch of DDFPack with its weights in LDS, as device functions: on the
// matrix cores (channel_mma, fp16) and on the vector ALU (channel_rows).  A layer's kernels
// (ddf_branches.hip) are nothing else, a network's run them beside the spatial branch
// (ddf_net.hip).
#pragma once

#include <algorithm>

#include "ddf_common.h"
#include "ddf_rows.h"

namespace ddf {

// Both 1x1 convolutions are matrix products with the batch as one dimension:
//   hidden[m, n] = relu(b1[m] + sum_c w1[m, c] * v[n, c])           (mid x C) . (C x N)
//   taps[r, n]   = b2[r] + sum_m w2[r, m] * hidden[m, n]            (C*KK x mid) . (mid x N)
// v_mfma_f32_16x16x32_f16 takes, per lane l of a wave, eight values of a row of A
// (row l % 16, positions 8 * (l / 16) + 0..7 of the 32 the step covers: one
// 16-byte load from a row-major weight matrix) and the eight values of column
// l % 16 of B at the same positions, and leaves D[4 * (l / 16) + 0..3][l % 16].
// A workgroup takes sixteen samples (the columns) and sixteen channels:
//   * the pooled vectors go to LDS as [32 channels][sample][32], rounded to fp16
//     (what the reference's half-precision pooling returns);
//   * the hidden layer goes to LDS as [32 values][sample][32], rounded to fp16 (as
//     the reference's first convolution does);
//   * the rows of tile j of the second product are (channel c0 + i, tap j); the taps meet in
//     LDS as fp32, and a thread per sample and channel normalises and stores them.
// mid is no multiple of 16 or 32: rows of w1 past the last are whatever lies in LDS and make
// hidden values that are set to zero; the last step of a row of w2 is cut at its end.
//
// There is no arithmetic to speak of: the launch is a chain of round trips and the way the
// weights come in.  An operand read straight from memory is sixteen rows of 64 bytes per load
// instruction, which a compute unit takes 70 (aligned rows) to 110 clocks for, where 1 KB in a
// row takes 20 (eight waves, from L2); a workgroup of 256 channels has 68 such loads.  So w1
// and the block's part of w2 - one run of bytes each - come in as they lie, straight into
// LDS, before anything else, and operands are read from there; biases, gains and offsets
// are requested along with them by the other half of the waves.  Eight waves take the hidden
// tiles, five the nine taps, four the normalisation (one wave had taps and normalisation).  us a
// launch, before / now: 1 sample x 256 channels 8.2 / 4.7, 1 x 512 9.2 / 6.2, 128 x 256 9.9 / 5.8,
// 128 x 512 13.2 / 8.5, 4 x 1024 24.3 / 22.2 (an empty launch: 1.6).
constexpr int kMmaSamples = 16, kMmaChannels = 16;
constexpr int kMmaStep = 32;                          // values of the summed dimension per instruction
constexpr int kMmaTile = kMmaSamples * kMmaStep;      // halves of one [sample][32] tile in LDS
constexpr int kMmaWaves = 8, kMmaThreads = kMmaWaves * kWave;
constexpr int kMmaSpread = 4 * kWave;                 // channels up to which waves share a value's partial sums
constexpr int kMmaRound = 8;                          // partial sums requested together
constexpr int kMmaLds = 160 * 1024;

// LDS, bytes: pooled vectors | rows of w1 | the block's rows of w2 | hidden vectors | partial
// sums on their way to the pooled vectors.  All rows of w1 and w2 where they fit; else w1 by
// `chunk` rows and w2 in the same place after it, or (stage_w2 false) from memory.  The block's
// taps go where w1 and the pooled vectors were.
struct ChannelMmaLds {
    int pitch;                  // bytes of a row of w1
    int chunk;                  // rows of w1 at a time, whole tiles
    int w1, w2, hidden, sums, total;
    bool stage_w2, shared;      // shared: the taps reach into the rows of w2
};
inline int mma_round(int64_t v) { return (int)((v + 15) / 16 * 16); }
inline ChannelMmaLds channel_mma_lds(int64_t C, int64_t mid, int kk, int64_t most = kMmaLds) {
    ChannelMmaLds l{};
    // (a wave's load is 1 KB: two rows of up to 256 channels, or one in pieces of 512)
    l.pitch = C <= 256 ? 512 : (int)((C + 511) / 512 * 1024);
    const int64_t pooled = C * kMmaSamples * 2, rows = (mid + 15) / 16 * 16;
    const int64_t w2 = (int64_t)kMmaChannels * kk * mid * 2;
    const int64_t hidden = (mid + kMmaStep - 1) / kMmaStep * kMmaTile * 2, sums = C <= kMmaSpread ? kMmaThreads * 16 : 0;
    const int64_t taps = kMmaSamples * (kMmaChannels * kk + 1) * 4;
    const int64_t left = most - pooled - hidden - sums;
    l.w1 = (int)pooled;
    int64_t space;
    if (rows * l.pitch + w2 <= left) {
        l.chunk = (int)rows;
        l.stage_w2 = true;
        l.w2 = l.w1 + (int)rows * l.pitch;
        space = rows * l.pitch + w2;
    } else {
        l.chunk = (int)std::min<int64_t>(rows, std::max<int64_t>(left / l.pitch / 16 * 16, 0));
        l.stage_w2 = w2 <= left;
        l.w2 = l.w1;
        space = std::max<int64_t>((int64_t)l.chunk * l.pitch, l.stage_w2 ? w2 : 0);
    }
    space = std::max(space, taps - pooled);
    l.shared = l.stage_w2 && l.w2 < taps;
    l.hidden = mma_round(l.w1 + space);
    l.sums = l.hidden + (int)hidden;
    l.total = l.sums + (int)sums;
    return l;
}
inline bool channel_mma_covers(int64_t C, int64_t mid, int kk) {
    if (mid < kMmaStep || C % kMmaStep != 0 || C * kk * mid >= ((int64_t)1 << 31)) return false;
    if (C / kMmaStep + (mid + kMmaStep - 1) / kMmaStep > 64) return false;
    const ChannelMmaLds l = channel_mma_lds(C, mid, kk);
    return l.chunk > 0 && l.total <= kMmaLds;
}

struct ChannelMma {
    const __half *pooled, *w1, *b1, *w2, *b2;
    __half *cf;
    int N, C, mid;
    float gain;
    const __half *gain_vec, *offset_vec;
    const float *parts;    // (nparts per sample; null: `pooled`)
    int nparts;
    float scale;
    ChannelSave save;
    ChannelMmaLds lds;
};

#ifdef __HIPCC__

// Gains, offsets and biases of the KK taps of filter group `g`, read once (all
// loads go out together; read tap by tap where they are used, every one of
// them is a round trip of its own at the end of the kernel).
template <typename T, int KK>
struct TapParams {
    float gain[KK], offset[KK], bias[KK];
    __device__ __forceinline__ void load(int64_t g, float scalar_gain, const T *gain_vec,
                                         const T *offset_vec, const T *bias_vec) {
#pragma unroll
        for (int t = 0; t < KK; ++t) {
            gain[t] = scalar_gain;
            offset[t] = 0.f;
            bias[t] = 0.f;
        }
        if (gain_vec) {
#pragma unroll
            for (int t = 0; t < KK; ++t) gain[t] = ld(gain_vec + g * KK + t);
        }
        if (offset_vec) {
#pragma unroll
            for (int t = 0; t < KK; ++t) offset[t] = ld(offset_vec + g * KK + t);
        }
        if (bias_vec) {
#pragma unroll
            for (int t = 0; t < KK; ++t) bias[t] = ld(bias_vec + g * KK + t);
        }
    }
};

// v[0..KK) + bias, standardised in place, times gain plus offset.
template <typename T, int KK>
__device__ __forceinline__ void normalise(float (&v)[KK], const TapParams<T, KK> &p) {
    float sum = 0;
#pragma unroll
    for (int t = 0; t < KK; ++t) {
        v[t] += p.bias[t];
        sum += v[t];
    }
    const float mean = sum / (float)KK;
    float sq = 0;
#pragma unroll
    for (int t = 0; t < KK; ++t) {
        v[t] -= mean;
        sq += v[t] * v[t];
    }
    const float inv = 1.f / (sqrtf(sq / (float)(KK - 1)) + 1e-10f);
#pragma unroll
    for (int t = 0; t < KK; ++t) v[t] = v[t] * inv * p.gain[t] + p.offset[t];
}


typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// Sum over the wave's four rows of sixteen lanes (the same value in every lane of a column).
__device__ __forceinline__ float rows_total(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(h[0]) + __uint_as_float(h[1]);
}

// 16 bytes per lane to LDS at `lds` + lane * 16.  (Written out because the compiler waits for
// every such load in flight before any LDS read.  The address is an operand in m0, so that the
// compiler itself writes m0 and knows it; the load must not follow that write at once.)
__device__ __forceinline__ void load_to_lds(uint32_t lds, const void *p) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(lds), "v"(p) : "memory");
}
// The same from a uniform address and a lane's offset.  (A scalar register that a vector instruction
// has written - a spilled one that comes back by v_readlane - may be read by a vector memory instruction
// five wait states later; the compiler does not see one in here.)
__device__ __forceinline__ void load_to_lds(uint32_t lds, const char *base, int offset) {
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds), "v"(offset), "s"(base) : "memory");
}
// This wave's are there.
__device__ __forceinline__ void loads_to_lds_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// What a workgroup does beside the branch - in front of its first requests, behind them in a wave that fetches weights
// (true); while they are on their way; once a wave's hidden values are made - and where a channel's taps go.
struct Nothing {
    template <typename... A>
    __device__ __forceinline__ void operator()(A...) const {}
};
template <typename T, int KK>
struct ToFilter {    // (sample, channel, taps) to a tensor
    T *cf;
    int C;
    __device__ __forceinline__ void operator()(int64_t n, int c, const float (&u)[KK]) const {
        T o[KK];
#pragma unroll
        for (int j = 0; j < KK; ++j) st(&o[j], u[j]);
        __builtin_memcpy(cf + (n * C + c) * KK, o, sizeof(o));
    }
};

// Channels 16 * bx on of the ns (up to 16) samples from n0 on, kMmaThreads threads.  SAVE: a.save
// is wanted (compiled in, as a branch around every store has the loads before it wait one by one).
template <int KK, bool SAVE, typename Begin, typename Meanwhile, typename After, typename Sink>
__device__ __forceinline__ void channel_mma(const ChannelMma &a, int bx, int n0, int ns, unsigned char *smem,
                                            const Begin &begin, const Meanwhile &meanwhile, const After &after, const Sink &sink) {
    constexpr int TPW = KK <= 9 ? 2 : 4, TAP_WAVES = (KK + TPW - 1) / TPW;      // taps per wave
    constexpr int NORM_WAVES = kMmaSamples * kMmaChannels / kWave;
    static_assert(TAP_WAVES <= kMmaWaves && NORM_WAVES <= kMmaWaves && KK % 8 == 1);
    constexpr int ZP = kMmaChannels * KK + 1;            // (odd: samples in different banks)
    at_once(a.w1, a.w2, a.parts, a.b1, a.C, a.mid, a.nparts, a.lds.w1, a.lds.w2, a.lds.chunk, a.lds.pitch, a.lds.hidden);
    const int C = a.C, mid = a.mid;
    _Float16 *pv = reinterpret_cast<_Float16 *>(smem);   // [C / 32][16 samples][32]: pooled vectors
    float *z = reinterpret_cast<float *>(smem);          // [sample][channel][tap], in their place and w1's
    const unsigned char *w1s = smem + a.lds.w1, *w2s = smem + a.lds.w2;
    _Float16 *hv = reinterpret_cast<_Float16 *>(smem + a.lds.hidden);   // [steps of mid][16 samples][32]: hidden vectors
    float4_t *ps = reinterpret_cast<float4_t *>(smem + a.lds.sums);
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int col = lane & 15, quad = lane >> 4;
    const int c0 = bx * kMmaChannels;
    const int ktiles = (mid + kMmaStep - 1) / kMmaStep;  // steps of the second product
    const int nk = C / kMmaStep;                         // steps of the first product
    const int c4s = C >> 2;                              // vectors of four pooled values per sample
    const bool together = a.lds.w2 != a.lds.w1;

    // ---- weights, as they lie in memory, by `loaders` waves of which this is number w ----
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    // Rows r0 .. r0 + chunk of w1; row r's 16-byte chunk c in place c ^ (r & 15), so that the
    // sixteen rows of an operand spread over the banks.  (A wave's rows are `loaders`, four or
    // eight, loads apart: r & 15 comes round after four or two, the lanes' offsets are constants.)
    auto stage_w1 = [&](int r0, int w, auto loader_waves) __attribute__((always_inline)) {
        constexpr int LOADERS = decltype(loader_waves)::value;
        const int rows = min(a.lds.chunk, mid - r0), chunks = C >> 3;
        const char *base = reinterpret_cast<const char *>(a.w1 + (int64_t)r0 * C);
        const uint32_t to = lds0 + a.lds.w1;
        if (C <= 256) {
            // two rows per load
            constexpr int ROUND = 8 / LOADERS;
            const int hi = lane >> 5;
            int c[ROUND], q0 = w;
#pragma unroll
            for (int i = 0; i < ROUND; ++i) c[i] = (lane & 31) ^ (2 * (w + i * LOADERS) + hi);
            // (whole rounds of rows that fill the lanes: no masks, which cost as many instructions again)
            if (chunks == 32)
                for (; 2 * (q0 + 8 - LOADERS) + 1 < rows; q0 += 8)
#pragma unroll
                    for (int i = 0; i < ROUND; ++i) {
                        const int q = q0 + i * LOADERS;
                        load_to_lds(to + q * 1024, base + q * 1024, (hi * 32 + c[i]) * 16);
                    }
            for (; 2 * q0 < rows; q0 += 8)
#pragma unroll
                for (int i = 0; i < ROUND; ++i) {
                    const int q = q0 + i * LOADERS;
                    if (2 * q + hi < rows && c[i] < chunks)
                        load_to_lds(to + q * 1024, base + q * (C * 4), (hi * chunks + c[i]) * 16);
                }
        } else {
            constexpr int ROUND = 16 / LOADERS;
            const int pieces = a.lds.pitch >> 10;
            for (int piece = 0; piece < pieces; ++piece) {
                int c[ROUND];
#pragma unroll
                for (int i = 0; i < ROUND; ++i) c[i] = (piece * kWave + lane) ^ (w + i * LOADERS);
                int q0 = w;
                if (piece * kWave + kWave <= chunks)
                    for (; q0 + 16 - LOADERS < rows; q0 += 16)
#pragma unroll
                        for (int i = 0; i < ROUND; ++i) {
                            const int r = q0 + i * LOADERS;
                            load_to_lds(to + (r * pieces + piece) * 1024, base + r * (C * 2), c[i] * 16);
                        }
                for (; q0 < rows; q0 += 16)
#pragma unroll
                    for (int i = 0; i < ROUND; ++i) {
                        const int r = q0 + i * LOADERS;
                        if (r < rows && c[i] < chunks)
                            load_to_lds(to + (r * pieces + piece) * 1024, base + r * (C * 2), c[i] * 16);
                    }
            }
        }
    };
    // The KK rows of each of the block's channels: one run of bytes.
    auto stage_w2 = [&](int w, int loaders) __attribute__((always_inline)) {
        const int chunks = kMmaChannels * KK * mid / 8;
        const char *base = reinterpret_cast<const char *>(a.w2 + (int64_t)c0 * KK * mid);
        for (int q = w; q * kWave < chunks; q += loaders)
            if (q * kWave + lane < chunks) load_to_lds(lds0 + a.lds.w2 + q * 1024, base + q * 1024, lane * 16);
    };
    // Half of the waves fetch the weights, the others the pooled vectors and what the threads
    // that normalise will need (the first NORM_WAVES waves, a sample's channel per thread).
    constexpr int kPoolWaves = 4;
    static_assert(kPoolWaves == NORM_WAVES);
    const int zs = tid / kMmaChannels, zc = tid % kMmaChannels;
    struct Values { half8_t v[KK / 8]; _Float16 last; };    // a channel's KK contiguous values of a parameter
    Values gain, offset, bias;
    uint16_t b1v[4];    // biases of a wave's first tile of hidden values
    auto request_bias = [&](int t) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t r = rows::plane_rsrc(a.b1, a.b1 ? (uint32_t)mid * 2u : 0u);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            b1v[e] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (t * 16 + quad * 4 + e) * 2, 0, 0);
    };
    // (hidden values past the last are zero)
    if (tid < kMmaTile / 2) reinterpret_cast<uint32_t *>(hv + (ktiles - 1) * kMmaTile)[tid] = 0u;
    static_assert(kMmaTile / 2 <= kMmaThreads);
    if (wave >= kPoolWaves) {
        stage_w1(0, wave - kPoolWaves, std::integral_constant<int, kMmaWaves - kPoolWaves>{});
        if (together) stage_w2(wave - kPoolWaves, kMmaWaves - kPoolWaves);
        request_bias(wave);
    }
    begin(wave >= kPoolWaves);

    // ---- the pooled vectors: given, or scale * the sum of nparts partial sums per value ----
    // A wave takes a sample, a lane four channels; where there are fewer samples than waves,
    // several waves share a sample's partial sums, which meet in LDS.  (Samples there are only:
    // the other columns of the products are read by nothing.)
    auto put_pooled = [&](int s, int c4, half4_t v) __attribute__((always_inline)) {
        *reinterpret_cast<half4_t *>(pv + ((c4 >> 3) * kMmaSamples + s) * kMmaStep + (c4 & 7) * 4) = v;
        if constexpr (SAVE) {
            if (a.save.pooled && bx == 0) {
#pragma unroll
                for (int e = 0; e < 4; ++e) a.save.pooled[(int64_t)(n0 + s) * C + c4 * 4 + e] = (float)v[e];
            }
        }
    };
    auto scaled = [&](float4_t sum) __attribute__((always_inline)) {
        half4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (_Float16)(sum[e] * a.scale);
        return v;
    };
    const int share = !a.parts || C > kMmaSpread || a.nparts <= kMmaRound ? 1 : ns == 1 ? 4 : ns == 2 ? 2 : 1;
    const int g = wave & (share - 1);    // (this wave's part of a sample's)
    if (wave < kPoolWaves) {
        const int stride = kPoolWaves / share;    // samples at a time
        if (a.parts) {
            // (a sample at a time behind a descriptor: beyond its partial sums there are zeros.  The row is in the lane's
            // offset: a scalar one is left out of the range check)
            const uint32_t bytes = (uint32_t)(a.nparts * C) * 4u, row = (uint32_t)(share * C) * 4u;
            auto sample = [&](int s) __attribute__((always_inline)) {
                return rows::plane_rsrc(a.parts + (int64_t)(n0 + min(s, ns - 1)) * a.nparts * C, s < ns ? bytes : 0u);
            };
            for (int s = wave / share; s < ns; s += 2 * stride) {
                const __amdgpu_buffer_rsrc_t r[2] = {sample(s), sample(s + stride)};
                for (int c4 = lane; c4 < c4s; c4 += kWave) {
                    float4_t sum[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
                    uint32_t at = (uint32_t)(g * C + c4 * 4) * 4u;
                    for (int q0 = g; q0 < a.nparts; q0 += kMmaRound * share) {
                        float4_t x[2][kMmaRound];
#pragma unroll
                        for (int u = 0; u < kMmaRound; ++u, at += row)
#pragma unroll
                            for (int i = 0; i < 2; ++i)
                                x[i][u] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(r[i], (int)at, 0, 0));
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int i = 0; i < 2; ++i)
                            sum[i] += ((x[i][0] + x[i][1]) + (x[i][2] + x[i][3])) + ((x[i][4] + x[i][5]) + (x[i][6] + x[i][7]));
                    }
                    if (share > 1) {    // (one sample per wave, one round of channels at most)
                        ps[wave * kWave + lane] = sum[0];
                    } else {
                        put_pooled(s, c4, scaled(sum[0]));
                        if (s + stride < ns) put_pooled(s + stride, c4, scaled(sum[1]));
                    }
                }
            }
        } else {
            for (int s = wave; s < ns; s += kPoolWaves)
                for (int c4 = lane; c4 < c4s; c4 += kWave)
                    put_pooled(s, c4, *reinterpret_cast<const half4_t *>(a.pooled + (int64_t)(n0 + s) * C + c4 * 4));
        }
        auto get = [&](const __half *p, Values &to) __attribute__((always_inline)) {
            // (no such parameter: anything that is there, C * KK values of it at least)
            const __half *at = (p ? p : a.w2) + (int64_t)c0 * KK + (uint32_t)(zc * KK);
#pragma unroll
            for (int k = 0; k < KK / 8; ++k) __builtin_memcpy(&to.v[k], at + k * 8, sizeof(half8_t));
            __builtin_memcpy(&to.last, at + KK - 1, 2);
        };
        request_bias(wave);
        get(a.gain_vec, gain);
        get(a.offset_vec, offset);
        get(a.b2, bias);
    }
    if (share > 1) {
        __syncthreads();
        if (wave < kPoolWaves && g == 0 && wave / share < ns && lane < c4s) {
            float4_t x[kPoolWaves], sum = ps[wave * kWave + lane];
#pragma unroll
            for (int k = 1; k < kPoolWaves; ++k) x[k] = ps[min(wave + k, kPoolWaves - 1) * kWave + lane];
#pragma unroll
            for (int k = 1; k < kPoolWaves; ++k)
                if (k < share) sum += x[k];
            put_pooled(wave / share, lane, scaled(sum));
        }
    }
    meanwhile(wave >= kPoolWaves);
    if (wave >= kPoolWaves) loads_to_lds_done();
    __syncthreads();

    // ---- hidden layer: tiles of sixteen rows of w1 dealt out to the waves ----
    for (int r0 = 0; r0 < mid; r0 += a.lds.chunk) {
        if (r0 > 0) {
            __syncthreads();
            stage_w1(r0, wave, std::integral_constant<int, kMmaWaves>{});
            loads_to_lds_done();
            __syncthreads();
        }
        const int rend = min(r0 + a.lds.chunk, mid);
        for (int t = r0 / 16 + wave; t * 16 < rend; t += kMmaWaves) {
            if (t != wave) request_bias(t);
            const unsigned char *arow = w1s + (t * 16 + col - r0) * a.lds.pitch;
            const _Float16 *brow = pv + min(col, ns - 1) * kMmaStep + quad * 8;    // (columns past the last: not used; fewer rows, fewer conflicts)
            float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            constexpr int U = 8;
#pragma unroll 1
            for (int k0 = 0; k0 < nk; k0 += U) {
                half8_t av[U], bv[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int k = min(k0 + u, nk - 1);
                    av[u] = *reinterpret_cast<const half8_t *>(arow + ((k * 4 + quad) ^ col) * 16);
                    bv[u] = *reinterpret_cast<const half8_t *>(brow + k * kMmaTile);
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (k0 + u < nk) acc[u & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[u], bv[u], acc[u & 1], 0, 0, 0);
            }
            // (rows past the last: zero)
            half4_t h;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t bias = b1v[e];
                asm volatile("" : "+v"(bias));    // (converted here, not where it is asked for, which would be a wait there)
                const float v = relu(acc[0][e] + acc[1][e] + (float)__builtin_bit_cast(_Float16, (uint16_t)bias));
                h[e] = t * 16 + quad * 4 + e < mid ? (_Float16)v : (_Float16)0;
            }
            *reinterpret_cast<half4_t *>(hv + ((t >> 1) * kMmaSamples + col) * kMmaStep + (t & 1) * 16 + quad * 4) = h;
            if constexpr (SAVE) {
                if (a.save.hidden && bx == 0 && col < ns) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int m = t * 16 + quad * 4 + e;
                        if (m < mid) a.save.hidden[(int64_t)(n0 + col) * mid + m] = (float)h[e];
                    }
                }
            }
        }
    }
    after();
    __syncthreads();
    if (!together && a.lds.stage_w2) {
        stage_w2(wave, kMmaWaves);
        loads_to_lds_done();
        __syncthreads();
    }

    // ---- taps: TPW taps of sixteen channels and samples per wave ----
    float4_t acc[TPW];
    if (wave < TAP_WAVES) {
#pragma unroll
        for (int j = 0; j < TPW; ++j) acc[j] = float4_t{0.f, 0.f, 0.f, 0.f};
        const _Float16 *brow = hv + col * kMmaStep + quad * 8;
        // (a tap past the last: the last again, not used)
        uint32_t at[TPW];    // first of the lane's values in the row of channel col, tap j: halves
#pragma unroll
        for (int j = 0; j < TPW; ++j) at[j] = (uint32_t)((col * KK + min(wave * TPW + j, KK - 1)) * mid + quad * 8);
        // Values t * 32 .. + 8 of them.  The row's last step ends with values of the next row
        // (staged: whatever follows), which are made zero: times zero a NaN would stay one.
        auto cut = [&](half8_t &v, int t) __attribute__((always_inline)) {
            const int left = mid - t * kMmaStep - quad * 8;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (e >= left) v[e] = (_Float16)0;
        };
        auto staged = [&](int j, int t) __attribute__((always_inline)) {
            // eight values from any even byte on: five words, shifted by half a word or not
            const uint32_t *p = reinterpret_cast<const uint32_t *>(w2s + (at[j] * 2u & ~3u)) + t * (kMmaStep / 2);
            const uint32_t by = (at[j] & 1u) * 16u;
            uint4 q;
            q.x = __builtin_amdgcn_alignbit(p[1], p[0], by);
            q.y = __builtin_amdgcn_alignbit(p[2], p[1], by);
            q.z = __builtin_amdgcn_alignbit(p[3], p[2], by);
            q.w = __builtin_amdgcn_alignbit(p[4], p[3], by);
            return __builtin_bit_cast(half8_t, q);
        };
        auto step = [&](int t, half8_t (&w)[TPW]) __attribute__((always_inline)) {
            const half8_t b = *reinterpret_cast<const half8_t *>(brow + t * kMmaTile);
#pragma unroll
            for (int j = 0; j < TPW; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[j], b, acc[j], 0, 0, 0);
        };
        if (a.lds.stage_w2) {
            int t = 0;
#pragma unroll 1
            for (; t + 2 < ktiles; t += 2) {
                half8_t w[2][TPW];
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < TPW; ++j) w[i][j] = staged(j, t + i);
                step(t, w[0]);
                step(t + 1, w[1]);
            }
            if (t + 1 < ktiles) {
                half8_t w[TPW];
#pragma unroll
                for (int j = 0; j < TPW; ++j) w[j] = staged(j, t);
                step(t++, w);
            }
            half8_t w[TPW];
#pragma unroll
            for (int j = 0; j < TPW; ++j) {
                w[j] = staged(j, t);
                cut(w[j], t);
            }
            step(t, w);
        } else {
            const __half *base = a.w2 + (int64_t)c0 * KK * mid;
#pragma unroll 1
            for (int t = 0; t < ktiles; ++t) {
                half8_t w[TPW];
#pragma unroll
                for (int j = 0; j < TPW; ++j) {
                    if (t + 1 < ktiles) {
                        __builtin_memcpy(&w[j], base + at[j] + t * kMmaStep, sizeof(w[j]));
                    } else {
                        const int left = mid - t * kMmaStep - quad * 8;
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            w[j][e] = e < left ? *reinterpret_cast<const _Float16 *>(base + at[j] + t * kMmaStep + e) : (_Float16)0;
                    }
                }
                step(t, w);
            }
        }
    }
    if (a.lds.shared) __syncthreads();
    if (wave < TAP_WAVES) {
#pragma unroll
        for (int j = 0; j < TPW; ++j)
            if (wave * TPW + j < KK) {
#pragma unroll
                for (int e = 0; e < 4; ++e) z[col * ZP + (quad * 4 + e) * KK + wave * TPW + j] = acc[j][e];
            }
    }
    __syncthreads();
    if (wave >= NORM_WAVES || zs >= ns) return;
    float u[KK];
    TapParams<__half, KK> params;
#pragma unroll
    for (int j = 0; j < KK; ++j) {
        auto value = [&](const Values &p) __attribute__((always_inline)) { return (float)(j < KK - 1 ? p.v[j / 8][j % 8] : p.last); };
        u[j] = z[zs * ZP + zc * KK + j];
        params.gain[j] = a.gain_vec ? value(gain) : a.gain;
        params.offset[j] = a.offset_vec ? value(offset) : 0.f;
        params.bias[j] = a.b2 ? value(bias) : 0.f;
    }
    const int64_t to = ((int64_t)(n0 + zs) * C + c0 + zc) * KK;
    if constexpr (SAVE) {
        if (a.save.taps) {
#pragma unroll
            for (int j = 0; j < KK; ++j) a.save.taps[to + j] = u[j] + params.bias[j];
        }
    }
    normalise<__half, KK>(u, params);
    sink(n0 + zs, c0 + zc, u);
}

#endif  // __HIPCC__

// ---- one sample per workgroup, on the vector ALU (3 x 3 taps) ----------------------------
// A workgroup of sixteen waves takes one sample and `block` channels.  All of w1 and the block's
// rows of w2 come into LDS as runs of bytes, requested by one half of the waves while the other
// adds up the pooled vector; sixteen lanes then take a row, four rows a wave at a time.  Read
// straight from memory by those lanes, a row is 32 or 64 bytes per load: 880 loads of a quarter
// KB for 256 fp32 channels, which is what the launch waited for, where 110 of 1 KB do.  Sums
// and what passes between the layers are fp32.  us a launch, straight from memory / now: fp32,
// samples x channels, 32 x 256 7.9 / 5.1, 8 x 512 24.5 / 8.6, 64 x 128 6.1 / 4.2; fp16, 128 x 128
// 6.3 / 5.1, 32 x 432 16.8 / 9.1; 8 x 64 with 118 partial sums per value 15.2 / 5.1.
constexpr int kRowsKK = 9;
constexpr int kRowsThreads = 1024, kRowsWaves = kRowsThreads / kWave, kRowsPoolWaves = kRowsWaves / 2;
constexpr int kRowsMaxBlock = 64;

template <typename T>
struct ChannelRows {
    const T *pooled, *w1, *b1, *w2, *b2;
    T *cf;
    int N, C, mid;
    float gain;
    const T *gain_vec, *offset_vec;
    const float *parts;    // (nparts per sample; null: `pooled`)
    int nparts;
    float scale;
    ChannelSave save;
    // LDS, bytes: pooled vector, hidden vector, taps, partial sums | w1 by `chunk` rows | the
    // first `early` of the block's rows of w2, the others where w1 was
    int block, chunk, early, w1_at, w2_at, total;
    // waves that have a value of the pooled vector per lane, that share a value's partial sums, both; 256 / width, rounded up
    int width, share, pool_waves, width_magic;
};
// The layout for blocks of `block` channels; false: rows too long.
template <typename T>
inline bool channel_rows_lds(ChannelRows<T> &a, int block) {
    const int64_t row1 = (int64_t)a.C * sizeof(T), row2 = (int64_t)a.mid * sizeof(T), rows = (int64_t)block * kRowsKK;
    a.block = block;
    a.width = (a.C + kWave - 1) / kWave;
    a.share = a.parts && a.nparts > kMmaRound && a.width <= kRowsPoolWaves / 2 ? kRowsPoolWaves / a.width : 1;
    a.pool_waves = std::min(a.width * a.share, kRowsPoolWaves);
    a.width_magic = (256 + a.width - 1) / a.width;
    a.w1_at = mma_round(((int64_t)a.C + a.mid + rows + kRowsPoolWaves * kWave) * 4);
    const int64_t left = kMmaLds - a.w1_at - 32;
    if (left < 8 * row1) return false;
    // (parts of eight rows are whole 16 bytes)
    a.chunk = a.mid * row1 <= left ? a.mid : (int)(left / row1 / 8 * 8);
    const int64_t w1 = mma_round(a.chunk * row1);
    a.early = (int)std::min(rows, std::max<int64_t>((left - w1) / row2, 0) / 8 * 8);
    a.w2_at = a.w1_at + (int)w1;
    a.total = a.w2_at + mma_round(a.early * row2);
    return (rows - a.early) * row2 <= w1;
}
// Blocks of 16, 32 or 64 channels: the smallest that give every compute unit one workgroup at
// most.  False: not covered.  (Where there are more workgroups, loads that serve several samples
// are faster: 512 x 64 fp32 6.4 us and 9.6 here, 128 x 256 12.8 and 16.2, 48 x 432 fp16 20.5 and
// 19.3.  Weights must be whole 16 bytes from their start on.)
template <typename T>
inline bool channel_rows_plan(ChannelRows<T> &a) {
    auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (!aligned(a.w1) || !aligned(a.w2) || a.mid < 1 || a.C < 1) return false;
    if ((int64_t)a.C * a.mid * kRowsKK * (int64_t)sizeof(T) >= ((int64_t)1 << 31)) return false;
    for (int block = 16; block <= kRowsMaxBlock; block *= 2)
        if ((int64_t)a.N * ((a.C + block - 1) / block) <= 256) return channel_rows_lds(a, block);
    return false;
}

// Partial sums per pooled value that the channel branch is left (3 x 3 taps).  Every workgroup adds
// up those of its samples, in rounds of kMmaRound requests per lane with a round trip to memory
// each; `spare` rounds more than one value takes are cheaper than a launch that makes totals of them.
// us, kept as they are less totals first, medians over 668 sizes: matrix cores 4 rounds more -0.5, 6
// -0.1, 8 +1.2, 16 +5.9; rows 4 -0.9, 6 0.0, 8 +1.5, 16 +5.3; k_channel_branch 2 -0.9, 3 +0.4, 6 +1.8.
// (8 x 64 x 200 x 300 fp16, 118 sums: 21.8 kept, 24.9 with totals.)
inline int64_t channel_parts_left(int64_t N, int64_t C, int64_t mid, int esz) {
    auto div = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
    const int64_t width = div(C, kWave);
    int64_t share = 1, trips, spare;           // waves that share a value's sums, round trips per round
    if (esz == 2 && channel_mma_covers(C, mid, kRowsKK)) {
        const int64_t ns = std::min<int64_t>(N, kMmaSamples);
        share = C > kMmaSpread || ns > 2 ? 1 : 4 / ns;
        trips = div(C, 4 * kWave) * div(div(ns * share, 4), 2);
        spare = 5;
    } else if (N * div(C, kRowsMaxBlock) <= 256) {
        share = width <= kRowsPoolWaves / 2 ? kRowsPoolWaves / width : 1;
        trips = div(width * share, kRowsPoolWaves);
        spare = 6;
    } else {
        const int64_t values = std::max<int64_t>(std::min<int64_t>(N * width / 256, 4), 1) * C;
        share = std::max<int64_t>(kRowsThreads / values, 1);
        trips = div(values, kRowsThreads);
        spare = 3;
    }
    return kMmaRound * share * ((spare + trips) / trips);
}

#ifdef __HIPCC__

// Butterfly steps through the VALU's lane-permute path.  (Shuffles through the
// LDS crossbar cost a round trip each and made these kernels several times slower.)
template <int CTRL>
__device__ __forceinline__ float add_permuted(float x) {
    return x + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, true));
}
// Sum over each row of 16 lanes (the same value in every lane of the row).
__device__ __forceinline__ float row_sum(float v) {
    v = add_permuted<0xB1>(v);    // quad_perm [1,0,3,2]
    v = add_permuted<0x4E>(v);    // quad_perm [2,3,0,1]
    v = add_permuted<0x141>(v);   // row_half_mirror
    return add_permuted<0x140>(v);   // row_mirror
}


// Block bx of sample n's channels, kRowsThreads threads.
template <typename T, bool SAVE, typename Begin, typename Meanwhile, typename After, typename Sink>
__device__ __forceinline__ void channel_rows(const ChannelRows<T> &a, int bx, int64_t n, unsigned char *smem,
                                             const Begin &begin, const Meanwhile &meanwhile, const After &after, const Sink &sink) {
    constexpr int KK = kRowsKK, VE = 16 / sizeof(T);
    at_once(a.w1, a.w2, a.parts, a.b1, a.C, a.mid, a.nparts, a.block, a.w1_at, a.w2_at, a.chunk, a.early);
    at_once(a.gain_vec, a.offset_vec, a.b2, a.width, a.share, a.pool_waves, a.width_magic, a.scale);
    const int C = a.C, mid = a.mid;
    float *v = reinterpret_cast<float *>(smem);     // [C]
    float *h = v + C;                               // [mid]
    float *f = h + mid;                             // [block * KK]
    float *sums = f + a.block * KK;                 // [pool waves][64]
    const T *w1s = reinterpret_cast<const T *>(smem + a.w1_at), *w2s = reinterpret_cast<const T *>(smem + a.w2_at);
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int cb = bx * a.block, channels = min(a.block, C - cb), rows = channels * KK;
    const int early = min(a.early, rows);           // rows of w2 that come in with w1
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;

    // `count` values from `from` (whole 16 bytes into its tensor) on to LDS, by `loaders` waves
    // of which this is number w; the last ones that fill no 16 bytes one by one.
    auto stage = [&](const T *from, int count, int to, int w, int loaders) __attribute__((always_inline)) {
        const char *base = reinterpret_cast<const char *>(from);
        const int chunks = count / VE, whole = chunks / kWave;
        int q = w;
        for (; q < whole; q += loaders) load_to_lds(lds0 + to + q * 1024, base + q * 1024, lane * 16);
        if (q == whole) {
            if (q * kWave + lane < chunks) load_to_lds(lds0 + to + q * 1024, base + q * 1024, lane * 16);
            const int at = chunks * VE + lane;
            if (at < count) *reinterpret_cast<T *>(smem + to + at * (int)sizeof(T)) = from[at];
        }
    };
    // a channel's KK contiguous values of a parameter, in 16 bytes at a time and the last one
    typedef typename std::conditional<sizeof(T) == 2, _Float16, float>::type raw_t;
    typedef raw_t vec_t __attribute__((ext_vector_type(VE)));
    static_assert(KK % VE == 1);
    struct Values {
        vec_t v[KK / VE];
        raw_t last;
        __device__ __forceinline__ float at(int j) const { return (float)(j < KK - 1 ? v[j / VE][j % VE] : last); }
    };
    Values gain, offset, bias;
    // (a lane of the first waves takes a channel of the pooled vector; of many partial sums several
    // waves share a channel's; the others fetch the weights)
    const int width = a.width, share = a.share, pool_waves = a.pool_waves;
    if (wave >= pool_waves) {
        stage(a.w1, min(a.chunk, mid) * C, a.w1_at, wave - pool_waves, kRowsWaves - pool_waves);
        stage(a.w2 + (int64_t)cb * KK * mid, early * mid, a.w2_at, wave - pool_waves, kRowsWaves - pool_waves);
    }

    begin(wave >= pool_waves);

    const int seg = lane >> 4, sl = lane & 15;
    // (behind a descriptor that holds nothing where there is no bias: a branch would be waited in)
    float b1_first;
    {
        const __amdgpu_buffer_rsrc_t r = rows::plane_rsrc(a.b1, a.b1 ? (uint32_t)(mid * sizeof(T)) : 0u);
        const int at = min(wave * 4 + seg, mid - 1) * (int)sizeof(T);
        if constexpr (sizeof(T) == 2) b1_first = (float)__builtin_bit_cast(_Float16, (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, at, 0, 0));
        else b1_first = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0));
    }

    // The pooled vector: given, or scale * the sum of nparts partial sums per value.
    const int g = (wave * a.width_magic) >> 8;      // (used where width is four at most: wave / width)
    if (wave < pool_waves) {
        auto put = [&](int c, float x) __attribute__((always_inline)) {
            v[c] = x;
            if constexpr (SAVE) {
                if (a.save.pooled && bx == 0) a.save.pooled[n * C + c] = x;
            }
        };
        if (a.parts) {
            const __amdgpu_buffer_rsrc_t r = rows::plane_rsrc(a.parts + n * a.nparts * C, (uint32_t)(a.nparts * C) * 4u);
            for (int c = (share > 1 ? wave - g * width : wave) * kWave + lane; c < width * kWave;
                 c += kRowsPoolWaves * kWave) {
                float sum = 0.f;
                for (int q0 = share > 1 ? g : 0; q0 < a.nparts; q0 += kMmaRound * share) {
                    float x[kMmaRound];    // (beyond the last: zeros)
#pragma unroll
                    for (int u = 0; u < kMmaRound; ++u) {
                        const int q = q0 + u * share;
                        x[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                            r, c < C && q < a.nparts ? c * 4 : (int)rows::kOutside, q * C * 4, 0));
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    sum += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
                }
                if (share > 1) sums[wave * kWave + lane] = sum;
                else if (c < C) put(c, sum * a.scale);
            }
        } else {
            for (int c = tid; c < C; c += pool_waves * kWave) put(c, ld(a.pooled + n * C + c));
        }
        // gains, offsets and biases of the channel that the thread normalises
        if (tid < channels) {
            // (no such parameter: anything that is there, C * KK values of it at least.  Under a branch each, and in
            // single values, they took a trip to memory in front of the barrier.)
            const int64_t at = (int64_t)(cb + tid) * KK;
            auto get = [&](const T *p, Values &to) __attribute__((always_inline)) {
                const T *from = (p ? p : a.w2) + at;
#pragma unroll
                for (int k = 0; k < KK / VE; ++k) __builtin_memcpy(&to.v[k], from + k * VE, sizeof(vec_t));
                __builtin_memcpy(&to.last, from + KK - 1, sizeof(raw_t));
            };
            get(a.gain_vec, gain);
            get(a.offset_vec, offset);
            get(a.b2, bias);
        }
    }
    if (share > 1) {
        __syncthreads();
        if (wave < width && tid < C) {
            float x[kRowsPoolWaves];
#pragma unroll
            for (int k = 0; k < kRowsPoolWaves; ++k) x[k] = sums[min(k * width + wave, kRowsPoolWaves - 1) * kWave + lane];
            float sum = x[0];
#pragma unroll
            for (int k = 1; k < kRowsPoolWaves; ++k) sum += k < share ? x[k] : 0.f;
            v[tid] = sum * a.scale;
            if constexpr (SAVE) {
                if (a.save.pooled && bx == 0) a.save.pooled[n * C + tid] = sum * a.scale;
            }
        }
    }
    meanwhile(wave >= pool_waves);
    if (wave >= pool_waves) loads_to_lds_done();
    __syncthreads();

    // ---- hidden vector: rows of w1, sixteen lanes each ----
    for (int r0 = 0; r0 < mid; r0 += a.chunk) {
        if (r0 > 0) {
            __syncthreads();
            stage(a.w1 + (int64_t)r0 * C, min(a.chunk, mid - r0) * C, a.w1_at, wave, kRowsWaves);
            loads_to_lds_done();
            __syncthreads();
        }
        const int rend = min(r0 + a.chunk, mid);
        for (int m0 = r0 + wave * 4; m0 < rend; m0 += kRowsWaves * 4) {
            const int m = min(m0 + seg, rend - 1);
            const float b = m0 == wave * 4 ? b1_first : a.b1 ? ld(a.b1 + m) : 0.f;
            const T *row = w1s + (m - r0) * C;
            float p = 0.f;
            if (C % VE == 0) {
                const int vectors = C / VE;
#pragma unroll 2
                for (int j = sl; j < vectors; j += 16) {
                    T w[VE];
                    float x[VE];
                    __builtin_memcpy(w, __builtin_assume_aligned(row + j * VE, 16), sizeof(w));
#pragma unroll
                    for (int e = 0; e < VE; e += 4)
                        __builtin_memcpy(x + e, __builtin_assume_aligned(v + j * VE + e, 16), 16);
#pragma unroll
                    for (int e = 0; e < VE; ++e) p = fmaf(ld(&w[e]), x[e], p);
                }
            } else {
#pragma unroll 4
                for (int c = sl; c < C; c += 16) p = fmaf(ld(row + c), v[c], p);
            }
            const float hm = relu(row_sum(p) + b);
            if (sl == 0 && m0 + seg < rend) {
                h[m] = hm;
                if constexpr (SAVE) {
                    if (a.save.hidden && bx == 0) a.save.hidden[n * mid + m] = hm;
                }
            }
        }
    }
    after();
    __syncthreads();
    if (early < rows) stage(a.w2 + ((int64_t)cb * KK + early) * mid, (rows - early) * mid, a.w1_at, wave, kRowsWaves);

    // ---- taps: rows of w2, the lane's values of the hidden vector in registers ----
    // NI: values per lane, G: rows at a time (no value is read under a branch: it would be waited
    // for alone)
    auto taps_of = [&](auto ni, const T *first, int from, int to) __attribute__((always_inline)) {
        constexpr int NI = decltype(ni)::value, G = NI >= 8 ? 1 : 8 / NI;
        float hm[NI];
        int at[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            at[i] = min(sl + i * 16, mid - 1);
            hm[i] = h[at[i]];
        }
        for (int r0 = from + wave * 4; r0 < to; r0 += G * kRowsWaves * 4) {
            float x[G][NI];
#pragma unroll
            for (int k = 0; k < G; ++k) {
                const T *row = first + (min(r0 + k * kRowsWaves * 4 + seg, to - 1) - from) * mid;
#pragma unroll
                for (int i = 0; i < NI; ++i) x[k][i] = ld(row + at[i]);
            }
#pragma unroll
            for (int k = 0; k < G; ++k) {
                float p = 0.f;
#pragma unroll
                for (int i = 0; i < NI; ++i) p = fmaf(sl + i * 16 < mid ? x[k][i] : 0.f, hm[i], p);
                if (NI == 8)
                    for (int m = sl + NI * 16; m < mid; m += 16)
                        p = fmaf(ld(first + (min(r0 + seg, to - 1) - from) * mid + m), h[m], p);
                const float tot = row_sum(p);
                const int r = r0 + k * kRowsWaves * 4 + seg;
                if (sl == 0 && r < to) f[r] = tot;
            }
        }
    };
    auto taps = [&](const T *first, int from, int to) __attribute__((always_inline)) {
        if (mid <= 16) taps_of(std::integral_constant<int, 1>{}, first, from, to);
        else if (mid <= 32) taps_of(std::integral_constant<int, 2>{}, first, from, to);
        else if (mid <= 64) taps_of(std::integral_constant<int, 4>{}, first, from, to);
        else taps_of(std::integral_constant<int, 8>{}, first, from, to);
    };
    taps(w2s, 0, early);
    if (early < rows) {
        loads_to_lds_done();
        __syncthreads();
        taps(w1s, early, rows);
    }
    __syncthreads();
    if (tid >= channels) return;
    float u[KK];
    TapParams<T, KK> params;
#pragma unroll
    for (int j = 0; j < KK; ++j) {
        u[j] = f[tid * KK + j];
        params.gain[j] = a.gain_vec ? gain.at(j) : a.gain;
        params.offset[j] = a.offset_vec ? offset.at(j) : 0.f;
        params.bias[j] = a.b2 ? bias.at(j) : 0.f;
    }
    const int64_t to = (n * C + cb + tid) * KK;
    if constexpr (SAVE) {
        if (a.save.taps) {
#pragma unroll
            for (int j = 0; j < KK; ++j) a.save.taps[to + j] = u[j] + params.bias[j];
        }
    }
    normalise<T, KK>(u, params);
    sink(n, cb + tid, u);
}

#endif  // __HIPCC__

}  // namespace ddf

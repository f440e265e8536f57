// Gradients of the two filter branches of DDFPack (3 x 3 taps), given the gradients of
// the filters they predict: what autograd derives in the reference from
// build_spatial_branch / build_channel_branch (ddf/ddf.py:176-192) behind the operator's
// backward pass.  With dZ2 the gradient of the channel branch's un-normalised taps (dCF
// through the normalisation), h / v its hidden and pooled vectors and dR the gradient of
// the spatial branch's un-normalised taps:
//
//   dW2 = sum_n dZ2 (x) h      db2 = sum_n dZ2      dgain = sum_n dCF * z      dh = W2^T dZ2
//   dz1 = dh where h > 0       dW1 = sum_n dz1 (x) v    db1 = sum_n dz1        dv = W1^T dz1
//   dWs[t, c] = sum_{n, p} dR[n, t, p] x[n, c, p*s]     dbs[t] = sum_{n, p} dR[n, t, p]
//   dX[n, c, q] += sum_t Ws[t, c] dR[n, t, q/s] + dv[n, c] / (H*W)
//
// Four launches; independent pieces share one (a launch costs the host more than the
// small pieces cost the GPU):
//   k_pack_fc2     dW2, db2, dgain, partial dh   |  partial dWs, dbs (matrix cores)
//   k_pack_hidden  dz1                           |  dWs, dbs
//   k_pack_fc1     dW1, db1                      |  dv
//   k_pack_dx      dX
// Through the convolution library, torch's reductions and element-wise launches the same
// took some twenty launches: a training step of a 64 x 128 x 28 x 28 fp16 layer spent
// 0.7 ms, nearly all of it on the host.
// Sums are fp32 throughout, added in a fixed order (no atomics).
#include <algorithm>

#include "ddf_common.h"

namespace ddf {
namespace {

constexpr int KK = 9;
constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

struct PackDims {
    int N, C, mid, H, W, Ho, Wo, s, head;
};

// ---- second convolution of the channel branch --------------------------------
// A workgroup takes CW channels (9 * CW rows of W2) and 64 hidden values, a lane one
// hidden value; samples come in chunks of 64 through LDS.  dW2: every wave owns one channel's
// rows for a CW-th quarter of the samples and reads their dZ2 as LDS broadcasts; dh: every wave owns
// every fourth sample, with the lane's column of the rows of W2 in registers.  LDS reads bound it (a
// wave's 36 multiply-adds of a sample are nine reads of 16 bytes) and, behind them, the chain from the
// first load over the normalisation to the last sum: everything is asked for before anything is waited for
// (W2's rows, the gains and the hidden values under conditions, one after another, cost 2 us; W2's rows first, their
// addresses would not fit the registers of four waves per SIMD behind the others).
constexpr int kFc2Samples = 64, kFc2MaxChannels = kWaves, kUnits = 256;    // (compute units)
constexpr int kFc2Pitch = 12;    // a channel's nine values, 16-byte rows

// Channels per workgroup: one or two as long as the workgroups do not outnumber the compute units, else four.  Every channel block
// leaves a partial dh of all samples, so no more of them than fill the chip where there is a choice.  The launch with four channels
// each and this, us (fp16, medians under the profiler): 64 x 128 x 28 x 28 18.2 / 8.8, 64 x 64 x 56 x 56 19.4 / 8.8, 64 x 256 x 14 x 14 17.6 / 8.5, 256 x 128 x
// 14 x 14 55.4 / 19.6, 1 x 512 x 14 x 14 6.4 / 5.8, fp32 32 x 256 x 28 x 28 15.0 / 10.4; four of them with the loads asked for at once: 64 x 512 x 7 x 7
// 18.9 / 13.6, 3 x 2048 x 7 x 7 31.8 / 23.9.  (8 x 64 x 200 x 300, whose time is the other half's: 13.0 / 13.7.)
// Batches whose parts would pass 64 MB, 25 us to write and read again at a copy's rate, take more channels: one or two of them never ask for more
// workspace than that.  Four are the most (registers), and their parts grow with the batch: 256 x 2048 with 512 hidden values 256 MB.
constexpr int64_t kFc2MostParts = 1 << 24;
inline int fc2_channels(int64_t N, int64_t C, int64_t mid) {
    int cw = 1;
    while (cw < kFc2MaxChannels && (cdiv(C, cw) * cdiv(mid, kWave) > kUnits || cdiv(C, cw) * N * mid > kFc2MostParts)) cw *= 2;
    return cw;
}

template <typename T>
struct Fc2Args {
    const T *dcf, *w2, *gain_vec;
    float gain;
    const float *taps, *hidden;
    T *dw2, *db2, *dgain;
    float *dh_part;     // [channel block][N][mid]
    int mchunks;
};

template <int CW>
struct Fc2Smem {
    static constexpr int rows = CW * KK, parts = kWaves / CW;
    float dz[kFc2Samples][CW][kFc2Pitch];
    float dg[kFc2Samples][rows];
    union {
        float h[kFc2Samples][kWave];
        struct { float dw[kWaves][KK][kWave], col[parts][2 * rows]; } sums;    // at the end
    };
};

template <typename T, int CW>
__device__ __forceinline__ void fc2_block(const PackDims &d, const Fc2Args<T> &a, int block, Fc2Smem<CW> &sm) {
    constexpr int ROWS = Fc2Smem<CW>::rows, PARTS = Fc2Smem<CW>::parts, PASSES = kFc2Samples / kWaves;
    constexpr int HELD = CW < 4 ? PASSES : 4;    // (four channels' weights leave few registers)
    static_assert(2 * ROWS * PARTS <= kThreads && CW * kFc2Samples <= kThreads);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int blk = block / a.mchunks, m0 = (block - blk * a.mchunks) * kWave;
    const int cb = blk * CW;
    const int rows = min(ROWS, (d.C - cb) * KK);
    const int m = m0 + lane;
    const bool mok = m < d.mid;
    const int mc = mok ? m : d.mid - 1;
    float acc[KK];
#pragma unroll
    for (int t = 0; t < KK; ++t) acc[t] = 0.f;
    float col_sum = 0.f;
    const int item_n = threadIdx.x / CW, item_c = threadIdx.x % CW, wc = wave % CW, part = wave / CW;
    const int col_part = threadIdx.x / (2 * ROWS), col_at = threadIdx.x % (2 * ROWS);
    const bool col_mine = m0 == 0 && col_part < PARTS;
    float w2[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) w2[r] = ld(a.w2 + ((int64_t)cb * KK + min(r, rows - 1)) * d.mid + mc);
    for (int n0 = 0; n0 < d.N; n0 += kFc2Samples) {
        const int cnt = min(kFc2Samples, d.N - n0);
        // (addresses clamped instead of loads under conditions, which would wait for one another)
        const int n = min(n0 + item_n, d.N - 1), c = min(cb + item_c, d.C - 1);
        const int64_t at = ((int64_t)n * d.C + c) * KK;
        float z[KK], dc[KK], gain[KK], held[HELD];
        auto hold = [&](int first) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < HELD; ++k) held[k] = a.hidden[(int64_t)(n0 + min(wave + (first + k) * kWaves, cnt - 1)) * d.mid + mc];
        };
#pragma unroll
        for (int t = 0; t < KK; ++t) {
            z[t] = a.taps[at + t];
            dc[t] = ld(a.dcf + at + t);
        }
#pragma unroll
        for (int t = 0; t < KK; ++t) gain[t] = a.gain;
        if (a.gain_vec) {
#pragma unroll
            for (int t = 0; t < KK; ++t) gain[t] = ld(a.gain_vec + c * KK + t);
        }
        if (HELD == PASSES) hold(0);
        if (n0 > 0) __syncthreads();    // (the chunk before has been read)
        if (item_n < kFc2Samples) {
            // one filter per thread: dCF through the normalisation (see ddf_filter_norm.hip)
            const bool there = n0 + item_n < d.N && cb + item_c < d.C;
            float g[KK], sum = 0.f;
#pragma unroll
            for (int t = 0; t < KK; ++t) {
                g[t] = dc[t] * gain[t];
                sum += z[t];
            }
            const float mean = sum / (float)KK;
            float sq = 0.f, s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int t = 0; t < KK; ++t) {
                z[t] -= mean;
                sq += z[t] * z[t];
                s1 += g[t];
                s2 += g[t] * z[t];
            }
            const float sd = sqrtf(sq / (float)(KK - 1));
            const float inv = 1.f / (sd + 1e-10f);
            const float m1 = s1 / (float)KK, k2 = inv * inv * s2 / (sd * (float)(KK - 1));
#pragma unroll
            for (int t = 0; t < KK; ++t) {
                sm.dz[item_n][item_c][t] = there ? inv * (g[t] - m1) - z[t] * k2 : 0.f;
                sm.dg[item_n][item_c * KK + t] = there ? dc[t] * z[t] * inv : 0.f;
            }
        }
        for (int first = 0; first < PASSES; first += HELD) {
            if (HELD < PASSES && first * kWaves >= cnt) break;
            if (HELD < PASSES) hold(first);
#pragma unroll
            for (int k = 0; k < HELD; ++k) sm.h[wave + (first + k) * kWaves][lane] = held[k];
        }
        __syncthreads();
#pragma unroll 4
        for (int i = part; i < cnt; i += PARTS) {
            const float hv = sm.h[i][lane];
#pragma unroll
            for (int t = 0; t < KK; ++t) acc[t] = fmaf(sm.dz[i][wc][t], hv, acc[t]);
        }
#pragma unroll 2
        for (int i = wave; i < cnt; i += kWaves) {
            float p[CW];
#pragma unroll
            for (int c = 0; c < CW; ++c) {
                p[c] = 0.f;
#pragma unroll
                for (int t = 0; t < KK; ++t) p[c] = fmaf(sm.dz[i][c][t], w2[c * KK + t], p[c]);
            }
            float sum = p[0];
            if constexpr (CW == 2) sum = p[0] + p[1];
            if constexpr (CW == 4) sum = (p[0] + p[1]) + (p[2] + p[3]);
            if (mok) a.dh_part[((int64_t)blk * d.N + n0 + i) * d.mid + m] = sum;
        }
        if (col_mine) {
            const bool gains = col_at >= ROWS;
            const int col = gains ? col_at - ROWS : col_at;
            const float *src = gains ? &sm.dg[0][col] : &sm.dz[0][col / KK][col % KK];
            const int pitch = gains ? ROWS : CW * kFc2Pitch;
#pragma unroll 8
            for (int i = col_part; i < cnt; i += PARTS) col_sum += src[i * pitch];
        }
    }
    if constexpr (PARTS > 1) {
        // (the sums of a channel's parts, in order)
        __syncthreads();
#pragma unroll
        for (int t = 0; t < KK; ++t) sm.sums.dw[wave][t][lane] = acc[t];
        if (col_mine) sm.sums.col[col_part][col_at] = col_sum;
        __syncthreads();
        for (int r = wave; r < rows; r += kWaves) {
            const int c = r / KK, t = r - c * KK;
            float total = sm.sums.dw[c][t][lane];
#pragma unroll
            for (int k = 1; k < PARTS; ++k) total += sm.sums.dw[k * CW + c][t][lane];
            if (mok) st(a.dw2 + ((int64_t)cb * KK + r) * d.mid + m, total);
        }
        if (col_mine && col_part == 0) {
#pragma unroll
            for (int k = 1; k < PARTS; ++k) col_sum += sm.sums.col[k][col_at];
        }
    } else if (mok && cb + wave < d.C) {
#pragma unroll
        for (int t = 0; t < KK; ++t) st(a.dw2 + ((int64_t)(cb + wave) * KK + t) * d.mid + m, acc[t]);
    }
    if (col_mine && col_part == 0) {
        if (col_at < rows) {
            if (a.db2) st(a.db2 + cb * KK + col_at, col_sum);
        } else if (col_at >= ROWS && col_at < ROWS + rows) {
            if (a.dgain) st(a.dgain + cb * KK + col_at - ROWS, col_sum);
        }
    }
}

// ---- weight gradient of the spatial branch's convolution ----------------------
// A product with the pixels as the summed dimension: rows are the 9 taps of a head (of the
// matrix instruction's 16), columns 16 channels, and both operands have their pixels
// contiguous in memory: 16-byte loads straight from NCHW.  A wave takes 16 channels and a
// range of a sample's pixels; the ranges' sums are added up by k_pack_hidden.
// fp32: four 16x16x4 steps per 16-byte load (pixel 4 * quad + j of the sixteen in step j: the
// order of the summed dimension is the same for both operands, so any will do).
constexpr int kRowTile = 16;

template <typename T>
struct WsArgs {
    const T *x, *draw;
    float *part;        // [N * splits][head * 9 * (C + 1)]: the weights' sums [tap][C], then the biases'
    int ctiles, splits, split_pix, nwork;
};

template <typename T> struct Quad;    // the pixels of one step that a lane loads
template <> struct Quad<__half> { using type = half8_t; static constexpr int n = 8; };
template <> struct Quad<float> { using type = float4_t; static constexpr int n = 4; };

__device__ __forceinline__ float4_t mma_step(half8_t a, half8_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4_t mma_step(float4_t a, float4_t b, float4_t c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
    return c;
}

// One wave's work item.
template <typename T, int S>
__device__ __forceinline__ void ws_item(const PackDims &d, const WsArgs<T> &a, int item, int lane) {
    using V = typename Quad<T>::type;
    constexpr int P = Quad<T>::n, STEP = 4 * P, U = 4;
    const int npix = d.Ho * d.Wo;
    const int ct = item % a.ctiles, np = item / a.ctiles;
    const int n = np / a.splits, sp = np - n * a.splits;
    const int p_begin = sp * a.split_pix, p_end = min(p_begin + a.split_pix, npix);
    const int row = lane & 15, quad = lane >> 4;
    const int c = ct * kRowTile + row;
    const T *xc = a.x + ((int64_t)n * d.C + min(c, d.C - 1)) * d.H * d.W;
    float *out = a.part + (int64_t)np * d.head * KK * (d.C + 1);
    auto load_x = [&](int p) {      // P result pixels from p, all inside the plane
        V v;
        if constexpr (S == 1) {
            __builtin_memcpy(&v, xc + p, sizeof(v));
        } else {
            int y = p / d.Wo, xx = p - y * d.Wo;
#pragma unroll
            for (int e = 0; e < P; ++e) {
                v[e] = *reinterpret_cast<const typename std::conditional<sizeof(T) == 2, _Float16, float>::type *>(
                    xc + (int64_t)y * d.s * d.W + xx * d.s);
                if (++xx == d.Wo) { xx = 0; ++y; }
            }
        }
        return v;
    };
    for (int h = 0; h < d.head; ++h) {
        const T *rt = a.draw + (((int64_t)n * d.head + h) * KK + min(row, KK - 1)) * npix;
        float4_t acc = {0.f, 0.f, 0.f, 0.f}, sums = {0.f, 0.f, 0.f, 0.f};
        V ones;
#pragma unroll
        for (int e = 0; e < P; ++e) ones[e] = 1;
        int p = p_begin;
        for (; p + U * STEP <= p_end; p += U * STEP) {
            V av[U], bv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                __builtin_memcpy(&av[u], rt + p + u * STEP + quad * P, sizeof(V));
                bv[u] = load_x(p + u * STEP + quad * P);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                acc = mma_step(av[u], bv[u], acc);
                if (ct == 0) sums = mma_step(av[u], ones, sums);
            }
        }
        for (; p < p_end; p += STEP) {
            V av, bv;
            const int q = p + quad * P;
            if (q + P <= p_end) {
                __builtin_memcpy(&av, rt + q, sizeof(V));
                bv = load_x(q);
            } else {
#pragma unroll
                for (int e = 0; e < P; ++e) {
                    const bool in = q + e < p_end;
                    const int qq = in ? q + e : p_end - 1;
                    const int y = qq / d.Wo, xx = qq - y * d.Wo;
                    av[e] = in ? (typename std::remove_reference<decltype(av[0])>::type)ld(rt + qq) : 0;
                    bv[e] = in ? (typename std::remove_reference<decltype(bv[0])>::type)ld(xc + (S == 1 ? qq : y * d.s * d.W + xx * d.s)) : 0;
                }
            }
            acc = mma_step(av, bv, acc);
            if (ct == 0) sums = mma_step(av, ones, sums);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = quad * 4 + e;
            if (t >= KK) continue;
            if (c < d.C) out[(int64_t)(h * KK + t) * d.C + c] = acc[e];
            if (ct == 0 && row == 0) out[(int64_t)d.head * KK * d.C + h * KK + t] = sums[e];
        }
    }
}

template <typename T, int CW>
__global__ __launch_bounds__(kThreads, 4) void k_pack_fc2(PackDims d, Fc2Args<T> f, WsArgs<T> w, int fc2_blocks) {
    __shared__ __align__(16) Fc2Smem<CW> sm;
    if ((int)blockIdx.x < fc2_blocks) {
        fc2_block<T, CW>(d, f, blockIdx.x, sm);
        return;
    }
    const int item = ((int)blockIdx.x - fc2_blocks) * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (item >= w.nwork) return;
    if (d.s == 1) ws_item<T, 1>(d, w, item, threadIdx.x & (kWave - 1));
    else ws_item<T, 2>(d, w, item, threadIdx.x & (kWave - 1));
}

// ---- hidden layer's gradient, and the sums of the partial dWs ------------------
// (sixteen threads share an output's parts, eight of them on their way at a time; four threads, us: 8 x 64 x 200 x 300 fp16
// 8.4 / 4.6, 64 x 64 x 56 x 56 6.6 / 4.8, 3 x 2048 x 7 x 7 7.9 / 5.0)
constexpr int kSumGroups = 16, kSumCols = kThreads / kSumGroups, kSumAhead = 8;

// Sum of N values, neighbours first (one after another sixteen of them cost dW1 and db1 5 to 7 % of their precision).
template <int N>
__device__ __forceinline__ float sum_in_pairs(float (&v)[N]) {
#pragma unroll
    for (int step = 1; step < N; step *= 2)
#pragma unroll
        for (int k = 0; k + step < N; k += 2 * step) v[k] += v[k + step];
    return v[0];
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_pack_hidden(PackDims d, const float *__restrict__ dh_part,
                                                          const float *__restrict__ hidden,
                                                          float *__restrict__ dz1, int parts, int sum_blocks,
                                                          const float *__restrict__ ws_part, int ws_parts,
                                                          T *__restrict__ dws, T *__restrict__ dbs) {
    __shared__ float red[kSumGroups][kSumCols];
    const int col = threadIdx.x % kSumCols, grp = threadIdx.x / kSumCols;
    const bool hid = (int)blockIdx.x < sum_blocks;
    const int64_t i = (int64_t)(hid ? blockIdx.x : blockIdx.x - sum_blocks) * kSumCols + col;
    const int64_t count = hid ? (int64_t)d.N * d.mid : (int64_t)d.head * KK * (d.C + 1);
    const float *src = hid ? dh_part : ws_part;
    const int np = hid ? parts : ws_parts;
    float a = 0.f;
    if (i < count) {
        for (int q0 = grp; q0 < np; q0 += kSumGroups * kSumAhead) {
            float v[kSumAhead];
#pragma unroll
            for (int k = 0; k < kSumAhead; ++k) v[k] = src[min(q0 + k * kSumGroups, np - 1) * count + i];
#pragma unroll
            for (int k = 0; k < kSumAhead; ++k) v[k] = q0 + k * kSumGroups < np ? v[k] : 0.f;
            a += sum_in_pairs(v);
        }
    }
    red[grp][col] = a;
    __syncthreads();
    if (grp != 0 || i >= count) return;
    float v[kSumGroups];
#pragma unroll
    for (int k = 0; k < kSumGroups; ++k) v[k] = red[k][col];
    a = sum_in_pairs(v);
    if (hid) {
        dz1[i] = hidden[i] <= 0.f ? 0.f : a;    // (a hidden NaN passes its gradient on, as torch has it)
    } else {
        const int64_t weights = (int64_t)d.head * KK * d.C;
        if (i < weights) st(dws + i, a);
        else if (dbs) st(dbs + i - weights, a);
    }
}

// ---- first convolution of the channel branch ----------------------------------
// Lanes are channels.  dW1: a workgroup takes kFc1 rows of W1, its waves a quarter of the
// samples each; dv: kFc1 samples and a quarter of the rows per wave.  The other factor, dz1,
// is the same for every lane.
constexpr int kFc1 = 4;

template <typename T>
__global__ __launch_bounds__(kThreads) void k_pack_fc1(PackDims d, const float *__restrict__ dz1,
                                                       const float *__restrict__ pooled,
                                                       const T *__restrict__ w1, T *__restrict__ dw1,
                                                       T *__restrict__ db1, float *__restrict__ dv, int cblks,
                                                       int mblks) {
    __shared__ float red[kWaves][2 * kFc1][kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int cblk = blockIdx.x % cblks, rest = blockIdx.x / cblks;
    const int c = cblk * kWave + lane;
    const int cc = min(c, d.C - 1);
    const bool weights = rest < mblks;
    const int q0 = (weights ? rest : rest - mblks) * kFc1;       // first hidden value / sample
    const int summed = weights ? d.N : d.mid;
    const int per = (summed + kWaves - 1) / kWaves;
    const int i0 = wave * per, i1 = min(i0 + per, summed);
    float acc[kFc1], bsum[kFc1];
#pragma unroll
    for (int q = 0; q < kFc1; ++q) acc[q] = bsum[q] = 0.f;
    if (weights) {
#pragma unroll 8
        for (int n = i0; n < i1; ++n) {
            const float p = pooled[(int64_t)n * d.C + cc];
#pragma unroll
            for (int q = 0; q < kFc1; ++q) {
                const float z = dz1[(int64_t)n * d.mid + min(q0 + q, d.mid - 1)];
                acc[q] = fmaf(z, p, acc[q]);
                bsum[q] += z;
            }
        }
    } else {
#pragma unroll 8
        for (int m = i0; m < i1; ++m) {
            const float wv = ld(w1 + (int64_t)m * d.C + cc);
#pragma unroll
            for (int q = 0; q < kFc1; ++q)
                acc[q] = fmaf(dz1[(int64_t)min(q0 + q, d.N - 1) * d.mid + m], wv, acc[q]);
        }
    }
#pragma unroll
    for (int q = 0; q < kFc1; ++q) {
        red[wave][q][lane] = acc[q];
        red[wave][kFc1 + q][lane] = bsum[q];
    }
    __syncthreads();
    // (wave q finishes output q)
    const int q = q0 + wave;
    float tot = 0.f, btot = 0.f;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) {
        tot += red[k][wave][lane];
        btot += red[k][kFc1 + wave][lane];
    }
    if (weights) {
        if (q >= d.mid) return;
        if (c < d.C) st(dw1 + (int64_t)q * d.C + c, tot);
        if (db1 && cblk == 0 && lane == 0) st(db1 + q, btot);
    } else if (q < d.N && c < d.C) {
        dv[(int64_t)q * d.C + c] = tot;
    }
}
static_assert(kFc1 == kWaves, "a wave finishes one output");

// ---- feature gradient ----------------------------------------------------------
// A lane owns VP neighbouring pixels of a sample and keeps the spatial branch's tap
// gradients that reach them (zero between the sampled pixels under a stride); the waves of
// a workgroup walk a range of channels each: one read and one write of dX per pixel and
// channel, nine multiply-adds in between.  The weights of the range and the pooled
// gradient sit in LDS, a 48-byte row per channel, read as broadcasts.
constexpr int kDxMaxChannels = 128;

template <typename T, int VP, int HEAD>
__global__ __launch_bounds__(kThreads) void k_pack_dx(PackDims d, const T *__restrict__ draw,
                                                      const T *__restrict__ ws, const float *__restrict__ dv,
                                                      T *dx, int cw, float inv_plane) {
    constexpr int TAPS = HEAD * KK, PITCH = (TAPS + 1 + 3) / 4 * 4;
    __shared__ __align__(16) float tab[kDxMaxChannels][PITCH];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int n = blockIdx.z, c0 = blockIdx.y * cw;
    const int nc = min(cw, d.C - c0);
    for (int i = threadIdx.x; i < nc; i += kThreads) {
#pragma unroll
        for (int t = 0; t < TAPS; ++t) tab[i][t] = ld(ws + (int64_t)t * d.C + c0 + i);
        tab[i][TAPS] = dv[(int64_t)n * d.C + c0 + i] * inv_plane;
    }
    const int plane = d.H * d.W, npix = d.Ho * d.Wo;
    const int p = (blockIdx.x * kWave + lane) * VP;
    const bool live = p < plane;
    struct alignas(VP * sizeof(T)) Pack { T e[VP]; };
    float dr[TAPS][VP];
#pragma unroll
    for (int t = 0; t < TAPS; ++t)
#pragma unroll
        for (int k = 0; k < VP; ++k) dr[t][k] = 0.f;
    if (live) {
        const T *rn = draw + (int64_t)n * TAPS * npix;
        if (d.s == 1) {
#pragma unroll
            for (int t = 0; t < TAPS; ++t) {
                const Pack q = *reinterpret_cast<const Pack *>(rn + (int64_t)t * npix + p);
#pragma unroll
                for (int k = 0; k < VP; ++k) dr[t][k] = ld(&q.e[k]);
            }
        } else {
#pragma unroll
            for (int k = 0; k < VP; ++k) {
                const int y = (p + k) / d.W, xx = (p + k) - y * d.W;
                if (y % d.s == 0 && xx % d.s == 0) {
                    const int q = (y / d.s) * d.Wo + xx / d.s;
#pragma unroll
                    for (int t = 0; t < TAPS; ++t) dr[t][k] = ld(rn + (int64_t)t * npix + q);
                }
            }
        }
    }
    __syncthreads();
    if (!live) return;
    const int per = (nc + kWaves - 1) / kWaves;
    const int i0 = wave * per, i1 = min(i0 + per, nc);
    T *xp = dx + ((int64_t)n * d.C + c0) * plane + p;
    constexpr int U = 4;
    auto channel = [&](int i, Pack q) {
        const float *w = tab[i];
        Pack o;
        float v[VP];
#pragma unroll
        for (int k = 0; k < VP; ++k) v[k] = ld(&q.e[k]) + w[TAPS];
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
            const float wv = w[t];
#pragma unroll
            for (int k = 0; k < VP; ++k) v[k] = fmaf(wv, dr[t][k], v[k]);
        }
#pragma unroll
        for (int k = 0; k < VP; ++k) st(&o.e[k], v[k]);
        *reinterpret_cast<Pack *>(xp + (int64_t)i * plane) = o;
    };
    int i = i0;
    for (; i + U <= i1; i += U) {
        Pack q[U];
#pragma unroll
        for (int u = 0; u < U; ++u) q[u] = *reinterpret_cast<const Pack *>(xp + (int64_t)(i + u) * plane);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u) channel(i + u, q[u]);
    }
    for (; i < i1; ++i) channel(i, *reinterpret_cast<const Pack *>(xp + (int64_t)i * plane));
}

size_t floats256(int64_t n) { return ((size_t)n * sizeof(float) + 255) / 256 * 256; }

// Pixel ranges of k_pack_fc2's weight-gradient items: enough waves to fill the machine,
// ranges of at least 128 pixels and whole steps.
void ws_split(int64_t N, int64_t C, int64_t npix, int step, int *splits, int *split_pix) {
    const int64_t base = N * cdiv(C, kRowTile);
    const int64_t want = std::max<int64_t>(1, cdiv(2048, base));
    int64_t per = std::max<int64_t>(cdiv(npix, want), 128);
    per = cdiv(per, 4 * step) * (4 * step);
    *split_pix = (int)per;
    *splits = (int)cdiv(npix, per);
}

}  // namespace

bool pack_backward_supported(int64_t N, int64_t C, int64_t mid, int64_t H, int64_t W, int head, int k,
                             int stride, int dtype) {
    const int64_t esz = dtype == DDF_F16 ? 2 : 4;
    if (k != 3 || (stride != 1 && stride != 2) || (head != 1 && head != 2 && head != 4)) return false;
    if (N <= 0 || C <= 0 || mid <= 0 || H / stride <= 0 || W / stride <= 0) return false;
    // the forward launches: channels in the streaming kernel's groups, 32-bit offsets inside
    // a sample, the channel branch's vectors in LDS
    if (C % (dtype == DDF_F16 ? 4 : 2) != 0 || H % stride != 0 || W % stride != 0 || N > 65535 ||
        C * H * W * esz >= (1ll << 31) || KK * H * W * esz >= (1ll << 31) || C + mid > 11000)
        return false;
    return N * cdiv(C, kRowTile) * cdiv(H * W, 128) < (1ll << 30) && N * mid < (1ll << 30);
}

size_t pack_backward_workspace(int64_t N, int64_t C, int64_t mid, int64_t H, int64_t W, int head, int stride,
                               int dtype) {
    int splits, split_pix;
    const int64_t npix = (H / stride) * (W / stride);
    ws_split(N, C, npix, dtype == DDF_F16 ? 32 : 16, &splits, &split_pix);
    return floats256(cdiv(C, fc2_channels(N, C, mid)) * N * mid) + floats256(N * mid) + floats256(N * C) +
           floats256(N * splits * head * KK * (C + 1));
}

template <typename T>
hipError_t pack_backward(const PackBackward<T> &b, int64_t N, int64_t C, int64_t H, int64_t W, int64_t mid,
                         int head, int stride, void *ws, hipStream_t st) {
    PackDims d{(int)N, (int)C, (int)mid, (int)H, (int)W, (int)(H / stride), (int)(W / stride), stride, head};
    const int64_t npix = (int64_t)d.Ho * d.Wo, plane = H * W;
    constexpr int STEP = 4 * Quad<T>::n;
    int splits, split_pix;
    ws_split(N, C, npix, STEP, &splits, &split_pix);
    const int cw2 = fc2_channels(N, C, mid), cblocks = (int)cdiv(C, cw2);
    unsigned char *q = static_cast<unsigned char *>(ws);
    float *dh_part = reinterpret_cast<float *>(q); q += floats256((int64_t)cblocks * N * mid);
    float *dz1 = reinterpret_cast<float *>(q); q += floats256(N * mid);
    float *dv = reinterpret_cast<float *>(q); q += floats256(N * C);
    float *ws_part = reinterpret_cast<float *>(q);

    Fc2Args<T> f{b.dcf, b.w2, b.gain_vec, (float)b.gain, b.taps, b.hidden, b.dw2, b.db2, b.dgain, dh_part,
                 (int)cdiv(mid, kWave)};
    WsArgs<T> w{b.x, b.draw, ws_part, (int)cdiv(C, kRowTile), splits, split_pix, 0};
    w.nwork = (int)(N * splits * w.ctiles);
    const int fc2_blocks = cblocks * f.mchunks;
    const dim3 grid2((unsigned)(fc2_blocks + cdiv(w.nwork, kWaves)));
    if (cw2 == 1) hipLaunchKernelGGL((k_pack_fc2<T, 1>), grid2, dim3(kThreads), 0, st, d, f, w, fc2_blocks);
    else if (cw2 == 2) hipLaunchKernelGGL((k_pack_fc2<T, 2>), grid2, dim3(kThreads), 0, st, d, f, w, fc2_blocks);
    else hipLaunchKernelGGL((k_pack_fc2<T, 4>), grid2, dim3(kThreads), 0, st, d, f, w, fc2_blocks);
    const int hid_blocks = (int)cdiv(N * mid, kSumCols);
    hipLaunchKernelGGL((k_pack_hidden<T>), dim3((unsigned)(hid_blocks + cdiv((int64_t)head * KK * (C + 1), kSumCols))),
                       dim3(kThreads), 0, st, d, dh_part, b.hidden, dz1, cblocks, hid_blocks, ws_part,
                       (int)(N * splits), b.dws, b.dbs);
    const int cblks = (int)cdiv(C, kWave), mblks = (int)cdiv(mid, kFc1);
    const int nblks = b.dx ? (int)cdiv(N, kFc1) : 0;
    hipLaunchKernelGGL((k_pack_fc1<T>), dim3((unsigned)(cblks * (mblks + nblks))), dim3(kThreads), 0, st, d, dz1,
                       b.pooled, b.w1, b.dw1, b.db1, dv, cblks, mblks);
    if (b.dx) {
        // the widest vector that planes and addresses allow; 72 tap gradients in registers at most
        int vp = 16 / (int)sizeof(T);
        while (vp > 1 && (vp * head > 8 || plane % vp != 0 || (stride == 1 && npix % vp != 0) ||
                          (((uintptr_t)b.dx | (uintptr_t)b.draw) % (vp * sizeof(T))) != 0))
            vp /= 2;
        const int64_t tiles = cdiv(plane, kWave * vp);
        // (channels per workgroup: 2048 waves where the walks stay at four channels or more)
        int64_t cw = cdiv(C, std::max<int64_t>(1, 512 / (tiles * N)));
        cw = std::min<int64_t>(std::max<int64_t>(cdiv(cw, 16) * 16, 16), kDxMaxChannels);
        const dim3 grid((unsigned)tiles, (unsigned)cdiv(C, cw), (unsigned)N);
#define DDF_DX_CASE(VP_, HEAD_)                                                                     \
    if (vp == VP_ && head == HEAD_)                                                                 \
        hipLaunchKernelGGL((k_pack_dx<T, VP_, HEAD_>), grid, dim3(kThreads), 0, st, d, b.draw, b.ws, dv, \
                           b.dx, (int)cw, (float)(1.0 / (double)plane))
        if constexpr (sizeof(T) == 2) DDF_DX_CASE(8, 1);
        DDF_DX_CASE(4, 1); DDF_DX_CASE(2, 1); DDF_DX_CASE(1, 1);
        DDF_DX_CASE(4, 2); DDF_DX_CASE(2, 2); DDF_DX_CASE(1, 2);
        DDF_DX_CASE(2, 4); DDF_DX_CASE(1, 4);
#undef DDF_DX_CASE
    }
    return hipGetLastError();
}

template hipError_t pack_backward<__half>(const PackBackward<__half> &, int64_t, int64_t, int64_t, int64_t,
                                          int64_t, int, int, void *, hipStream_t);
template hipError_t pack_backward<float>(const PackBackward<float> &, int64_t, int64_t, int64_t, int64_t,
                                         int64_t, int, int, void *, hipStream_t);

}  // namespace ddf

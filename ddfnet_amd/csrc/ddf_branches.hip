// The two filter branches of DDFPack as one launch each (gfx950, inference):
//
//   spatial (ddf/ddf.py:176-180 of the reference, FilterNorm 'spatial' :145-157):
//     sf[n, g*KK + t, yo, xo] = norm_t( bias[g*KK + t] + sum_c w[g*KK + t, c] * x[n, c, yo*s, xo*s] )
//   a 1x1 convolution with the operator's stride followed by the filter
//   normalisation over the KK taps of every pixel.  It reads x once and writes
//   the normalised taps; the un-normalised taps never reach memory.
//
//   channel (ddf/ddf.py:183-192, FilterNorm 'channel' :158-170), after the global
//   average pool:
//     cf[n, c, t] = norm_t( b2[c*KK + t] + sum_m w2[c*KK + t, m] * relu(b1[m] + sum_c' w1[m, c'] * v[n, c']) )
//   the two 1x1 convolutions on the pooled (n, c) vector are small matrix
//   products (ddf_channel.h): one workgroup computes the hidden vector of its sample and 16
//   to 64 channels' filters out of LDS (k_channel_branch_rows), or, in fp16 with a hidden
//   layer of 32 values or more, sixteen samples x sixteen channels on the matrix cores
//   (k_channel_branch_mma); large batches, 5 x 5 taps and unaligned weights go through
//   k_channel_branch, whose loads serve several samples.
//
// norm_t(u) = gain_t * (u_t - mean(u)) / (std(u) + 1e-10) + offset_t with the
// unbiased standard deviation over the KK taps, as in ddf_filter_norm.hip.
// Both kernels are bound by memory and launch latency, not by arithmetic: the
// spatial branch does KK multiply-adds per 4-byte (2-byte) load.
#include <algorithm>
#include <type_traits>

#include "ddf_channel.h"
#include "ddf_common.h"
#include "ddf_rows.h"

namespace ddf {
int tune_int(const char *name, int fallback);

namespace {
using rows::kOutside;
using rows::load_vec;
using rows::plane_rsrc;
using rows::store_vec_nt;
using rows::vec_words;

constexpr int kChunk = 256;   // channels whose weights sit in LDS at a time (64 per wave)

// VP storage-type values at p (aligned to VP * sizeof(T)), widened.
template <typename T, int VP>
__device__ __forceinline__ void load_pixels(const T *p, float (&v)[VP]) {
    if constexpr (VP == 1) {
        v[0] = ld(p);
    } else {
        struct alignas(VP * sizeof(T)) Pack { T e[VP]; };
        const Pack q = *reinterpret_cast<const Pack *>(p);
#pragma unroll
        for (int k = 0; k < VP; ++k) v[k] = ld(&q.e[k]);
    }
}

// grid (pixel tiles of 64 * VP, head, N); the WAVES waves of a workgroup cover
// the same result pixels (a lane owns VP consecutive pixels of a row: VP > 1
// needs stride 1 and rows that are a whole number of such vectors) and
// 1/WAVES of every channel chunk each, U channels' loads in flight at a time.
template <typename T, int KK, int WAVES, int VP>
__global__ __launch_bounds__(WAVES * kWave) void k_spatial_branch(
    const T *__restrict__ x, const T *__restrict__ w, const T *__restrict__ bias,
    T *__restrict__ sf, int C, int H, int W, int Ho, int Wo, int stride, int chunk, float gain,
    const T *__restrict__ gain_vec, const T *__restrict__ offset_vec) {
    constexpr int U = VP >= 4 ? 4 : 8;
    // weights of the chunk, [channel][tap], rows padded to 16 bytes (wide LDS reads)
    __shared__ __align__(16) float wt[kChunk][(KK + 3) / 4 * 4];
    __shared__ float red[WAVES][KK][kWave];             // per-wave sums of one pixel of the vector
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int g = blockIdx.y, heads = gridDim.y;
    const int64_t n = blockIdx.z;
    const int npix = Ho * Wo;
    const int pix = (blockIdx.x * kWave + lane) * VP;   // first of the lane's pixels
    const bool live = pix < npix;
    const int yo = live ? pix / Wo : 0, xo = live ? pix - yo * Wo : 0;
    const int64_t plane = (int64_t)H * W;
    const T *xp = x + n * C * plane + (int64_t)yo * stride * W + (int64_t)xo * stride;
    const T *wg = w + (int64_t)g * KK * C;
    const int per = chunk / WAVES;                      // channels of a chunk per wave (multiple of U)
    TapParams<T, KK> params;
    if (wave == 0) params.load(g, gain, gain_vec, offset_vec, bias);   // (wave 0 writes the taps)

    float acc[KK][VP];
#pragma unroll
    for (int t = 0; t < KK; ++t)
#pragma unroll
        for (int k = 0; k < VP; ++k) acc[t][k] = 0.f;
    for (int c0 = 0; c0 < C; c0 += chunk) {
        if (c0 > 0) __syncthreads();
        // weights of channels c0 .. c0+chunk-1 (zero past C), coalesced along a weight row
        for (int i = threadIdx.x; i < chunk; i += WAVES * kWave) {
            const int c = c0 + i;
#pragma unroll
            for (int t = 0; t < KK; ++t) wt[i][t] = c < C ? ld(wg + (int64_t)t * C + c) : 0.f;
        }
        __syncthreads();
        const int cw = c0 + wave * per;                 // this wave's channels of the chunk
        const int nc = min(per, C - cw);                // (<= 0: none left)
        for (int i0 = 0; i0 < nc; i0 += U) {
            float xv[U][VP];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = min(i0 + u, nc - 1);      // past the end: repeats, with zero weights
                if (live) {
                    load_pixels<T, VP>(xp + (int64_t)(cw + i) * plane, xv[u]);
                } else {
#pragma unroll
                    for (int k = 0; k < VP; ++k) xv[u][k] = 0.f;
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // (rows past the wave's last channel belong to channels >= C: zeros)
                const float *wr = wt[wave * per + i0 + u];
#pragma unroll
                for (int t = 0; t < KK; ++t) {
                    const float wv = wr[t];
#pragma unroll
                    for (int k = 0; k < VP; ++k) acc[t][k] = fmaf(wv, xv[u][k], acc[t][k]);
                }
            }
        }
    }
    // one pixel of the vectors at a time through LDS: the waves' sums, then wave 0
    // normalises and writes that pixel's taps
#pragma unroll
    for (int k = 0; k < VP; ++k) {
        if (k > 0) __syncthreads();
#pragma unroll
        for (int t = 0; t < KK; ++t) red[wave][t][lane] = acc[t][k];
        __syncthreads();
        if (wave == 0 && live) {
            float v[KK];
#pragma unroll
            for (int t = 0; t < KK; ++t) {
                float s = 0.f;
#pragma unroll
                for (int q = 0; q < WAVES; ++q) s += red[q][t][lane];
                v[t] = s;
            }
            normalise<T, KK>(v, params);
            T *op = sf + ((n * heads + g) * KK) * (int64_t)npix + pix + k;
#pragma unroll
            for (int t = 0; t < KK; ++t) st(op + (int64_t)t * npix, v[t]);
        }
    }
}

// The same for planes with many pixels: every wave of the workgroup has its own
// 64 * VP result pixels and walks all channels, so nothing is added up across
// waves and the taps are normalised in registers.  grid (tiles of 4 * 64 * VP
// pixels, head, N).
template <typename T, int KK, int VP>
__global__ __launch_bounds__(4 * kWave) void k_spatial_branch_tiles(
    const T *__restrict__ x, const T *__restrict__ w, const T *__restrict__ bias,
    T *__restrict__ sf, int C, int H, int W, int Ho, int Wo, int stride, int chunk, float gain,
    const T *__restrict__ gain_vec, const T *__restrict__ offset_vec) {
    constexpr int U = 16;   // channels in flight per wave: what the run time hangs on
    __shared__ __align__(16) float wt[kChunk][(KK + 3) / 4 * 4];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int g = blockIdx.y, heads = gridDim.y;
    const int64_t n = blockIdx.z;
    const int npix = Ho * Wo;
    const int pix = ((blockIdx.x * 4 + wave) * kWave + lane) * VP;
    const bool live = pix < npix;
    const int yo = live ? pix / Wo : 0, xo = live ? pix - yo * Wo : 0;
    const int64_t plane = (int64_t)H * W;
    const T *xp = x + n * C * plane + (int64_t)yo * stride * W + (int64_t)xo * stride;
    const T *wg = w + (int64_t)g * KK * C;
    TapParams<T, KK> params;
    params.load(g, gain, gain_vec, offset_vec, bias);

    float acc[KK][VP];
#pragma unroll
    for (int t = 0; t < KK; ++t)
#pragma unroll
        for (int k = 0; k < VP; ++k) acc[t][k] = 0.f;
    for (int c0 = 0; c0 < C; c0 += chunk) {
        if (c0 > 0) __syncthreads();
        for (int i = threadIdx.x; i < chunk; i += 4 * kWave) {
            const int c = c0 + i;
#pragma unroll
            for (int t = 0; t < KK; ++t) wt[i][t] = c < C ? ld(wg + (int64_t)t * C + c) : 0.f;
        }
        __syncthreads();
        const int nc = min(chunk, C - c0);
        for (int i0 = 0; i0 < nc; i0 += U) {
            float xv[U][VP];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = min(i0 + u, nc - 1);      // past the end: repeats, with zero weights
                if (live) {
                    load_pixels<T, VP>(xp + (int64_t)(c0 + i) * plane, xv[u]);
                } else {
#pragma unroll
                    for (int k = 0; k < VP; ++k) xv[u][k] = 0.f;
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float *wr = wt[i0 + u];           // (i0 + u < chunk: chunk is a multiple of U)
                float wv[KK];
#pragma unroll
                for (int t = 0; t < KK; ++t) wv[t] = wr[t];
#pragma unroll
                for (int t = 0; t < KK; ++t)
#pragma unroll
                    for (int k = 0; k < VP; ++k) acc[t][k] = fmaf(wv[t], xv[u][k], acc[t][k]);
            }
        }
    }
    if (!live) return;
#pragma unroll
    for (int k = 0; k < VP; ++k) {
        float v[KK];
#pragma unroll
        for (int t = 0; t < KK; ++t) v[t] = acc[t][k];
        normalise<T, KK>(v, params);
#pragma unroll
        for (int t = 0; t < KK; ++t) acc[t][k] = v[t];
    }
    // taps of the lane's VP pixels, one vector store per tap plane
    T *op = sf + ((n * heads + g) * KK) * (int64_t)npix + pix;
#pragma unroll
    for (int t = 0; t < KK; ++t) {
        if constexpr (VP == 1) {
            st(op + (int64_t)t * npix, acc[t][0]);
        } else {
            struct alignas(VP * sizeof(T)) Pack { T e[VP]; } q;
#pragma unroll
            for (int k = 0; k < VP; ++k) st(&q.e[k], acc[t][k]);
            *reinterpret_cast<Pack *>(op + (int64_t)t * npix) = q;
        }
    }
}

// ---------------------------------------------------------------------------
// Spatial branch, 3 x 3 taps, as a stream over the channels (the kernel the
// launcher prefers).  A lane owns VP neighbouring result pixels of one sample
// (stride 1: the plane is one run of pixels, so a vector may cross image rows;
// stride 2: the 2 * VP feature pixels under VP result pixels of one row come in
// as one vector; see vector_of) and adds up KK taps for each.  The WAVES waves of a workgroup
// cover the same pixels and a range of channels each, U at a time; their sums
// meet in LDS at the end.  Like the operator's own kernels it has
//   * every channel plane behind a buffer descriptor (an idle lane's offset and
//     the planes past the last channel read zero, no bounds branch),
//   * the loads of NST - 1 channel groups in flight while one is computed,
//   * the weights - the same for every lane - in scalar registers.
struct SpatialGeom {
    int C, W, Wo;
    int plane;      // H * W
    int npix;       // Ho * Wo
    int nvec;       // vectors of VP result pixels (see vector_of)
    int vrow;       // stride 2: vectors of a row
    int lpt;        // lanes of a workgroup's pixel tile that have a vector
    int ngroups;    // C / U
    int gpw;        // channel groups per wave
    int steps;      // gpw rounded up to a multiple of NST
};

// Where vector v of a sample's begins: its first result pixel, its first feature element.  The last vector of
// the run (stride 2: of a row) ends with it: it begins further left where VP does not divide the
// run, and its first `again` pixels are the vector's before, too - made twice, alike, and counted once
// in the planes' sums.  So planes of any size have full vectors (at any element address), no
// tails and no branches.
struct VectorAt { int p, in, again; };
template <int VP, int S>
__device__ __forceinline__ VectorAt vector_of(const SpatialGeom &g, int v) {
    if constexpr (S == 1) {
        const int p = min(v * VP, g.npix - VP);
        return {p, p, v * VP - p};
    } else {
        const int yo = v / g.vrow, at = (v - yo * g.vrow) * VP, xo = min(at, g.Wo - VP);
        return {yo * g.Wo + xo, 2 * yo * g.W + 2 * xo, at - xo};
    }
}
// Masks of the words of a vector without its first `again` elements (bitwise: an infinity among
// those must not reach the sums).
template <typename T, int NW>
__device__ __forceinline__ void words_from(int again, uint32_t (&mask)[NW]) {
#pragma unroll
    for (int k = 0; k < NW; ++k) {
        if constexpr (sizeof(T) == 4) mask[k] = k >= again ? ~0u : 0u;
        else mask[k] = (2 * k >= again ? 0xffffu : 0u) | (2 * k + 1 >= again ? 0xffff0000u : 0u);
        asm volatile("" : "+v"(mask[k]));    // (not as comparisons: pairs of scalar registers, of which there are none left)
    }
}

// Sums of U (2 or 4) values per lane over the wave: every lane ends up with the total of
// value number (lane % U).  The first steps halve the
// number of values a lane carries instead of adding U full sums side by side: lane
// pairs exchange the value the other keeps (quad permutes); then the quads of a row add
// up by rotation, and the rows of the wave by swapping rows and halves of it (gfx950's lane
// swaps, on the vector ALU: reads through the LDS unit would share the counter of the
// kernel's scalar weight loads - waiting for one drains the other's prefetch).
template <int CTRL>
__device__ __forceinline__ float from_permuted(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int U>
__device__ __forceinline__ float wave_sums(const float (&v)[U], int lane) {
    static_assert(U == 2 || U == 4, "two or four values per lane");
    const bool b0 = lane & 1, b1 = lane & 2;
    float k = (b0 ? v[1] : v[0]) + from_permuted<0xB1 /* quad_perm [1,0,3,2] */>(b0 ? v[0] : v[1]);
    if constexpr (U == 4) {
        const float k1 = (b0 ? v[3] : v[2]) + from_permuted<0xB1>(b0 ? v[2] : v[3]);
        k = (b1 ? k1 : k) + from_permuted<0x4E /* quad_perm [2,3,0,1] */>(b1 ? k : k1);
    } else {
        k += from_permuted<0x4E>(k);
    }
    k += from_permuted<0x124 /* row_ror:4 */>(k);
    k += from_permuted<0x128 /* row_ror:8 */>(k);
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(k), __float_as_uint(k), false, false);
    k = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(k), __float_as_uint(k), false, false);
    return __uint_as_float(h[0]) + __uint_as_float(h[1]);
}

// POOL: the kernel also leaves, per sample, pixel tile and channel, the sum of the
// feature map over the pixels of the tile in pool_part[(n * tiles + tile) * C + c] (fp32) -
// the global average pool in front of the channel branch, from the values this kernel
// has in registers anyway.  Under stride 2 (even H and W) the lane also loads the
// feature row below its own, and both columns where it otherwise takes one; those lines
// come in with their neighbours in any case.
// RAGGED: VP does not divide the run (or the row) of pixels.
template <typename T, int KK, int VP, int S, int WAVES, int U, int NST, bool POOL = false, bool RAGGED = false>
__global__ __launch_bounds__(WAVES * kWave) void k_spatial_stream(
    SpatialGeom g, const T *__restrict__ x, const T *__restrict__ w, const T *__restrict__ bias,
    T *__restrict__ sf, float gain, const T *__restrict__ gain_vec, const T *__restrict__ offset_vec,
    float *__restrict__ pool_part, T *__restrict__ raw) {
    // feature elements a lane loads per channel (pooling under stride 2: both columns)
    constexpr int XE = S == 1 ? VP : (VP == 1 && !POOL ? 1 : 2 * VP);
    constexpr int kXB = XE * sizeof(T), NWX = vec_words(kXB);
    constexpr int kOB = VP * sizeof(T), NWO = vec_words(kOB);
    constexpr int WPU = U * sizeof(T) / 4;                     // 32-bit words of U weights
    static_assert(U * sizeof(T) % 4 == 0 && U % 2 == 0, "weights come in whole words, channels in pairs");
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int head = blockIdx.y, heads = gridDim.y;
    const int64_t n = blockIdx.z;
    const int v = blockIdx.x * g.lpt + lane;
    const bool live = lane < g.lpt && v < g.nvec;
    const VectorAt at = vector_of<VP, S>(g, v);
    const int p = at.p;                                        // first of the lane's result pixels
    const uint32_t xb = live ? (uint32_t)at.in * (uint32_t)sizeof(T) : kOutside;
    // The row below, which the sums of head 0 need.  For the other heads its offsets lie outside: under a branch
    // per channel the compiler asks for a step's lower rows before the upper ones.  us, branches / offsets:
    // fp16 128 x 128 x 56 x 56 26.0 / 24.1, with two heads 35.8 / 35.2, 128 x 256 x 28 x 28 16.4 / 15.0, 8 x 64 x
    // 200 x 304 16.8 / 15.9, fp32 32 x 128 x 56 x 56 13.3 / 12.9; single pixels keep the branch (128 x 512 x 14 x 14
    // 16.6 / 17.4).
    const uint32_t low = live && head == 0 ? xb + (uint32_t)g.W * (uint32_t)sizeof(T) : kOutside;
    constexpr bool kMasked = POOL && RAGGED && VP > 1;
    uint32_t mask[NWX];
    if constexpr (kMasked) words_from<T, NWX>(S * at.again, mask);
    auto counted = [&](uint32_t word, int k) __attribute__((always_inline)) { return kMasked ? word & mask[k] : word; };
    const uint32_t plane_bytes = (uint32_t)g.plane * (uint32_t)sizeof(T);
    // the sample's C planes behind one descriptor; a channel is a scalar offset into it
    const __amdgpu_buffer_rsrc_t xr = plane_rsrc(x + n * g.C * (int64_t)g.plane, (uint32_t)g.C * plane_bytes);
    const char *wg = reinterpret_cast<const char *>(w + (int64_t)head * KK * g.C);
    const uint32_t row_bytes = (uint32_t)g.C * (uint32_t)sizeof(T);
    const int j0 = wave * g.gpw;                               // the wave's first channel group

    uint32_t xw[NST][U][NWX];
    uint32_t xlow[POOL && S == 2 ? NST : 1][U][NWX];           // (pooling under stride 2: the row below)
    short xh[NST][U];                                          // (single fp16 elements: as loaded)
    uint32_t ww[NST][KK][WPU];
    // channel group i of this wave's gpw consecutive ones, stage ST (consecutive: a wave's
    // weights of consecutive steps then share scalar-cache lines)
    auto issue = [&](auto st_tag, int i) __attribute__((always_inline)) {
        constexpr int ST = decltype(st_tag)::value;
        const bool have = i < g.gpw && j0 + i < g.ngroups;
        // (a group the wave does not have: every lane's offset lies outside, the loads
        // return zero - whatever weights they then meet)
        const int j = have ? j0 + i : (j0 < g.ngroups ? j0 : 0);
        const uint32_t vb = have ? xb : kOutside;
        const uint32_t cb = (uint32_t)(j * U) * plane_bytes;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if constexpr (kXB == 2) {
                xh[ST][u] = __builtin_amdgcn_raw_buffer_load_b16(xr, (int)vb, (int)(cb + (uint32_t)u * plane_bytes), 0);
            } else if constexpr (kXB == 4) {
                xw[ST][u][0] = __builtin_amdgcn_raw_buffer_load_b32(xr, (int)vb, (int)(cb + (uint32_t)u * plane_bytes), 0);
            } else if constexpr (kXB == 8) {
                const auto q = __builtin_amdgcn_raw_buffer_load_b64(xr, (int)vb, (int)(cb + (uint32_t)u * plane_bytes), 0);
                xw[ST][u][0] = q[0]; xw[ST][u][1] = q[1];
            } else {
                static_assert(kXB <= 16, "vectors of 16 bytes at most");
                const auto q = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)vb, (int)(cb + (uint32_t)u * plane_bytes), 0);
#pragma unroll
                for (int k = 0; k < 4; ++k) xw[ST][u][k] = q[k];
            }
            if constexpr (POOL && S == 2) {
                if (VP > 1 || head == 0)
                    load_vec<kXB>(xr, have && low != kOutside ? low + cb + (uint32_t)u * plane_bytes : kOutside, xlow[ST][u]);
            }
        }
    };
    // The weights of group i, stage ST.  They are requested one step ahead only (a scalar
    // load is back well within a step), so two of the NST register sets are alive at any
    // time: with all of them the pooled variants run out of scalar registers.
    auto issue_weights = [&](auto st_tag, int i) __attribute__((always_inline)) {
        constexpr int ST = decltype(st_tag)::value;
        const bool have = i < g.gpw && j0 + i < g.ngroups;
        const int j = have ? j0 + i : (j0 < g.ngroups ? j0 : 0);
        const uint32_t wb = (uint32_t)(j * U) * (uint32_t)sizeof(T);
#pragma unroll
        for (int t = 0; t < KK; ++t)
#pragma unroll
            for (int q = 0; q < WPU; ++q)
                ww[ST][t][q] = *reinterpret_cast<const uint32_t *>(wg + (wb + (uint32_t)t * row_bytes + 4u * q));
    };
    float acc[KK][VP];
#pragma unroll
    for (int t = 0; t < KK; ++t)
#pragma unroll
        for (int k = 0; k < VP; ++k) acc[t][k] = 0.f;
    // POOL: where this lane's sums of the wave's first channel group go (one partial sum
    // per tile), and how many groups the wave keeps sums of (head
    // 0 of a sample does it for all heads).  Worked out here and pinned: formed inside the
    // walk they take a scalar load of a launch dimension, and the wait for it also waits
    // for the weights that were just requested for the next step.  The sums go out through
    // a buffer descriptor of the tile's C values, lanes with nothing to write at an
    // offset outside it: a store under a branch leaves the compiler unable to count the
    // loads in flight where the branch joins, and it then waits for all of them.
    // (Collecting the sums in LDS and writing them after the walk was no faster.)
    __amdgpu_buffer_rsrc_t pool_rsrc = plane_rsrc(nullptr, 0u);
    uint32_t pool_off = kOutside;
    int pool_groups = 0;
    if constexpr (POOL) {
        pool_rsrc = plane_rsrc(pool_part + (n * gridDim.x + blockIdx.x) * g.C,
                               (uint32_t)g.C * (uint32_t)sizeof(float));
        if (head == 0 && lane < U) pool_off = (uint32_t)(j0 * U + lane) * (uint32_t)sizeof(float);
        pool_groups = head == 0 ? min(g.gpw, g.ngroups - j0) : 0;
        asm volatile("" : "+v"(pool_off), "+s"(pool_groups));
    }
    auto compute = [&](auto st_tag, int i) __attribute__((always_inline)) {
        constexpr int ST = decltype(st_tag)::value;
        if constexpr (POOL) {
            // (No branch around the arithmetic: it would cut the step into blocks, and the
            // waits the compiler then places at their joins cost more than the sums of a
            // group the wave does not have.)
            const bool keep = i < pool_groups;
            {
                float psum[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    float ps = 0.f;
                    if constexpr (sizeof(T) == 2 && kXB == 2) {
                        ps = (float)__builtin_bit_cast(_Float16, xh[ST][u]);
                    } else if constexpr (sizeof(T) == 2) {
                        // (every word on its own, then a tree of additions: one accumulator for
                        // all words is a chain of dependent dot products, each waiting out the
                        // latency of the one before)
                        const rows::half2_t ones = {(_Float16)1, (_Float16)1};
                        float part[NWX];
#pragma unroll
                        for (int k = 0; k < NWX; ++k) {
                            part[k] = __builtin_amdgcn_fdot2(__builtin_bit_cast(rows::half2_t, counted(xw[ST][u][k], k)), ones, 0.f, false);
                            if constexpr (S == 2)
                                part[k] = __builtin_amdgcn_fdot2(__builtin_bit_cast(rows::half2_t, counted(xlow[ST][u][k], k)), ones, part[k], false);
                        }
                        if constexpr (NWX == 4) ps = (part[0] + part[1]) + (part[2] + part[3]);
                        else if constexpr (NWX == 2) ps = part[0] + part[1];
                        else ps = part[0];
                    } else {
#pragma unroll
                        for (int k = 0; k < NWX; ++k) {
                            ps += __uint_as_float(counted(xw[ST][u][k], k));
                            if constexpr (S == 2) ps += __uint_as_float(counted(xlow[ST][u][k], k));
                        }
                    }
                    psum[u] = ps;
                }
                const float tot = wave_sums<U>(psum, lane);
                __builtin_amdgcn_raw_buffer_store_b32(
                    __float_as_uint(tot), pool_rsrc,
                    (int)(keep ? pool_off + (uint32_t)(i * U) * (uint32_t)sizeof(float) : kOutside), 0, 0);
            }
        }
        if constexpr (sizeof(T) == 2) {
            // two channels at a time: (x[c], x[c+1]) of a pixel against (w[c], w[c+1]), which is
            // one word of the weight row as it lies in memory; fp32 sums
#pragma unroll
            for (int pr = 0; pr < U / 2; ++pr)
#pragma unroll
                for (int k = 0; k < VP; ++k) {
                    constexpr uint32_t kLow = 0x05040100u, kHigh = 0x07060302u;
                    rows::half2_t xp;
                    if constexpr (kXB == 2) {
                        xp[0] = __builtin_bit_cast(_Float16, xh[ST][2 * pr]);
                        xp[1] = __builtin_bit_cast(_Float16, xh[ST][2 * pr + 1]);
                    } else {
                        const int e = S * k;
                        xp = __builtin_bit_cast(rows::half2_t,
                                                __builtin_amdgcn_perm(xw[ST][2 * pr + 1][e / 2], xw[ST][2 * pr][e / 2],
                                                                      (e & 1) ? kHigh : kLow));
                    }
#pragma unroll
                    for (int t = 0; t < KK; ++t)
                        acc[t][k] = __builtin_amdgcn_fdot2(xp, __builtin_bit_cast(rows::half2_t, ww[ST][t][pr]),
                                                           acc[t][k], false);
                }
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float xv[VP];
#pragma unroll
                for (int k = 0; k < VP; ++k) xv[k] = rows::elem<T>(xw[ST][u], S * k);
#pragma unroll
                for (int t = 0; t < KK; ++t) {
                    const float wv = rows::elem<T>(ww[ST][t], u);
#pragma unroll
                    for (int k = 0; k < VP; ++k) acc[t][k] = fmaf(wv, xv[k], acc[t][k]);
                }
            }
        }
    };
    // (in this order: the waits inside the walk count the loads that were issued later)
    issue(std::integral_constant<int, 0>{}, 0);
    issue_weights(std::integral_constant<int, 0>{}, 0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (NST > 2) issue(std::integral_constant<int, 1>{}, 1);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (NST > 3) issue(std::integral_constant<int, 2>{}, 2);
    __builtin_amdgcn_sched_barrier(0);
    auto step = [&](auto st_tag, int i) __attribute__((always_inline)) {
        constexpr int ST = decltype(st_tag)::value;
        issue(std::integral_constant<int, (ST + NST - 1) % NST>{}, i + NST - 1);
        issue_weights(std::integral_constant<int, (ST + 1) % NST>{}, i + 1);
        __builtin_amdgcn_sched_barrier(0);
        compute(st_tag, i);
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int i = 0; i < g.steps; i += NST) {
        step(std::integral_constant<int, 0>{}, i);
        if constexpr (NST > 1) step(std::integral_constant<int, 1>{}, i + 1);
        if constexpr (NST > 2) step(std::integral_constant<int, 2>{}, i + 2);
        if constexpr (NST > 3) step(std::integral_constant<int, 3>{}, i + 3);
    }

    if constexpr (WAVES > 1) {
        // The waves' sums meet in LDS, [slot][tap][lane][pixel], half of the waves handing theirs to
        // the other half at a time (each round has slots of its own, so one barrier will do):
        // wave 0 alone adding up fifteen others waited for LDS fifteen times.
        __shared__ __align__(16) float red[WAVES - 1][KK][kWave][VP];
        rows::static_for<0, WAVES == 2 ? 1 : WAVES == 4 ? 2 : WAVES == 8 ? 3 : 4>([&](auto round) __attribute__((always_inline)) {
            constexpr int HALF = WAVES >> (decltype(round)::value + 1), FIRST = WAVES - 2 * HALF;
            if (wave >= HALF && wave < 2 * HALF) {
#pragma unroll
                for (int t = 0; t < KK; ++t)
#pragma unroll
                    for (int k = 0; k < VP; ++k) red[FIRST + wave - HALF][t][lane][k] = acc[t][k];
            }
            __syncthreads();
            if (wave < HALF) {
#pragma unroll
                for (int t = 0; t < KK; ++t)
#pragma unroll
                    for (int k = 0; k < VP; ++k) acc[t][k] += red[FIRST + wave][t][lane][k];
            }
        });
        if (wave > 0) return;
    }
    TapParams<T, KK> params;
    params.load(head, gain, gain_vec, offset_vec, bias);
    const int64_t taps_at = ((n * heads + head) * KK) * (int64_t)g.npix;
    const uint32_t ob = live ? (uint32_t)p * (uint32_t)sizeof(T) : kOutside;
    if (raw) {   // (training: the gradient of the normalisation wants the taps as they go into it)
        const __amdgpu_buffer_rsrc_t rr = plane_rsrc(raw + taps_at, (uint32_t)KK * (uint32_t)g.npix * (uint32_t)sizeof(T));
#pragma unroll
        for (int t = 0; t < KK; ++t) {
            float r[VP];
#pragma unroll
            for (int k = 0; k < VP; ++k) r[k] = acc[t][k] + params.bias[t];
            uint32_t ow[NWO];
            rows::pack<T, VP, float>(r, ow);
            store_vec_nt<kOB>(rr, ob + (uint32_t)t * (uint32_t)g.npix * (uint32_t)sizeof(T), ow);
        }
    }
#pragma unroll
    for (int k = 0; k < VP; ++k) {
        float r[KK];
#pragma unroll
        for (int t = 0; t < KK; ++t) r[t] = acc[t][k];
        normalise<T, KK>(r, params);
#pragma unroll
        for (int t = 0; t < KK; ++t) acc[t][k] = r[t];
    }
    const __amdgpu_buffer_rsrc_t orr = plane_rsrc(sf + taps_at, (uint32_t)KK * (uint32_t)g.npix * (uint32_t)sizeof(T));
#pragma unroll
    for (int t = 0; t < KK; ++t) {
        uint32_t ow[NWO];
        rows::pack<T, VP, float>(acc[t], ow);
        store_vec_nt<kOB>(orr, ob + (uint32_t)t * (uint32_t)g.npix * (uint32_t)sizeof(T), ow);
    }
}

// Spatial branch of fp16 planes on the matrix cores, 3 x 3 taps, stride 1: the taps are a product
// of nine weight rows with the pixels' channels.  A wave owns 16 * VP neighbouring pixels, its lane
// (l & 15) VP of them, and its quarter (l >> 4) of the lanes four of 16 channels: four loads of a
// vector of pixels, which pairs of channels turn into VP operands of 16 pixels x 16 channels in the
// order that the 16x16x16 step wants (4 * VP / 2 permutes; the product itself is VP steps).  Pixel e
// of every lane is column l & 15 of result e, taps 4 * quarter + 0..3 in its four registers, so a
// pixel's nine taps are spread over three quarters, which meet in the normalisation; a tap's VP
// pixels lie in one lane and leave as a vector.  A workgroup is four such waves next to each other,
// their sums over the pixels (see k_spatial_stream) meet in LDS.
// k_spatial_stream spends nine dot products on a pixel's pair of channels, 1230 vector
// instructions per 128 pixels of 64 channels, where this takes half of it and memory is what bounds
// it: 8 x 64 x 200 x 300 in 16.4 us, 13.5 at copy rate.  Groups of 32 channels (the 16x16x32 step)
// took 155 registers, three waves per SIMD and 17.4 us; three groups of 16 in flight 19.0.
constexpr int kSpatialMmaWaves = 4, kSpatialMmaStages = 2, kSpatialMmaGroup = 16, kSpatialMmaChannels = 2048;

template <int VP, bool POOL, bool RAGGED>
__global__ __launch_bounds__(kSpatialMmaWaves * kWave, VP == 8 ? 4 : 6) void k_spatial_mma(
    SpatialGeom g, const __half *__restrict__ x, const __half *__restrict__ w, const __half *__restrict__ bias,
    __half *__restrict__ sf, float gain, const __half *__restrict__ gain_vec, const __half *__restrict__ offset_vec,
    float *__restrict__ pool_part, __half *__restrict__ raw) {
    constexpr int KK = 9, NST = kSpatialMmaStages, G = kSpatialMmaGroup, NW = VP / 2, kVB = VP * 2;
    extern __shared__ __align__(16) float pool_sums[];             // [waves][C]
    const int lane = threadIdx.x & (kWave - 1), col = lane & 15, quarter = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int head = blockIdx.y, heads = gridDim.y;
    const int64_t n = blockIdx.z;
    const int v = (blockIdx.x * kSpatialMmaWaves + wave) * 16 + col;
    const bool live = v < g.nvec;
    const uint32_t plane_bytes = (uint32_t)g.plane * 2u;
    const __amdgpu_buffer_rsrc_t xr = plane_rsrc(x + n * g.C * (int64_t)g.plane, (uint32_t)g.C * plane_bytes);
    const VectorAt at = vector_of<VP, 1>(g, v);
    const uint32_t xb = live ? (uint32_t)at.in * 2u + (uint32_t)(quarter * 4) * plane_bytes : kOutside;
    constexpr bool kMasked = POOL && RAGGED;
    uint32_t mask[NW];
    if constexpr (kMasked) words_from<__half, NW>(at.again, mask);
    const __amdgpu_buffer_rsrc_t wr = plane_rsrc(w + (int64_t)head * KK * g.C, (uint32_t)(KK * g.C) * 2u);
    const uint32_t wb = col < KK ? (uint32_t)(col * g.C + quarter * 4) * 2u : kOutside;

    uint32_t xw[NST][4][NW], ww[NST][2];
    auto issue = [&](auto st_tag, int i) __attribute__((always_inline)) {
        constexpr int ST = decltype(st_tag)::value;
        const bool have = i < g.ngroups;
        const uint32_t vb = have ? xb : kOutside, cb = (uint32_t)(have ? i * G : 0) * plane_bytes;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if constexpr (VP == 8) {
                const auto q = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)vb, (int)(cb + (uint32_t)u * plane_bytes), 0);
#pragma unroll
                for (int k = 0; k < 4; ++k) xw[ST][u][k] = q[k];
            } else {
                const auto q = __builtin_amdgcn_raw_buffer_load_b64(xr, (int)vb, (int)(cb + (uint32_t)u * plane_bytes), 0);
                xw[ST][u][0] = q[0];
                xw[ST][u][1] = q[1];
            }
        }
        rows::load_words<2>(wr, have ? wb + (uint32_t)i * (G * 2u) : kOutside, ww[ST]);
    };
    float4_t acc[VP];
#pragma unroll
    for (int e = 0; e < VP; ++e) acc[e] = float4_t{0.f, 0.f, 0.f, 0.f};
    float *const sums = pool_sums + wave * g.C + quarter * 4 + (lane & 3);
    auto compute = [&](auto st_tag, int i) __attribute__((always_inline)) {
        constexpr int ST = decltype(st_tag)::value;
        if constexpr (POOL) {
            if (head == 0) {
                const rows::half2_t ones = {(_Float16)1, (_Float16)1};
                float ps[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    float part[NW];
#pragma unroll
                    for (int k = 0; k < NW; ++k)
                        part[k] = __builtin_amdgcn_fdot2(__builtin_bit_cast(rows::half2_t, kMasked ? xw[ST][u][k] & mask[k] : xw[ST][u][k]),
                                                         ones, 0.f, false);
                    ps[u] = NW == 4 ? (part[0] + part[1]) + (part[NW - 2] + part[NW - 1]) : part[0] + part[1];
                }
                // over the row of sixteen lanes: channel (lane & 3) in each (see wave_sums)
                const bool b0 = lane & 1, b1 = lane & 2;
                const float k0 = (b0 ? ps[1] : ps[0]) + from_permuted<0xB1>(b0 ? ps[0] : ps[1]);
                const float k1 = (b0 ? ps[3] : ps[2]) + from_permuted<0xB1>(b0 ? ps[2] : ps[3]);
                float k = (b1 ? k1 : k0) + from_permuted<0x4E>(b1 ? k0 : k1);
                k += from_permuted<0x124 /* row_ror:4 */>(k);
                k += from_permuted<0x128 /* row_ror:8 */>(k);
                if (col < 4 && i < g.ngroups) sums[i * G] = k;
            }
        }
        typedef uint32_t pair_t __attribute__((ext_vector_type(2)));
        const half4_t wv = __builtin_bit_cast(half4_t, pair_t{ww[ST][0], ww[ST][1]});
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            pair_t low, high;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                low[c] = __builtin_amdgcn_perm(xw[ST][2 * c + 1][k], xw[ST][2 * c][k], 0x05040100u);
                high[c] = __builtin_amdgcn_perm(xw[ST][2 * c + 1][k], xw[ST][2 * c][k], 0x07060302u);
            }
            acc[2 * k] = __builtin_amdgcn_mfma_f32_16x16x16f16(wv, __builtin_bit_cast(half4_t, low), acc[2 * k], 0, 0, 0);
            acc[2 * k + 1] = __builtin_amdgcn_mfma_f32_16x16x16f16(wv, __builtin_bit_cast(half4_t, high), acc[2 * k + 1], 0, 0, 0);
        }
    };
    rows::static_for<0, NST - 1>([&](auto q) __attribute__((always_inline)) { issue(q, decltype(q)::value); });
    // this lane's four taps, as stored: they wait for the end of the walk
    _Float16 taps_of[3][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int tap = head * KK + min(quarter * 4 + r, KK - 1);
        taps_of[0][r] = gain_vec ? *reinterpret_cast<const _Float16 *>(gain_vec + tap) : (_Float16)0;
        taps_of[1][r] = offset_vec ? *reinterpret_cast<const _Float16 *>(offset_vec + tap) : (_Float16)0;
        taps_of[2][r] = bias ? *reinterpret_cast<const _Float16 *>(bias + tap) : (_Float16)0;
    }
    // (whole rounds: a group past the last one reads zeros)
    for (int i = 0; i < g.ngroups; i += NST)
        rows::static_for<0, NST>([&](auto q) __attribute__((always_inline)) {
            constexpr int Q = decltype(q)::value;
            issue(std::integral_constant<int, (Q + NST - 1) % NST>{}, i + Q + NST - 1);
            __builtin_amdgcn_sched_barrier(0);
            compute(q, i + Q);
            __builtin_amdgcn_sched_barrier(0);
        });

    const int64_t taps_at = ((n * heads + head) * KK) * (int64_t)g.npix;
    const uint32_t tap_bytes = (uint32_t)g.npix * 2u, all_bytes = KK * tap_bytes;
    uint32_t ob[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int t = quarter * 4 + r;
        ob[r] = live && t < KK ? (uint32_t)at.p * 2u + (uint32_t)t * tap_bytes : kOutside;
    }
    // (taps past the ninth: zero weights, zero bias)
    float gains[4], offsets[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        gains[r] = gain_vec ? (float)taps_of[0][r] : gain;
        offsets[r] = (float)taps_of[1][r];
        const float b = quarter * 4 + r < KK ? (float)taps_of[2][r] : 0.f;
#pragma unroll
        for (int e = 0; e < VP; ++e) acc[e][r] += b;
    }
    auto leave = [&](__half *to) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rr = plane_rsrc(to + taps_at, all_bytes);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float f[VP];
#pragma unroll
            for (int e = 0; e < VP; ++e) f[e] = acc[e][r];
            uint32_t ow[NW];
            rows::pack<__half, VP, float>(f, ow);
            store_vec_nt<kVB>(rr, ob[r], ow);
        }
    };
    if (raw) leave(raw);
    // as normalise() has it, the sums over the taps across the quarters
#pragma unroll
    for (int e = 0; e < VP; ++e) {
        const float mean = rows_total((acc[e][0] + acc[e][1]) + (acc[e][2] + acc[e][3])) / (float)KK;
        float sq = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            acc[e][r] -= mean;
            if (quarter * 4 + r < KK) sq += acc[e][r] * acc[e][r];
        }
        const float inv = 1.f / (sqrtf(rows_total(sq) / (float)(KK - 1)) + 1e-10f);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[e][r] = acc[e][r] * inv * gains[r] + offsets[r];
    }
    leave(sf);
    if constexpr (POOL) {
        if (head != 0) return;
        __syncthreads();
        float *out = pool_part + (n * gridDim.x + blockIdx.x) * g.C;
        for (int c = threadIdx.x; c < g.C; c += kSpatialMmaWaves * kWave)
            out[c] = (pool_sums[c] + pool_sums[g.C + c]) + (pool_sums[2 * g.C + c] + pool_sums[3 * g.C + c]);
    }
}

// out[n * C + c] = sum of parts[(n * nparts + p) * C + c] over p, for 64 channels of a sample: a
// lane loads V of them, eight partial sums at a time, so that 512 of them (V = 4) are one round trip.
constexpr int kCollapseChannels = 64, kCollapseThreads = 1024, kCollapseWaves = kCollapseThreads / kWave;
template <int V>
__global__ __launch_bounds__(kCollapseThreads) void k_collapse_parts(const float *__restrict__ parts,
                                                                     float *__restrict__ out, int C, int nparts) {
    constexpr int LANES = kCollapseChannels / V, GROUPS = kCollapseThreads / LANES, ROUND = 8;
    __shared__ float red[kCollapseWaves][kCollapseChannels];
    const int at = threadIdx.x % LANES * V, grp = threadIdx.x / LANES;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int c = blockIdx.x * kCollapseChannels + at;
    const int64_t n = blockIdx.y;
    const __amdgpu_buffer_rsrc_t r = plane_rsrc(parts + n * nparts * C, (uint32_t)(nparts * C) * 4u);
    float sum[V];
#pragma unroll
    for (int v = 0; v < V; ++v) sum[v] = 0.f;
    for (int q0 = grp; q0 < nparts; q0 += GROUPS * ROUND) {
        uint32_t x[ROUND][V];
#pragma unroll
        for (int u = 0; u < ROUND; ++u) {
            const int q = q0 + u * GROUPS;
            load_vec<V * 4>(r, c < C && q < nparts ? (uint32_t)(q * C + c) * 4u : kOutside, x[u]);
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            auto y = [&](int u) __attribute__((always_inline)) { return __uint_as_float(x[u][v]); };
            sum[v] += ((y(0) + y(1)) + (y(2) + y(3))) + ((y(4) + y(5)) + (y(6) + y(7)));
        }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
        if constexpr (V == 4) sum[v] = rows_total(sum[v]);    // (four groups a wave)
        if (lane < LANES) red[wave][at + v] = sum[v];
    }
    __syncthreads();
    const int i = threadIdx.x, to = blockIdx.x * kCollapseChannels + i;
    if (i >= kCollapseChannels || to >= C) return;
    float total = 0.f;
#pragma unroll
    for (int k = 0; k < kCollapseWaves; ++k) total += red[k][i];
    out[n * C + to] = total;
}

constexpr int kChannelThreads = 1024;  // sixteen waves: the rows of a block's taps are dealt out to them
constexpr int kChannelWaves = kChannelThreads / kWave;

// Products of R weight rows (lane sl of sixteen) with NS vectors in LDS, `pitch` apart.  WIDE: as vectors of 16
// bytes at any element address; sixteen single elements are 64 bytes of a row, 32 in fp16, and the address path
// serves four such rows a load.
template <typename T, int R, int NS, bool WIDE>
__device__ __forceinline__ void row_products(const T *const (&row)[R], int len, const float *x, int pitch, int sl, float (&p)[R][NS]) {
    constexpr int V = WIDE ? 16 / (int)sizeof(T) : 1;
    struct Pack { T e[V]; };
#pragma unroll
    for (int u = 0; u < R; ++u)
#pragma unroll
        for (int s = 0; s < NS; ++s) p[u][s] = 0.f;
#pragma unroll 2
    for (int c = sl * V; c + V <= len; c += 16 * V) {
        Pack w[R];
#pragma unroll
        for (int u = 0; u < R; ++u) __builtin_memcpy(&w[u], row[u] + c, sizeof(Pack));
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            float xv[V];
            __builtin_memcpy(xv, x + s * pitch + c, sizeof(xv));
#pragma unroll
            for (int u = 0; u < R; ++u)
#pragma unroll
                for (int k = 0; k < V; ++k) p[u][s] = fmaf(ld(&w[u].e[k]), xv[k], p[u][s]);
        }
    }
    if constexpr (WIDE) {    // (what is left of a row: less than a vector)
        const int c = len / V * V + sl;
        if (c < len) {
#pragma unroll
            for (int u = 0; u < R; ++u) {
                const float wv = ld(row[u] + c);
#pragma unroll
                for (int s = 0; s < NS; ++s) p[u][s] = fmaf(wv, x[s * pitch + c], p[u][s]);
            }
        }
    }
}
// The same of one long row, eight elements in flight; with few samples the last of them, which may be fewer, too (a
// loop over what is left takes a memory latency for each).
template <typename T, int NS>
__device__ __forceinline__ void row_product(const T *row, int len, const float *x, int pitch, int sl, float (&p)[NS]) {
    constexpr int ROUND = 8, STEP = 16;
#pragma unroll
    for (int s = 0; s < NS; ++s) p[s] = 0.f;
    int c = sl;
    if constexpr (NS < 4) {
        // (zero on both sides past the end: neither may be an infinity's product)
        auto round = [&](auto partial) __attribute__((always_inline)) {
            constexpr bool PARTIAL = decltype(partial)::value;
            T w[ROUND];
#pragma unroll
            for (int k = 0; k < ROUND; ++k) w[k] = row[PARTIAL ? min(c + k * STEP, len - 1) : c + k * STEP];
#pragma unroll
            for (int k = 0; k < ROUND; ++k) {
                const bool in = !PARTIAL || c + k * STEP < len;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const float xv = x[s * pitch + (PARTIAL ? min(c + k * STEP, len - 1) : c + k * STEP)];
                    p[s] = fmaf(in ? ld(&w[k]) : 0.f, in ? xv : 0.f, p[s]);
                }
            }
        };
        for (; c - sl + ROUND * STEP <= len; c += ROUND * STEP) round(std::false_type{});
        if (c - sl < len) round(std::true_type{});
    } else {
#pragma unroll ROUND
        for (; c < len; c += STEP) {
            const float wv = ld(row + c);
#pragma unroll
            for (int s = 0; s < NS; ++s) p[s] = fmaf(wv, x[s * pitch + c], p[s]);
        }
    }
}

// grid (channel blocks of BLOCK channels, groups of NS samples).  LDS: the pooled
// vectors (NS * C floats), the hidden vectors (NS * mid floats), the block's
// un-normalised taps (NS * BLOCK * KK).  Every weight a lane loads serves the NS
// samples of its workgroup (the weights are the same for all samples; re-read
// per sample they cost more L2 bandwidth than anything else here).  Every
// workgroup of a sample recomputes the hidden vector, so the blocks are large:
// smaller ones had all compute units read the same rows of w1 at once, which
// the L2 serves one after the other.  WIDE: rows of w2 as vectors (see the launcher).
template <typename T, int KK, int BLOCK, int NS, bool WIDE>
__global__ __launch_bounds__(kChannelThreads) void k_channel_branch(
    const T *__restrict__ pooled, const T *__restrict__ w1, const T *__restrict__ b1,
    const T *__restrict__ w2, const T *__restrict__ b2, T *__restrict__ cf, int N, int C, int mid,
    float gain, const T *__restrict__ gain_vec, const T *__restrict__ offset_vec,
    const float *__restrict__ parts, int nparts, float scale, ChannelSave save) {
    extern __shared__ float branch_smem[];
    float *v = branch_smem;            // [NS][C]
    float *h = v + NS * C;             // [NS][mid]
    float *f = h + NS * mid;           // [NS][BLOCK * KK]
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int64_t n0 = (int64_t)blockIdx.y * NS;
    const int ns = min(NS, N - (int)n0);   // samples of this workgroup (the others: copies of the last)
    const int cb = blockIdx.x * BLOCK;
    constexpr int RT = NS >= 4 ? 1 : NS == 2 ? 2 : 3;
    const int seg = lane >> 4, sl = lane & 15;
    const int rows = min(BLOCK, C - cb) * KK;
    TapParams<T, KK> params;
    // the pooled vectors: given, or scale * the sum of nparts partial sums per value
    // (parts[(n * nparts + p) * C + c], what k_spatial_stream leaves); of many of them as many
    // threads share a value's as there are
    const int values = NS * C, share = parts && nparts > kMmaRound ? kChannelThreads / values : 1;
    const int g = threadIdx.x / values;
    auto part_sum = [&](int i, int first, int step) __attribute__((always_inline)) {
        const int s = i / C, c = i - s * C;
        const float *src = parts + (n0 + min(s, ns - 1)) * nparts * C + c;
        float a = 0.f;
#pragma unroll 8
        for (int q = first; q < nparts; q += step) a += src[(int64_t)q * C];
        return a;
    };
    auto put_pooled = [&](int i, float a) __attribute__((always_inline)) {
        v[i] = a;
        const int s = i / C;
        if (save.pooled && blockIdx.x == 0 && s < ns) save.pooled[n0 * C + i] = a;
    };
    if (share > 1) {
        __shared__ float red[kChannelThreads];
        if (g < share) red[threadIdx.x] = part_sum(threadIdx.x - g * values, g, share);
        __syncthreads();
        if (g == 0) {
            float a = red[threadIdx.x];
            for (int k = 1; k < share; ++k) a += red[k * values + threadIdx.x];
            put_pooled(threadIdx.x, a * scale);
        }
    } else {
        for (int i = threadIdx.x; i < values; i += kChannelThreads)
            put_pooled(i, parts ? part_sum(i, 0, 1) * scale : ld(pooled + (n0 + min(i / C, ns - 1)) * C + i % C));
    }
    __syncthreads();
    // Dot products with sixteen lanes along a weight row and four rows per wave at a
    // time: each ends in a reduction over a row of 16 lanes (four lane-permute
    // additions for four results; a whole wave per row paid thirteen for one).
    // hidden vectors: rows of w1
    for (int m0 = wave * 4; m0 < mid; m0 += kChannelWaves * 4) {
        const int m = min(m0 + seg, mid - 1);
        float p[NS];
        row_product<T, NS>(w1 + (int64_t)m * C, C, v, C, sl, p);
        const float bias = b1 ? ld(b1 + m) : 0.f;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const float tot = row_sum(p[s]);
            if (sl == 0 && m0 + seg < mid) {
                const float hm = relu(tot + bias);
                h[s * mid + m0 + seg] = hm;
                if (save.hidden && blockIdx.x == 0 && s < ns) save.hidden[(n0 + s) * mid + m0 + seg] = hm;
            }
        }
    }
    __syncthreads();
    // the block's taps: rows (cb * KK + r) of w2, RT passes of four rows in flight per wave
    auto emit = [&](int r, int s, float p, float bias) __attribute__((always_inline)) {
        const float tot = row_sum(p);
        if (sl == 0 && r < rows) {
            f[s * BLOCK * KK + r] = tot + bias;
            if (save.taps && s < ns) save.taps[((n0 + s) * C + cb) * KK + r] = tot + bias;
        }
    };
    for (int r0 = wave * 4 * RT; r0 < rows; r0 += kChannelWaves * 4 * RT) {
        float p[RT][NS];
        const T *wrow[RT];
#pragma unroll
        for (int u = 0; u < RT; ++u) wrow[u] = w2 + ((int64_t)cb * KK + min(r0 + 4 * u + seg, rows - 1)) * mid;
        row_products<T, RT, NS, WIDE>(wrow, mid, h, mid, sl, p);
#pragma unroll
        for (int u = 0; u < RT; ++u) {
            const int r = r0 + 4 * u + seg;
            const float bias = (b2 && r < rows) ? ld(b2 + (int64_t)cb * KK + r) : 0.f;
#pragma unroll
            for (int s = 0; s < NS; ++s) emit(r, s, p[u][s], bias);
        }
    }
    __syncthreads();
    // one thread per (sample, channel) normalises the KK taps
    for (int i = threadIdx.x; i < NS * BLOCK; i += kChannelThreads) {
        const int s = i / BLOCK, ch = i - s * BLOCK;
        if (s >= ns || cb + ch >= C) continue;
        float u[KK];
#pragma unroll
        for (int t = 0; t < KK; ++t) u[t] = f[(s * BLOCK + ch) * KK + t];
        params.load(cb + ch, gain, gain_vec, offset_vec, (const T *)nullptr);   // (b2 is in f already)
        normalise<T, KK>(u, params);
        T *op = cf + ((n0 + s) * C + cb + ch) * KK;
#pragma unroll
        for (int t = 0; t < KK; ++t) st(op + t, u[t]);
    }
}

template <typename T, bool SAVE>
__global__ __launch_bounds__(kRowsThreads) void k_channel_branch_rows(ChannelRows<T> a) {
    extern __shared__ __align__(16) unsigned char rows_smem[];
    channel_rows<T, SAVE>(a, blockIdx.x, blockIdx.y, rows_smem, Nothing(), Nothing(), Nothing(), ToFilter<T, kRowsKK>{a.cf, a.C});
}

template <int KK, bool SAVE>
__global__ __launch_bounds__(kMmaThreads) void k_channel_branch_mma(ChannelMma a) {
    extern __shared__ __align__(16) unsigned char mma_smem[];
    const int n0 = blockIdx.y * kMmaSamples;
    channel_mma<KK, SAVE>(a, blockIdx.x, n0, min(kMmaSamples, a.N - n0), mma_smem, Nothing(), Nothing(),
                          Nothing(), ToFilter<__half, KK>{a.cf, a.C});
}

}  // namespace

bool branch_kernel_size_built(int k) { return k == 3 || k == 5; }

int64_t parts_left(int64_t N, int64_t C, int64_t mid, int esz) { return channel_parts_left(N, C, mid, esz); }
hipError_t collapse_parts(const float *parts, int nparts, float *totals, int64_t N, int64_t C, hipStream_t st) {
    const dim3 grid((unsigned)cdiv(C, kCollapseChannels), (unsigned)N);
    if (C % 4 == 0 && (uintptr_t)parts % 16 == 0)
        hipLaunchKernelGGL((k_collapse_parts<4>), grid, dim3(kCollapseThreads), 0, st, parts, totals, (int)C, nparts);
    else
        hipLaunchKernelGGL((k_collapse_parts<1>), grid, dim3(kCollapseThreads), 0, st, parts, totals, (int)C, nparts);
    return hipGetLastError();
}

// Launch of k_spatial_stream; hipErrorNotSupported where it does not cover the problem
// (the caller then takes the kernels above).
template <typename T>
hipError_t spatial_stream(const T *x, const T *w, const T *bias, T *sf, int64_t N, int64_t C, int64_t H,
                          int64_t W, int head, int stride, double gain, const T *gain_vec,
                          const T *offset_vec, hipStream_t st, float *pool_part = nullptr,
                          int64_t pool_capacity = 0, int *pool_parts = nullptr, T *raw = nullptr) {
    constexpr int KK = 9, NST = 3;
    constexpr int U = sizeof(T) == 2 ? 4 : 2;
    constexpr int esz = (int)sizeof(T);
    const int64_t Ho = H / stride, Wo = W / stride, npix = Ho * Wo;
    if (tune_int("DDF_TUNE_SPATIAL_STREAM", 1) == 0) return hipErrorNotSupported;
    if (stride != 1 && stride != 2) return hipErrorNotSupported;
    if (C % U != 0 || ((uintptr_t)w % 4) != 0) return hipErrorNotSupported;
    if (C * H * W * esz >= (1ll << 31) || KK * npix * esz >= (1ll << 31)) return hipErrorNotSupported;
    // pixels per lane: the widest vector the shapes and addresses allow ...
    const bool pool = pool_part != nullptr;
    if (pool && stride == 2 && (H % 2 != 0 || W % 2 != 0)) return hipErrorNotSupported;   // (pixels no lane covers)
    // (vectors lie at any element address; a run or a row as long as one has them, see vector_of)
    auto fits = [&](int vp) {
        if (pool && stride == 2 && vp == 1) return ((uintptr_t)x % (2 * esz)) == 0;   // (pairs of columns)
        return (stride == 1 ? npix : Wo) >= vp;
    };
    auto divides = [&](int vp) { return (stride == 1 ? npix : Wo) % vp == 0; };
    auto vectors = [&](int vp) { return stride == 1 ? cdiv(npix, (int64_t)vp) : Ho * cdiv(Wo, (int64_t)vp); };
    const int vp_max = (stride == 1 ? 16 : 8) / esz;
    // ... that still leaves enough waves to fill the machine: the waves of a workgroup
    // share its pixels and split the channels, at least two pipeline rounds each
    // (measured over batches of 1 to 128, 7 x 7 to 200 x 300, 64 to 512 channels: 1 280 waves
    // are enough at four or eight pixels per lane, and single-pixel loads only pay where two
    // pixels per lane leave fewer than 448 - 64 x 128 x 56 x 56 fp16 under stride 2 took
    // 23.7 us at one pixel and takes 15.3 at two, 16 x 128 x 28 x 28 8.5 and 6.5)
    auto enough = [](int vp) { return vp == 2 ? 448 : 1280; };
    const int64_t want = 2048;
    int vp = 0, waves = 1;
    for (int cand = vp_max; cand >= 1; cand /= 2) {
        if (!fits(cand)) continue;
        const int64_t nvec = vectors(cand);
        const int64_t tiles = cdiv(nvec, kWave) * N * head;
        int wv = 1;
        // (nearly a wave per SIMD with whole channel walks: better than splitting them.  With few waves the walk is all
        // there is: four share it where that leaves one round each, eight where they are fewest.  us of a layer's
        // inference, two rounds each at least / so: fp16 7 x 44 x 30 x 24 with two heads 20.1 / 14.4, 1 x 40 x 40 x 43 18.0 / 12.7, 8 x 40 x
        // 23 x 32 19.7 / 14.1, fp32 54 x 88 x 12 x 8 under stride 2 14.8 / 13.9; eight from more waves on 61 x 140 x 8 x 7 15.2 /
        // 16.2, sixteen 7 x 144 x 25 x 24 14.9 / 15.9; 200 sizes drawn at random 2.3 % on average.)
        auto round_is_enough = [&](int wv) { return tiles * wv <= (wv <= 2 ? 512 : wv == 4 ? 128 : 0); };
        if (tiles < tune_int("DDF_TUNE_SPATIAL_WHOLE", 768))
            while (wv < 16 && wv * 2 * cand <= 32 && tiles * wv < want &&
                   (C / U) / (wv * 2) >= (round_is_enough(wv) ? NST : 2 * NST))
                wv *= 2;
        // Vectors that do not divide the run, where half as wide ones do not either (or are single pixels): where they
        // fill the machine, with a quarter to spare where a workgroup is sixteen waves, whose sums meet in
        // four rounds, or from 1 280 whole walks on, and leave a fifth of the lanes idle at most.  us of a layer's
        // inference, single pixels (or pairs) / such vectors: fp32 11 x 184 x 79 x 77 56.4 / 43.9, 16 x 128 x 57 x 55 37.9 /
        // 27.2, 26 x 48 x 65 x 145 41.9 / 39.4, stride 2 8 x 256 x 98 x 98 45.2 / 40.2, fp16 8 x 64 x 199 x 301 71.8 / 60.4,
        // 16 x 176 x 57 x 55 39.3 / 30.6; left alone 64 x 256 x 15 x 15 26.7 / 27.3, 32 x 256 x 7 x 7 17.1 / 18.1, two heads of
        // 48 x 432 x 15 x 19 48.0 / 49.8 and 1 x 324 x 165 x 238 52.4 / 56.0, stride 2 32 x 256 x 26 x 30 23.2 / 26.5.
        // Under stride 2 the workgroups of head 0 add up the planes and take longest: not where several heads' of eight waves
        // are a round and a part (branch alone, fp32, four heads: 5 x 412 x 74 x 82 23.7 / 40.2, 43 x 360 x 34 x 26 30.3 / 43.9, 4 x 312 x 92 x 98
        // 25.6 / 33.8; a round of fp16 2 x 428 x 136 x 118 26.8 / 17.7, more 6 x 260 x 78 x 102 31.2 / 19.6; rows of a few pixels not measured).
        const bool part_round = stride == 2 && head > 1 && Wo >= 8 && wv == 8 && tiles * wv > want && tiles * wv < 2800;
        if (!divides(cand) && (part_round || (cand > 2 && divides(cand / 2)) || nvec * 5 < cdiv(nvec, kWave) * kWave * 4 ||
                               tiles * wv < (wv == 16 ? want + want / 4 : wv == 1 ? 1280 : want)))
            continue;
        vp = cand;
        waves = wv;
        if (tiles * wv >= enough(cand) || wv == 1) break;
    }
    const int fvp = tune_int("DDF_TUNE_SPATIAL_VP", 0), fwv = tune_int("DDF_TUNE_SPATIAL_WAVES", 0);
    if (fvp > 0 && fvp <= vp_max && fits(fvp)) vp = fvp;
    if (fwv > 0) waves = fwv;
    // fp16, stride 1: on the matrix cores where that leaves enough workgroups at work: its four waves
    // walk all channels of their pixels, so few of them are one long walk behind another, which
    // k_spatial_stream splits over waves.  Counted in workgroups full of pixels: 64 at up to 80
    // channels, 128 at up to 256, 256 beyond.  Vectors of eight pixels from 256 on (768 at up to 64
    // channels), of four below, or of eight where those of four leave too many partial sums.  An odd
    // number of 16-channel groups walks one more: of three that is too much for large planes.  (With
    // the sums or without: the same kernel, so the same bits.)  us without the pooled sums / with them
    // and the channel branch behind, operands from memory, k_spatial_stream -> here: 128 x 64 x 56 x 56
    // 13.6 / 20.7 -> 14.2 / 20.2, 128 x 128 x 28 x 28 10.9 / 17.8 -> 9.6 / 15.8, 8 x 64 x 200 x 300 16.0 / 22.2 ->
    // 15.5 / 21.8, 16 x 64 x 56 x 56 6.7 / 13.2 -> 5.8 / 12.0, 21 x 320 x 48 x 68 18.4 / 28 -> 14.6 / 24; left to
    // it: 128 x 256 x 14 x 14 (98 full ones) 8.0 / 15.7, here 9.5 / 16.4; 64 x 256 x 14 x 14 7.3 / 14.9, 9.3 /
    // 16.4; 32 x 256 x 28 x 28 8.0 / 15.6, 9.6 / 16.9; 24 x 512 x 28 x 28 9.9 / 20.5, 14.6 / 25.4; 54 x 48 x 106 x 84
    // 12.8 / 18.9, 14.0 / 20.9.  (943 sizes: 1.6 / 0.8 % over the best of the three on average,
    // k_spatial_stream throughout 2.9 / 4.3 %.)
    bool mma = false;
    if constexpr (esz == 2) {
        if (stride == 1 && C % kSpatialMmaGroup == 0 && C <= kSpatialMmaChannels && (uintptr_t)w % 16 == 0 &&
            tune_int("DDF_TUNE_SPATIAL_MMA", 1) != 0) {
            constexpr int kPixels = 4 * kWave;     // of a workgroup, four per lane
            const int64_t tiles8 = cdiv(vectors(8), kWave), tiles4 = cdiv(vectors(4), kWave), left = channel_parts_left(N, C, C / 5, esz);
            // Vectors that do not divide the plane: of eight where seven tenths of the lanes have one, of four where half
            // have (three tenths from four channel groups on), all of them counted in pixels.  Small odd planes leave a
            // workgroup with a few vectors whatever their number: us, both branches, k_spatial_stream / vectors of four / of eight,
            // 1563 x 32 x 7 x 7 18.3 / 21.5 / 26.3, 700 x 256 x 7 x 7 22.9 / 27.7 / -, 819 x 32 x 11 x 11 13.6 / 14.3 / 16.8, 537 x 48 x 14 x 14
            // - / 15.1 / 17.2, 148 x 80 x 26 x 26 18.7 / 15.8 / 17.7, but 635 x 160 x 9 x 9 27 / 21.6, 114 x 80 x 29 x 29 16.1 / - / 13.4.  (900 sizes:
            // 1.9 % over the best of the three, 4.8 % without, a third of the worst 1.4 times as long as k_spatial_stream.)
            auto lanes = [&](int vp, int64_t tiles, int tenths) { return divides(vp) || vectors(vp) * 10 >= tiles * kWave * tenths; };
            const int64_t full = head * (C <= 64 && divides(4) ? N * tiles4 : N * npix / kPixels);
            const bool odd = (C / kSpatialMmaGroup) % 2 != 0 && C < 64;
            const bool wide = fits(8) && lanes(8, tiles8, 7) && full >= (odd ? 2048 : C <= 64 ? 768 : 256);
            const bool narrow = fits(4) && lanes(4, tiles4, C < 64 ? 5 : 3) && full >= (C <= 80 ? 64 : C <= 256 ? 128 : 256) &&
                                !(odd && full >= 512);
            if (wide || narrow) {
                mma = true;
                vp = wide || (pool && fits(8) && tiles4 > left && tiles8 <= left) ? 8 : 4;
                waves = 1;
            }
        }
    }
    if (vp == 0) return hipErrorNotSupported;
    if (vp * waves > 32 || (waves & (waves - 1)) != 0 || waves > 16) return hipErrorNotSupported;   // (the variants built)
    SpatialGeom g;
    g.C = (int)C; g.W = (int)W; g.Wo = (int)Wo;
    g.plane = (int)(H * W);
    g.npix = (int)npix;
    g.nvec = (int)vectors(vp);
    g.vrow = (int)cdiv(Wo, (int64_t)vp);
    const bool ragged = !divides(vp);
    const int tiles = (int)cdiv(g.nvec, kWave);
    g.lpt = (int)cdiv(g.nvec, tiles);                   // (tiles of equal size)
    g.ngroups = (int)(mma ? C / kSpatialMmaGroup : C / U);
    g.gpw = (int)cdiv(g.ngroups, waves);
    g.steps = (int)cdiv(g.gpw, NST) * NST;
    if (N > 65535 || head > 65535) return hipErrorNotSupported;
    bool collapse = false;
    if (pool) {
        // (more tiles than the channel branch is left - with the hidden layer that a layer has unless
        // it is told otherwise, a fifth of the channels: their sums go behind the N * C totals that
        // k_collapse_parts then makes of them)
        collapse = tiles > tune_int("DDF_TUNE_COLLAPSE", (int)std::min<int64_t>(channel_parts_left(N, C, C / 5, esz), 1 << 30));
        if (N * (tiles + (collapse ? 1 : 0)) * C > pool_capacity) return hipErrorInvalidValue;
        *pool_parts = collapse ? 1 : tiles;
    }
    float *parts_out = collapse ? pool_part + N * C : pool_part;
    const dim3 grid((unsigned)tiles, (unsigned)head, (unsigned)N);
    if constexpr (esz == 2) {
        if (mma) {
            const int lds = pool ? kSpatialMmaWaves * g.C * (int)sizeof(float) : 0;
#define DDF_SPATIAL_MMA(VP_, POOL_, RAGGED_)                                                      \
    hipLaunchKernelGGL((k_spatial_mma<VP_, POOL_, RAGGED_>), grid, dim3(kSpatialMmaWaves * kWave), lds, st, g, x, w, bias, \
                       sf, (float)gain, gain_vec, offset_vec, parts_out, raw)
            if (vp == 8 && pool && ragged) DDF_SPATIAL_MMA(8, true, true);
            else if (vp == 8 && pool) DDF_SPATIAL_MMA(8, true, false);
            else if (vp == 8) DDF_SPATIAL_MMA(8, false, false);
            else if (pool && ragged) DDF_SPATIAL_MMA(4, true, true);
            else if (pool) DDF_SPATIAL_MMA(4, true, false);
            else DDF_SPATIAL_MMA(4, false, false);
#undef DDF_SPATIAL_MMA
            if (collapse) return collapse_parts(parts_out, tiles, pool_part, N, C, st);
            return hipGetLastError();
        }
    }
#define DDF_STREAM_LAUNCH(VP_, S_, WAVES_)                                                        \
    do {                                                                                          \
        if (pool && ragged) {                                                                     \
            hipLaunchKernelGGL((k_spatial_stream<T, KK, VP_, S_, WAVES_, U, NST, true, (VP_ > 1)>), grid, \
                               dim3(WAVES_ * kWave), 0, st, g, x, w, bias, sf, (float)gain,       \
                               gain_vec, offset_vec, parts_out, raw);                             \
            break;                                                                                \
        }                                                                                         \
        if (pool) {                                                                               \
            hipLaunchKernelGGL((k_spatial_stream<T, KK, VP_, S_, WAVES_, U, NST, true>), grid,    \
                               dim3(WAVES_ * kWave), 0, st, g, x, w, bias, sf, (float)gain,       \
                               gain_vec, offset_vec, parts_out, raw);                             \
            break;                                                                                \
        }                                                                                         \
        hipLaunchKernelGGL((k_spatial_stream<T, KK, VP_, S_, WAVES_, U, NST, false>), grid,       \
                           dim3(WAVES_ * kWave), 0, st, g, x, w, bias, sf, (float)gain, gain_vec, \
                           offset_vec, (float *)nullptr, (T *)nullptr);                           \
    } while (0)
#define DDF_STREAM_WAVES(VP_, S_)                                                                 \
    do {                                                                                          \
        if (waves == 1) DDF_STREAM_LAUNCH(VP_, S_, 1);                                            \
        else if (waves == 2) DDF_STREAM_LAUNCH(VP_, S_, 2);                                       \
        else if (waves == 4) DDF_STREAM_LAUNCH(VP_, S_, 4);                                       \
        else if (waves == 8 && VP_ <= 4) DDF_STREAM_LAUNCH((VP_ <= 4 ? VP_ : 1), S_, 8);          \
        else if (waves == 16 && VP_ <= 2) DDF_STREAM_LAUNCH((VP_ <= 2 ? VP_ : 1), S_, 16);        \
        else return hipErrorNotSupported;                                                         \
    } while (0)
    if (stride == 1) {
        if (vp == 8) { if constexpr (esz == 2) DDF_STREAM_WAVES(8, 1); else return hipErrorNotSupported; }
        else if (vp == 4) DDF_STREAM_WAVES(4, 1);
        else if (vp == 2) DDF_STREAM_WAVES(2, 1);
        else DDF_STREAM_WAVES(1, 1);
    } else {
        if (vp == 4) { if constexpr (esz == 2) DDF_STREAM_WAVES(4, 2); else return hipErrorNotSupported; }
        else if (vp == 2) DDF_STREAM_WAVES(2, 2);
        else DDF_STREAM_WAVES(1, 2);
    }
#undef DDF_STREAM_WAVES
#undef DDF_STREAM_LAUNCH
    if (collapse) return collapse_parts(parts_out, tiles, pool_part, N, C, st);
    return hipGetLastError();
}

template <typename T>
hipError_t spatial_branch(const T *x, const T *w, const T *bias, T *sf, int64_t N, int64_t C,
                          int64_t H, int64_t W, int head, int k, int stride, double gain,
                          const T *gain_vec, const T *offset_vec, hipStream_t st, float *pool_part,
                          int64_t pool_capacity, int *pool_parts, T *raw) {
    const int64_t Ho = H / stride, Wo = W / stride;
    if (N == 0 || C == 0 || Ho * Wo == 0 || head == 0) return hipSuccess;
    if (N > 65535 || head > 65535 || C > (1 << 24) || H * W >= (1ll << 31)) return hipErrorNotSupported;
    if (k == 3) {
        const hipError_t err = spatial_stream<T>(x, w, bias, sf, N, C, H, W, head, stride, gain, gain_vec,
                                                 offset_vec, st, pool_part, pool_capacity, pool_parts, raw);
        if (err != hipErrorNotSupported) return err;
    }
    if (pool_part) return hipErrorNotSupported;   // (only the streaming kernel pools)
    const int waves = k == 3 ? 8 : 4;
    // channels staged in LDS at a time: all of them up to kChunk, a multiple of 8 per wave
    // (and so of the 16 the tile kernel keeps in flight)
    const int chunk = (int)std::min<int64_t>(kChunk, (C + 8 * waves - 1) / (8 * waves) * (8 * waves));
    // Planes with many pixels: a wave per pixel tile, as wide a vector per lane as
    // rows and alignment allow while the waves still fill the machine.
    if (stride == 1 && tune_int("DDF_TUNE_SPATIAL_TILES", 1) != 0) {
        for (int vp = 16 / (int)sizeof(T); vp >= 1; vp /= 2) {
            if (k == 5 && vp > 2) continue;   // (25 taps: the accumulators of two pixels per lane)
            if (W % vp != 0 || (((uintptr_t)x | (uintptr_t)sf) % (vp * sizeof(T))) != 0) continue;
            if (vp == 1 && sizeof(T) == 2) continue;   // (2-byte loads: the shared-pixel kernel does better)
            if ((Ho * Wo) % vp != 0 || N * head * cdiv(Ho * Wo, kWave * vp) < tune_int("DDF_TUNE_SPATIAL_TILES_MIN", 1024)) continue;
            const dim3 grid((unsigned)cdiv(Ho * Wo, 4 * kWave * vp), (unsigned)head, (unsigned)N);
#define DDF_TILES_CASE(KK_, VP_)                                                                \
    hipLaunchKernelGGL((k_spatial_branch_tiles<T, KK_, VP_>), grid, dim3(4 * kWave), 0, st, x, w, \
                       bias, sf, (int)C, (int)H, (int)W, (int)Ho, (int)Wo, stride, chunk,       \
                       (float)gain, gain_vec, offset_vec)
            if (k == 3 && vp == 8) { if constexpr (sizeof(T) == 2) DDF_TILES_CASE(9, 8); }
            else if (k == 3 && vp == 4) DDF_TILES_CASE(9, 4);
            else if (k == 3 && vp == 2) DDF_TILES_CASE(9, 2);
            else if (k == 3) DDF_TILES_CASE(9, 1);
            else if (k == 5 && vp == 2) DDF_TILES_CASE(25, 2);
            else if (k == 5) DDF_TILES_CASE(25, 1);
            else return hipErrorNotSupported;
#undef DDF_TILES_CASE
            return hipGetLastError();
        }
    }
    // Few pixels (or strided sampling): the waves of a workgroup share 64 pixels and
    // split the channels (as many waves as the LDS of the per-wave sums allows).
    const dim3 grid((unsigned)cdiv(Ho * Wo, kWave), (unsigned)head, (unsigned)N);
#define DDF_SPATIAL_CASE(KK_, WAVES_, VP_)                                                      \
    hipLaunchKernelGGL((k_spatial_branch<T, KK_, WAVES_, VP_>), grid, dim3(WAVES_ * kWave), 0, st, x, \
                       w, bias, sf, (int)C, (int)H, (int)W, (int)Ho, (int)Wo, stride, chunk,    \
                       (float)gain, gain_vec, offset_vec)
    // (vectors of pixels per lane where rows and alignment allow: fewer, wider loads)
    int vp = 1;
    // (two-byte elements; four-byte ones gain nothing from it)
    if (stride == 1 && k == 3 && sizeof(T) == 2) {
        for (int cand = tune_int("DDF_TUNE_SPATIAL_VP", 4); cand > 1; cand /= 2)
            if (W % cand == 0 && (((uintptr_t)x | (uintptr_t)sf) % (cand * sizeof(T))) == 0 &&
                N * head * cdiv(Ho * Wo, kWave * cand) >= 256) {
                vp = cand;
                break;
            }
    }
    const dim3 grid_v((unsigned)cdiv(Ho * Wo, kWave * vp), (unsigned)head, (unsigned)N);
    if (k == 3 && vp == 4) {
        hipLaunchKernelGGL((k_spatial_branch<T, 9, 8, 4>), grid_v, dim3(8 * kWave), 0, st, x, w, bias, sf,
                           (int)C, (int)H, (int)W, (int)Ho, (int)Wo, stride, chunk, (float)gain, gain_vec,
                           offset_vec);
    } else if (k == 3 && vp == 2) {
        hipLaunchKernelGGL((k_spatial_branch<T, 9, 8, 2>), grid_v, dim3(8 * kWave), 0, st, x, w, bias, sf,
                           (int)C, (int)H, (int)W, (int)Ho, (int)Wo, stride, chunk, (float)gain, gain_vec,
                           offset_vec);
    } else if (k == 3) DDF_SPATIAL_CASE(9, 8, 1);
    else if (k == 5) DDF_SPATIAL_CASE(25, 4, 1);
    else return hipErrorNotSupported;
#undef DDF_SPATIAL_CASE
    return hipGetLastError();
}

// The matrix-core kernel where it applies (fp16, a hidden layer of at least one
// step of the matrix instruction, whole steps of channels, operands aligned for
// its vector loads); hipErrorNotSupported otherwise.
template <typename T>
hipError_t channel_branch_mma(const T *, const T *, const T *, const T *, const T *, T *, int64_t, int64_t,
                              int64_t, int, double, const T *, const T *, hipStream_t, const float *, int,
                              double, const ChannelSave &) {
    return hipErrorNotSupported;
}
template <>
hipError_t channel_branch_mma<__half>(const __half *pooled, const __half *w1, const __half *b1,
                                      const __half *w2, const __half *b2, __half *cf, int64_t N, int64_t C,
                                      int64_t mid, int k, double gain, const __half *gain_vec,
                                      const __half *offset_vec, hipStream_t st, const float *parts,
                                      int nparts, double scale, const ChannelSave &save) {
    if (tune_int("DDF_TUNE_CHANNEL_MMA", 1) == 0) return hipErrorNotSupported;
    auto aligned = [](const void *p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; };
    if ((k != 3 && k != 5) || !channel_mma_covers(C, mid, k * k) || N > (int64_t)65535 * kMmaSamples)
        return hipErrorNotSupported;
    if (!aligned(w1, 16) || !aligned(cf, 8) || !aligned(b2, 8) || !aligned(gain_vec, 8) ||
        !aligned(offset_vec, 8) || !aligned(w2, 2) || (parts ? !aligned(parts, 16) : !aligned(pooled, 8)))
        return hipErrorNotSupported;
    const ChannelMma a{pooled, w1, b1, w2, b2, cf, (int)N, (int)C, (int)mid, (float)gain, gain_vec, offset_vec,
                       parts, nparts, (float)scale, save, channel_mma_lds(C, mid, k * k)};
    const dim3 grid((unsigned)cdiv(C, kMmaChannels), (unsigned)cdiv(N, kMmaSamples));
    const size_t lds = a.lds.total;
    const bool saves = save.pooled || save.hidden || save.taps;
    if (k == 3 && saves) hipLaunchKernelGGL((k_channel_branch_mma<9, true>), grid, dim3(kMmaThreads), lds, st, a);
    else if (k == 3) hipLaunchKernelGGL((k_channel_branch_mma<9, false>), grid, dim3(kMmaThreads), lds, st, a);
    else if (saves) hipLaunchKernelGGL((k_channel_branch_mma<25, true>), grid, dim3(kMmaThreads), lds, st, a);
    else hipLaunchKernelGGL((k_channel_branch_mma<25, false>), grid, dim3(kMmaThreads), lds, st, a);
    return hipGetLastError();
}

template <typename T>
hipError_t channel_branch(const T *pooled, const T *w1, const T *b1, const T *w2, const T *b2,
                          T *cf, int64_t N, int64_t C, int64_t mid, int k, double gain,
                          const T *gain_vec, const T *offset_vec, hipStream_t st, const float *parts,
                          int nparts, double scale, ChannelSave save) {
    if (N == 0 || C == 0) return hipSuccess;
    const int kk = k * k;
    if (hipError_t e = channel_branch_mma(pooled, w1, b1, w2, b2, cf, N, C, mid, k, gain, gain_vec,
                                          offset_vec, st, parts, nparts, scale, save);
        e != hipErrorNotSupported)
        return e;
    if (k == 3) {
        ChannelRows<T> a{pooled, w1, b1, w2, b2, cf, (int)N, (int)C, (int)mid, (float)gain, gain_vec, offset_vec,
                         parts, nparts, (float)scale, save};
        if (channel_rows_plan(a) && N * cdiv(C, a.block) <= tune_int("DDF_TUNE_CHANNEL_ROWS", 1 << 30)) {
            const dim3 grid((unsigned)cdiv(C, a.block), (unsigned)N);
            if (save.pooled || save.hidden || save.taps)
                hipLaunchKernelGGL((k_channel_branch_rows<T, true>), grid, dim3(kRowsThreads), a.total, st, a);
            else
                hipLaunchKernelGGL((k_channel_branch_rows<T, false>), grid, dim3(kRowsThreads), a.total, st, a);
            return hipGetLastError();
        }
    }
    // (wide layers: fewer, larger blocks, as every block of a sample recomputes the hidden vector, unless smaller ones
    // still have a compute unit each: fp32 32 x 512 12.8 us in blocks of 128, 10.2 of 64; 44 x 512 13.2 and 13.9)
    const int block = C >= 512 && cdiv(C, 64) * N > 256 ? 128 : 64;
    // samples per workgroup: as many as keep every compute unit busy and fit the LDS
    auto lds_of = [&](int ns) { return ((size_t)C + (size_t)mid + (size_t)block * kk) * ns * sizeof(float); };
    int ns = 1;
    const int forced = tune_int("DDF_TUNE_CHANNEL_NS", 0);
    while (ns < 4 && cdiv(C, block) * cdiv(N, ns * 2) >= 256 && lds_of(ns * 2) <= 48 * 1024) ns *= 2;
    if (forced == 1 || forced == 2 || forced == 4) ns = forced;
    const size_t lds = lds_of(ns);
    if (N > 65535 * ns || mid < 1 || lds > 48 * 1024) return hipErrorNotSupported;
    const dim3 grid((unsigned)cdiv(C, block), (unsigned)cdiv(N, ns));
    // Rows of w2 as vectors: where they take fewer round trips to memory than single elements, two of either in flight and
    // what is less than a vector behind them, or as many where a row is longer than 32 (not of two samples in fp16).  us, single elements /
    // vectors: fp32 32 x 512 13.4 / 10.2, 64 x 512 20.6 / 14.3, 128 x 512 21.6 / 16.5, 250 x 200 11.5 / 10.4, 100 x 156 with 20 hidden values
    // 8.9 / 7.7, with 16 7.0 / 7.7, with 39 10.6 / 9.2, 5 x 5 taps 64 x 256 16.6 / 13.1, fp16 56 x 456 18.0 / 14.3, 40 x 1000 35.4 / 29.2, 100 x 156
    // with 24 9.3 / 8.6, with 32 8.0 / 8.6, two samples 307 x 164 with 41 12.3 / 13.3, with 56 13.1 / 12.0.
    // More samples, or longer rows of fp16: the vectors of x take their time in LDS (fp16 500 x 200 17.9 / 29.9, 128 x 456 20.8 / 25.8, two
    // samples 128 x 584 with 292 hidden values 50 / 59, fp32 391 x 346 42.6 / 47.6), which is had back where rows come from far: a block's are a
    // megabyte, or less where the blocks do not divide the XCDs, each of which otherwise keeps its block's rows in its L2 (fp32 300 x 1024
    // 125 / 150, but 132 x 998 with 499 hidden values 343 / 287, 253 x 896 80.3 / 73.1, 300 x 1028 201 / 167, fp16 5 x 5 taps 128 x 548 with 274
    // 256 / 170).  (Rows of w1 as vectors as well: fp32 300 x 1024 182, fp16 40 x 1000 38.5.)
    auto trips = [](int64_t n) { return n / 32 + (n % 32 == 0 ? 0 : n % 32 <= 16 ? 1 : 2); };
    constexpr int V = 16 / (int)sizeof(T);
    constexpr bool kHalf = sizeof(T) == 2;
    const int64_t singles = trips(mid), wide = trips(mid / V) + (mid % V ? 1 : 0), blocks = cdiv(C, block);
    const int64_t row_bytes = block * kk * mid * (int64_t)sizeof(T);
    const bool far = block == 128 && (row_bytes >= 1 << 20 || (8 % blocks != 0 && (row_bytes >= 3 << 18 || blocks > 6)));
    const bool fewer = wide < singles || (wide == singles && mid > 32 && !(kHalf && ns == 2));
    const bool vectors = ns == 1 ? wide < singles || mid > 32 : ns == 2 ? fewer && (!kHalf || mid <= 128 || far) : !kHalf && far;
#define DDF_CHANNEL_LAUNCH(KK_, BLOCK_, NS_, WIDE_)                                              \
    hipLaunchKernelGGL((k_channel_branch<T, KK_, BLOCK_, NS_, WIDE_>), grid, dim3(kChannelThreads), lds, \
                       st, pooled, w1, b1, w2, b2, cf, (int)N, (int)C, (int)mid, (float)gain,    \
                       gain_vec, offset_vec, parts, nparts, (float)scale, save)
#define DDF_CHANNEL_CASE(KK_, BLOCK_)                                                            \
    do {                                                                                         \
        if (ns == 4 && vectors) DDF_CHANNEL_LAUNCH(KK_, BLOCK_, 4, sizeof(T) == 4);              \
        else if (ns == 4) DDF_CHANNEL_LAUNCH(KK_, BLOCK_, 4, false);                             \
        else if (ns == 2 && vectors) DDF_CHANNEL_LAUNCH(KK_, BLOCK_, 2, true);                   \
        else if (ns == 2) DDF_CHANNEL_LAUNCH(KK_, BLOCK_, 2, false);                             \
        else if (vectors) DDF_CHANNEL_LAUNCH(KK_, BLOCK_, 1, true);                              \
        else DDF_CHANNEL_LAUNCH(KK_, BLOCK_, 1, false);                                          \
    } while (0)
    if (k == 3 && block == 64) DDF_CHANNEL_CASE(9, 64);
    else if (k == 3) DDF_CHANNEL_CASE(9, 128);
    else if (k == 5 && block == 64) DDF_CHANNEL_CASE(25, 64);
    else if (k == 5) DDF_CHANNEL_CASE(25, 128);
    else return hipErrorNotSupported;
#undef DDF_CHANNEL_LAUNCH
#undef DDF_CHANNEL_CASE
    return hipGetLastError();
}

#define DDF_INSTANTIATE_BRANCHES(T)                                                              \
    template hipError_t spatial_branch<T>(const T *, const T *, const T *, T *, int64_t, int64_t, \
                                          int64_t, int64_t, int, int, int, double, const T *,    \
                                          const T *, hipStream_t, float *, int64_t, int *, T *); \
    template hipError_t channel_branch<T>(const T *, const T *, const T *, const T *, const T *, \
                                          T *, int64_t, int64_t, int64_t, int, double, const T *, \
                                          const T *, hipStream_t, const float *, int, double, ChannelSave);
DDF_INSTANTIATE_BRANCHES(__half)
DDF_INSTANTIATE_BRANCHES(float)
#undef DDF_INSTANTIATE_BRANCHES

}  // namespace ddf

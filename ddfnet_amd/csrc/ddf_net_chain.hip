// A bottleneck's spatial filter branch and dynamic filter, its last 1x1 convolution and the next one's
// first in one launch (DDF-ResNet inference, fp16, channels-last; ddf_resnet.py:34-111 of the reference composes them).
#include <numeric>
#include <type_traits>

#include "ddf_net_device.h"

namespace ddf {
namespace {
using namespace net;
using rows::kOutside;
using rows::load_words;
using rows::plane_rsrc;

// out (M, N) = relu(norm(x . w) + res), or relu(norm(x . w) + norm'(side . side_w));
// next (M, N2) = relu(norm''(out . w2)), and next's sums over its pixels.
//
// The wide result is written once and not read back: a workgroup takes kChainRows pixels of all channels,
// goes over the wide channels by kChunk, and each chunk is the next block of the summed dimension of
// the second product, whose sums stay in registers.  A wave has 32 pixels: their x in registers as the
// operand of every chunk, a tile of LDS for the chunk's results, which are rounded, meet the residual
// and leave as whole 128-byte lines from there, and are read as the second product's operand.  The
// weights of a chunk are shared: w's rows come in while the second product of the chunk before is
// made, w2's during the first product, straight to LDS, two barriers a chunk.
// Memory bounds it at 56 x 56: 514 MB in 84 us behind the filter's launch (6.1 TB/s, the last-level cache
// has part of the residual; 103 us, a copy's rate, with everything from memory).  us, two launches /
// this, batch 128: 56 x 56 x 64 -> 256 -> 64 122 / 84, with the projection 141 / 95, -> 128 140 / 105, 28 x 28 x
// 128 -> 512 -> 128 68 / 62; batch 16: 24.0 / 16.0, 26.5 / 20.4, 24.2 / 18.4.  Tried there and no faster: the first product of the
// next chunk beside the second one of this, one barrier's work (65 -> 68 us at 28 x 28), waves in
// pairs that split the channels (66), 64 pixels a workgroup (73); at 14 x 14 x 256 -> 1024 -> 256 such pairs take
// 48 us where the two launches take 51, LDS bound (each weight fragment feeds one product of a wave).
constexpr int kChunk = 64, kTilePitch = kChunk + 8;
constexpr int kChainWaves = kThreads / kWave, kChainRows = 32 * kChainWaves;    // a wave: 32 pixels

template <int K, int K2, int N2>
struct ChainLds {    // halves; K2: channels of the side product, 0: none
    static constexpr int w = 0, wd = w + kChunk * K, w2 = wd + kChunk * K2, tile = w2 + N2 * kChunk,
                         norms = tile + kChainRows * kTilePitch;
    // at the end: a wave's tile of next's results, and the sums over its pixels
    static constexpr int red = kChainRows * kTilePitch;
    static_assert(red + kChainWaves * N2 * 2 <= norms, "next's results fit in front of the norms");
    static constexpr int filtered = norms - kChainRows * (K + 8);    // at the start: a wave's filtered pixels
    static_assert(filtered >= wd + kChunk * K2, "and do not meet the first weights");
    // scale, shift, what a sum starts with; of the wide channels (and of the side product), of next's
    static constexpr int floats(int N) { return N * (K2 ? 5 : 3) + N2 * 3; }
    // with a filter: behind them the spatial taps of the tile's pixels
    static constexpr int bytes(int N, bool filter) { return norms * 2 + floats(N) * 4 + (filter ? kChainRows * kTapPitch * 2 : 0); }
};

// ---- spatial branch and dynamic filter in front -----------------------------------------------
// A wave's 32 pixels of x, filtered, normalised and rounded as k_net_filter does it, to its part of LDS
// (rows of K + 8).  K / 8 lanes own four neighbouring pixels at a time, eight channels each, so a channel's
// taps are paired once for all of a lane's pixels and six columns serve four results; rows of images are
// whole runs of four (W % 4 == 0), as tiles are.  Pixels past the last are made from zeros.  The pixels' spatial
// taps are made from their channels, which the filter reads in any case (TapWeights: the same bits as
// k_net_branches), and stay in LDS.
// Neither the filter's results, 103 MB of a batch of 128 at 56 x 56, nor the taps reach memory, and the features are
// read once instead of twice; what is left is a chain of round trips in front of each tile's products, which the
// compute unit's other workgroups cover in part (44 registers more than four of them leave spill: 150 us where
// three take 105).  us, filter and the launch behind it / those in one, batch 128: 56 x 56 x 64 -> 256 -> 64 125 / 106, with
// the projection 128 / 116, -> 128 144 / 125, 28 x 28 x 128 -> 512 -> 128 72 / 63.  Both branches, filter and that
// launch / the channel branch and this, batch 128: 139 / 113, 143 / 127, 157 / 130, 84 / 72; batch 64: 69 / 57, 77 / 64, 76 / 64,
// 50 / 42; batch 8: 30 / 22 (as are all at 56 x 56).
constexpr int kRun = 4;
template <int K, bool MUL>
__device__ __forceinline__ void filter_pixels(const NetChain &a, int64_t m0, int wave, int lane, _Float16 *to, _Float16 *sf) {
    constexpr int KS = K / 32, LP = K / 8, SLOTS = kWave / LP, PER = 32 / SLOTS, RING = 5;
    static_assert(PER % kRun == 0);
    const int cl = lane % LP, H = (int)a.rows.by, W = a.W;
    // (all offsets from a pixel in front of the tile's neighbours: a tile's are 32-bit ones)
    const int64_t base = m0 - W - 1 > 0 ? m0 - W - 1 : 0;
    const __amdgpu_buffer_rsrc_t xr = plane_rsrc(static_cast<const _Float16 *>(a.x) + base * K,
                                                 (uint32_t)(min(a.M - base, (int64_t)(2 * W + 2 + kChainRows)) * K * 2));
    // the spatial taps of the wave's pixels, sixteen at a time
    TapWeights<KS> weights;
    weights.request(static_cast<const _Float16 *>(a.tap_w), static_cast<const _Float16 *>(a.tap_bias), lane);
    half8_t own[2][KS];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            own[i][ks] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(
                xr, (int)(((int)(m0 - base) + wave * 32 + i * 16 + (lane & 15)) * K + (lane >> 4) * 8) * 2, ks * 64, 0));
    const bool bn = a.filter_norm.var;
    auto parameter = [&](bool there, const void *p) __attribute__((always_inline)) {    // (zeros where there is none)
        return __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(plane_rsrc(p, there && p ? K * 2 : 0), cl * 16, 0, 0));
    };
    const half8_t nw = parameter(bn, a.filter_norm.weight), nb = parameter(bn, a.filter_norm.bias), nm = parameter(bn, a.filter_norm.mean),
                  nv = parameter(bn, a.filter_norm.var), nc = parameter(true, a.filter_norm.conv_bias);
    uint32_t cfa[3][8], cfb[3][4];
    float sc[8], sh[8];
#pragma unroll
    for (int run = 0; run < PER / kRun; ++run) {
        const int px = wave * 32 + lane / LP * PER + run * kRun;    // in the tile
        const bool live = m0 + px < a.M;
        const unsigned pix = live ? (unsigned)m0 + px : (unsigned)m0, row = a.row.of(pix);
        const int xx = (int)(pix - row * W), n = (int)a.rows.of(row), y = (int)(row - (unsigned)n * H);
        uint32_t rowo[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int yy = y - 1 + i;
            rowo[i] = live && yy >= 0 && yy < H ? (uint32_t)(((int)((int64_t)pix - base) + (i - 1) * W) * K + cl * 8) * 2 : kOutside;
        }
        uint32_t col[RING][3][4], tap[kRun][6];
        auto column = [&](auto slot) __attribute__((always_inline)) {
            constexpr int Q = decltype(slot)::value;    // column xx - 1 + Q
            const bool in = (Q > 0 || xx > 0) && (Q < kRun + 1 || xx + kRun < W);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                load_words<4>(xr, in && rowo[i] != kOutside ? rowo[i] + (uint32_t)((Q - 1) * K * 2) : kOutside, col[Q % RING][i]);
        };
        auto taps = [&](auto slot) __attribute__((always_inline)) {
            constexpr int Q = decltype(slot)::value;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const uint2 v = *reinterpret_cast<const uint2 *>(sf + (px - wave * 32 + Q) * kTapPitch + i * 4);
                tap[Q][2 * i] = v.x;
                tap[Q][2 * i + 1] = v.y;
            }
        };
        if (run == 0 || a.npix % PER) channel_taps(static_cast<const _Float16 *>(a.cf) + ((int64_t)n * K + cl * 8) * 9, cfa, cfb);
        rows::static_for<0, RING - 1>(column);
        if (run == 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i) weights.taps(own[i], a.tap_gain, true, sf, i * 16 + (lane & 15), lane);
            asm volatile("" ::: "memory");    // (a wave's LDS operations keep their order)
            const float eps = bn ? a.filter_norm.eps : 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sc[e] = (bn ? (float)nw[e] : 1.f) * rsqrtf((bn ? (float)nv[e] : 1.f) + eps);
                sh[e] = (float)nb[e] + ((float)nc[e] - (float)nm[e]) * sc[e];
            }
        }
        rows::static_for<0, 2>(taps);
        rows::static_for<0, kRun>([&](auto q) __attribute__((always_inline)) {
            constexpr int Q = decltype(q)::value;
            if constexpr (Q + RING - 1 < kRun + 2) column(std::integral_constant<int, Q + RING - 1>{});
            if constexpr (Q + 2 < kRun) taps(std::integral_constant<int, Q + 2>{});
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (Q == 0) {
                pair_column(col[0]);
                pair_column(col[1]);
            }
            pair_column(col[(Q + 2) % RING]);
            float acc[8];
            filter_sums<MUL, false>(cfa, cfb, col[Q % RING], col[(Q + 1) % RING], col[(Q + 2) % RING], tap[Q], acc);
            half8_t o;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float f = fmaf((float)(_Float16)acc[e], sc[e], sh[e]);    // (the sum is rounded as the operator's result is)
                asm volatile("" : "+v"(f));
                o[e] = (_Float16)f;
            }
            o = __builtin_elementwise_maximum(o, half8_t{0, 0, 0, 0, 0, 0, 0, 0});
            *reinterpret_cast<half8_t *>(to + (px - wave * 32 + Q) * (K + 8) + cl * 8) = o;
            __builtin_amdgcn_sched_barrier(0);
        });
    }
}

// chunk c of row r of a weight tile sits in place c ^ turn (see k_net_conv: sixteen lanes that LDS serves at
// once meet all of its banks)
template <int CH>
__device__ __forceinline__ int turn(int r) { return CH == 8 ? (r >> 1) & 7 : r & 15; }

// ROWS rows of LEN halves, `pitch` halves apart in memory, to LDS by all threads.
template <int ROWS, int LEN>
struct StageRows {
    static constexpr int CH = LEN / 8, STEP = kThreads / CH, COUNT = ROWS / STEP;
    static_assert(kThreads % CH == 0 && ROWS % STEP == 0 && STEP % 16 == 0);
    int offset;
    __device__ __forceinline__ StageRows(int tid, int pitch) {
        const int r = tid / CH, c = (tid % CH) ^ turn<CH>(r);
        offset = (r * pitch + c * 8) * 2;
    }
    __device__ __forceinline__ void load(uint32_t lds, int wave, const _Float16 *base, int pitch) const {
#pragma unroll
        for (int i = 0; i < COUNT; ++i)
            load_to_lds(lds + wave * (kWave * 16) + i * (kThreads * 16), reinterpret_cast<const char *>(base + (int64_t)i * STEP * pitch), offset);
    }
};

// Scale, shift and what a sum starts with, of all channels of a norm: four channels per thread and pass, asked for
// through descriptors that hold nothing where a parameter is not there (under a branch each, the loads
// waited for one another: 0.7 us of 16 at 16 x 56 x 56, 2 of 50 with 1024 channels).  Without a BatchNorm a bias is part of the sum, elsewhere the
// sum is rounded first (see k_net_conv).
template <int PASSES>
struct Norms {
    uint32_t w[PASSES][2], b[PASSES][2], m[PASSES][2], v[PASSES][2], cb[PASSES][2];
    __device__ __forceinline__ void request(const NetNorm &n, int channels, int tid) {
        const void *const p[5] = {n.var ? n.weight : nullptr, n.var ? n.bias : nullptr, n.var ? n.mean : nullptr, n.var, n.conv_bias};
        uint32_t(*const to[5])[2] = {w, b, m, v, cb};
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const __amdgpu_buffer_rsrc_t r = plane_rsrc(p[k], p[k] ? channels * 2 : 0);
#pragma unroll
            for (int i = 0; i < PASSES; ++i) rows::load_words<2>(r, (uint32_t)(i * kThreads + tid) * 8, to[k][i]);
        }
    }
    __device__ __forceinline__ void put(const NetNorm &n, int channels, int tid, float *scale, float *shift, float *start) const {
        const bool bn = n.var, in_sum = start && !bn;
        const float eps = bn ? n.eps : 0.f;
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
            const int c = (i * kThreads + tid) * 4;
            const half4_t wv = __builtin_bit_cast(half4_t, w[i]), bv = __builtin_bit_cast(half4_t, b[i]), mv = __builtin_bit_cast(half4_t, m[i]),
                          vv = __builtin_bit_cast(half4_t, v[i]), cv = __builtin_bit_cast(half4_t, cb[i]);
            float4_t sc, sh, st;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float conv = (float)cv[e];
                sc[e] = (bn && n.weight ? (float)wv[e] : 1.f) * rsqrtf((bn ? (float)vv[e] : 1.f) + eps);
                sh[e] = (float)bv[e] + ((in_sum ? 0.f : conv) - (float)mv[e]) * sc[e];
                st[e] = in_sum ? conv : 0.f;
            }
            if (c < channels) {
                *reinterpret_cast<float4_t *>(scale + c) = sc;
                *reinterpret_cast<float4_t *>(shift + c) = sh;
                if (start) *reinterpret_cast<float4_t *>(start + c) = st;
            }
        }
    }
};
// (passes of the wide channels: what a launch takes; a network's have 512 at most, past 1024 there are only other callers'.
// The second pass asks behind its descriptors then, which return zeros without a trip to memory)
constexpr int kMaxWide = 2048, kWidePasses = kMaxWide / (4 * kThreads);

enum { kNoFilter, kFilterMul, kFilterAdd };

template <int K, int K2, int N2, int WPS, int FILTER>
__global__ __launch_bounds__(kThreads, WPS) void k_net_chain(NetChain a) {
    typedef ChainLds<K, K2, N2> L;
    constexpr int BM = kChainRows;
    constexpr int TA = kChunk / 32, TB = N2 / 32, SB = N2 / kChunk;    // tiles of 32 channels; chunks of next's channels
    constexpr int RV = 4;                          // vectors of a chunk that a lane takes on their way out
    extern __shared__ __align__(16) _Float16 chain_smem[];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int l32 = lane & 31, hi = lane >> 5;
    at_once(a.x, a.w, a.w2, a.res, a.out, a.M, a.N, a.npix, a.tiles, a.norm.weight, a.norm.bias, a.norm.mean);
    at_once(a.norm.var, a.norm.conv_bias, a.norm2.weight, a.norm2.bias, a.norm2.mean, a.norm2.var, a.norm2.conv_bias, a.next);
    if constexpr (FILTER) at_once(a.cf, a.tap_w, a.tap_bias, a.W, a.row.by, a.row.magic, a.rows.by, a.rows.magic);
    const int block = xcd_block(blockIdx.x, a.tiles);
    if (block >= a.tiles) return;
    const int64_t m0 = (int64_t)block * BM;
    const int rows = (int)min((int64_t)BM, a.M - m0), N = a.N, chunks = N / kChunk;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) _Float16 *)chain_smem;
    float *const norms = reinterpret_cast<float *>(chain_smem + L::norms);
    float *const scale = norms, *const shift = norms + N, *const start = norms + 2 * N;
    float *const side_scale = norms + 3 * N, *const side_shift = norms + 4 * N;
    float *const scale2 = norms + (K2 ? 5 : 3) * N, *const shift2 = scale2 + N2, *const start2 = shift2 + N2;

    // (rows past the last pixel read zeros and are not stored: every one of these loads and stores is
    // issued whatever the tile, the waits below count them.  A row is in the lane's offset throughout: the
    // scalar offset, which moves inside a row, is left out of the descriptor's range check)
    const __amdgpu_buffer_rsrc_t rr = plane_rsrc(K2 ? nullptr : static_cast<const _Float16 *>(a.res) + m0 * N, K2 ? 0 : rows * N * 2);
    const __amdgpu_buffer_rsrc_t orr = plane_rsrc(static_cast<_Float16 *>(a.out) + m0 * N, rows * N * 2);
    const StageRows<kChunk, K> sw(tid, K);
    const StageRows<kChunk, K2 ? K2 : K> sd(tid, K2);
    const StageRows<N2, kChunk> sw2(tid, N);
    const _Float16 *const w = static_cast<const _Float16 *>(a.w), *const wd = static_cast<const _Float16 *>(a.side_w),
                   *const w2 = static_cast<const _Float16 *>(a.w2);
    auto stage_w = [&](int j) __attribute__((always_inline)) {
        sw.load(lds0 + L::w * 2, wave, w + (int64_t)j * kChunk * K, K);
        if constexpr (K2 > 0) sd.load(lds0 + L::wd * 2, wave, wd + (int64_t)j * kChunk * K2, K2);
    };
    stage_w(0);
    {
        Norms<kWidePasses> norm, side_norm;
        Norms<1> norm2;
        norm.request(a.norm, N, tid);
        if constexpr (K2 > 0) side_norm.request(a.side_norm, N, tid);
        norm2.request(a.norm2, N2, tid);
        norm.put(a.norm, N, tid, scale, shift, K2 ? nullptr : start);
        if constexpr (K2 > 0) side_norm.put(a.side_norm, N, tid, side_scale, side_shift, nullptr);
        norm2.put(a.norm2, N2, tid, scale2, shift2, start2);
    }
    half8_t xv[K / 16], dv[K2 ? K2 / 16 : 1];
    if constexpr (FILTER) {
        _Float16 *const mine = chain_smem + L::filtered + wave * 32 * (K + 8);
        _Float16 *const taps = reinterpret_cast<_Float16 *>(norms + L::floats(N)) + wave * 32 * kTapPitch;
        filter_pixels<K, FILTER == kFilterMul>(a, m0, wave, lane, mine, taps);
        asm volatile("" ::: "memory");    // (a wave's LDS operations keep their order)
#pragma unroll
        for (int k = 0; k < K / 16; ++k) xv[k] = *reinterpret_cast<const half8_t *>(mine + l32 * (K + 8) + k * 16 + hi * 8);
    } else {
        const __amdgpu_buffer_rsrc_t xr = plane_rsrc(static_cast<const _Float16 *>(a.x) + m0 * K, rows * K * 2);
#pragma unroll
        for (int k = 0; k < K / 16; ++k)
            xv[k] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(xr, ((wave * 32 + l32) * K + hi * 8) * 2, k * 32, 0));
    }
    if constexpr (K2 > 0) {
        const __amdgpu_buffer_rsrc_t dr = plane_rsrc(static_cast<const _Float16 *>(a.side) + m0 * K2, rows * K2 * 2);
#pragma unroll
        for (int k = 0; k < K2 / 16; ++k)
            dv[k] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(dr, ((wave * 32 + l32) * K2 + hi * 8) * 2, k * 32, 0));
    }
    const bool in_sum = !K2 && !a.norm.var && a.norm.conv_bias, in_sum2 = !a.norm2.var && a.norm2.conv_bias;
    // a lane's vectors on their way out: eight channels of every eighth pixel
    const int c8 = lane & 7, px0 = wave * 32 + (lane >> 3);
    rows_u4 rv[RV];
    // (worked out where it is used: four kept in registers spill where four waves share a SIMD's)
    auto vector_at = [&](int i) __attribute__((always_inline)) {
        int step = 8 * N * 2;
        asm volatile("" : "+s"(step));
        return (px0 * N + c8 * 8) * 2 + i * step;
    };
    auto residual = [&](int j) __attribute__((always_inline)) {
        if constexpr (K2 == 0) {
#pragma unroll
            for (int i = 0; i < RV; ++i)
                rv[i] = __builtin_amdgcn_raw_buffer_load_b128(rr, vector_at(i), j * (kChunk * 2), 0);
        }
    };
    residual(0);

    // a lane's column of a 32 x 32 step's result is pixel l32, rows (channels) 8 * q + 4 * hi + 0..3 in
    // registers 4 * q ..
    auto channel = [&](int t, int q) { return t * 32 + 8 * q + 4 * hi; };
    _Float16 *const tile = chain_smem + L::tile + wave * 32 * kTilePitch;
    float16_t sum2[TB];
    auto clear = [](float16_t &s) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = 0.f;
    };
#pragma unroll
    for (int t = 0; t < TB; ++t) clear(sum2[t]);
    auto product = [&](const _Float16 *weights, auto len, const auto &v, float16_t(&s)[TA]) __attribute__((always_inline)) {
        constexpr int LEN = decltype(len)::value;
#pragma unroll
        for (int k = 0; k < LEN / 16; ++k)
#pragma unroll
            for (int t = 0; t < TA; ++t) {
                const int r = t * 32 + l32;
                const half8_t wv = *reinterpret_cast<const half8_t *>(weights + r * LEN + ((k * 2 + hi) ^ turn<LEN / 8>(r)) * 8);
                s[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wv, v[k], s[t], 0, 0, 0);
            }
    };
    float one = 1.f;
    asm volatile("" : "+v"(one));    // (value * one + f: a conversion less than value + f)

    for (int j = 0; j < chunks; ++j) {
        // w's rows are there (the residual may be on its way); everybody is done with w2's
        arrive<K2 ? 0 : RV>();
        sw2.load(lds0 + L::w2 * 2, wave, w2 + j * kChunk, N);
        float16_t sum[TA];
        // sums rounded to fp16, to the wave's tile
        auto put = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < TA; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    half4_t v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = (_Float16)sum[t][4 * q + e];
                    *reinterpret_cast<half4_t *>(tile + l32 * kTilePitch + channel(t, q)) = v;
                }
            asm volatile("" ::: "memory");    // (a wave's LDS operations keep their order)
        };
        // scale and shift of a lane's eight channels of the chunk, and its vectors
        auto get = [&](const float *scales, const float *shifts, float (&sc)[8], float (&sh)[8], half8_t (&v)[RV]) __attribute__((always_inline)) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float4_t s = *reinterpret_cast<const float4_t *>(scales + j * kChunk + c8 * 8 + h * 4);
                const float4_t o = *reinterpret_cast<const float4_t *>(shifts + j * kChunk + c8 * 8 + h * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sc[4 * h + e] = s[e];
                    sh[4 * h + e] = o[e];
                }
            }
#pragma unroll
            for (int i = 0; i < RV; ++i)
                v[i] = *reinterpret_cast<const half8_t *>(tile + (px0 - wave * 32 + i * 8) * kTilePitch + c8 * 8);
        };
        float sc[8], sh[8];
        half8_t v[RV];
        // A projection's results take the residual's place.  Worked out where the product leaves them, four channels of a pixel at a
        // time, the scales and shifts of both products were 128 KB a chunk of the 290 that LDS was read for; here they are 32.
        // us, 56 x 56 x 64 + 64 -> 256 -> 64 of 128, 64, 32 and 16 images with all that is in front: 117.4 / 115.0, 61.9 / 60.6, 39.2 / 38.4, 24.0 /
        // 23.4.  (In k_net_conv's pairs, whose tiles are shared and take two barriers more: 128 x 128 in short stages 79.3 / 76.9, in long ones
        // no difference, tiles of 64 14.2 / 15.2.)
        if constexpr (K2 > 0) {
#pragma unroll
            for (int t = 0; t < TA; ++t) clear(sum[t]);
            product(chain_smem + L::wd, std::integral_constant<int, K2 ? K2 : 16>{}, dv, sum);
            put();
            get(side_scale, side_shift, sc, sh, v);
#pragma unroll
            for (int i = 0; i < RV; ++i) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[i][e] = (_Float16)fmaf((float)v[i][e], sc[e], sh[e]);    // (rounded once, as in k_net_conv's pairs)
                rv[i] = __builtin_bit_cast(rows_u4, v[i]);
            }
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int t = 0; t < TA; ++t) clear(sum[t]);
        if (in_sum) {
#pragma unroll
            for (int t = 0; t < TA; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4_t b = *reinterpret_cast<const float4_t *>(start + j * kChunk + channel(t, q));
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[t][4 * q + e] = b[e];
                }
        }
        product(chain_smem + L::w, std::integral_constant<int, K>{}, xv, sum);
        put();
        get(scale, shift, sc, sh, v);
#pragma unroll
        for (int i = 0; i < RV; ++i) {
            const half8_t r = __builtin_bit_cast(half8_t, rv[i]);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float f = fmaf((float)v[i][e], sc[e], sh[e]);
                f = fmaf((float)r[e], one, f);
                asm volatile("" : "+v"(f));    // (rounded to fp32 first in every instance)
                v[i][e] = (_Float16)f;
            }
            v[i] = __builtin_elementwise_maximum(v[i], half8_t{0, 0, 0, 0, 0, 0, 0, 0});
            *reinterpret_cast<half8_t *>(tile + (px0 - wave * 32 + i * 8) * kTilePitch + c8 * 8) = v[i];
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(rows_u4, v[i]), orr, vector_at(i), j * (kChunk * 2), 0);
        }
        // w2's rows are there; everybody is done with w's
        arrive<RV>();
        if (j + 1 < chunks) {
            stage_w(j + 1);
            residual(j + 1);
        }
#pragma unroll
        for (int k = 0; k < kChunk / 16; ++k) {
            const half8_t pv = *reinterpret_cast<const half8_t *>(tile + l32 * kTilePitch + (k * 2 + hi) * 8);
#pragma unroll
            for (int t = 0; t < TB; ++t) {
                const int r = t * 32 + l32;
                const half8_t wv = *reinterpret_cast<const half8_t *>(chain_smem + L::w2 + r * kChunk + ((k * 2 + hi) ^ turn<kChunk / 8>(r)) * 8);
                sum2[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wv, pv, sum2[t], 0, 0, 0);
            }
        }
    }

    // next's results, kChunk channels of the wave's pixels at a time, through a tile of its own
    __syncthreads();
    _Float16 *const last = chain_smem + wave * 32 * kTilePitch;
    const __amdgpu_buffer_rsrc_t nr = plane_rsrc(static_cast<_Float16 *>(a.next) + m0 * N2, rows * N2 * 2);
    half8_t v[SB][4];
#pragma unroll
    for (int s = 0; s < SB; ++s) {
        const int c0 = s * kChunk;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float4_t b = {0.f, 0.f, 0.f, 0.f};
                if (in_sum2) b = *reinterpret_cast<const float4_t *>(start2 + c0 + t * 32 + 8 * q + 4 * hi);
                half4_t h;
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = (_Float16)(sum2[s * 2 + t][4 * q + e] + b[e]);
                *reinterpret_cast<half4_t *>(last + l32 * kTilePitch + t * 32 + 8 * q + 4 * hi) = h;
            }
        asm volatile("" ::: "memory");
        float sc[8], sh[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            sc[e] = scale2[c0 + c8 * 8 + e];
            sh[e] = shift2[c0 + c8 * 8 + e];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int px = i * 8 + (lane >> 3);
            v[s][i] = *reinterpret_cast<const half8_t *>(last + px * kTilePitch + c8 * 8);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float f = fmaf((float)v[s][i][e], sc[e], sh[e]);
                asm volatile("" : "+v"(f));
                v[s][i][e] = (_Float16)f;
            }
            v[s][i] = __builtin_elementwise_maximum(v[s][i], half8_t{0, 0, 0, 0, 0, 0, 0, 0});
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(rows_u4, v[s][i]), nr, ((wave * 32 + px) * N2 + c0 + c8 * 8) * 2, 0, 0);
        }
        asm volatile("" ::: "memory");
    }
    // Sums over the tile's pixels of each sample it touches, to the sample's slot for this tile; the
    // tile with a sample's last pixel clears the slots that sample does not use (as k_net_conv's).
    float *const red = reinterpret_cast<float *>(chain_smem + L::red);    // [wave][N2]
    const int first = (int)m0, end = (int)min(m0 + BM, a.M), n_last = (end - 1) / a.npix;
    for (int n = first / a.npix; n <= n_last; ++n) {
        const int lo = n * a.npix - first, up = lo + a.npix;
#pragma unroll
        for (int s = 0; s < SB; ++s) {
            float sum[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) sum[e] = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = wave * 32 + i * 8 + (lane >> 3);
                const bool in = r >= lo && r < up && r < rows;
#pragma unroll
                for (int e = 0; e < 8; ++e) sum[e] += in ? (float)v[s][i][e] : 0.f;
            }
            float half[4], pair[2];
#pragma unroll
            for (int e = 0; e < 8; ++e) sum[e] = add_permuted<0x128 /* row_ror:8 */>(sum[e]);
#pragma unroll
            for (int e = 0; e < 4; ++e) half[e] = add_swapped32(sum[e], sum[e + 4]);
#pragma unroll
            for (int e = 0; e < 2; ++e) pair[e] = add_swapped16(half[e], half[e + 2]);
            if (!(lane & 8)) {
                typedef float float2_t __attribute__((ext_vector_type(2)));
                *reinterpret_cast<float2_t *>(red + wave * N2 + s * kChunk + c8 * 8 + (lane >> 4) * 2) = float2_t{pair[0], pair[1]};
            }
        }
        __syncthreads();
        for (int c = tid; c < N2; c += kThreads) {
            float *to = a.pool + (int64_t)n * a.pool_slots * N2 + c;
            int slot = block - (int)((int64_t)n * a.npix / BM);
            float total = red[c];
#pragma unroll
            for (int k = 1; k < kChainWaves; ++k) total += red[k * N2 + c];
            to[(int64_t)slot * N2] = total;
            if (up <= end - first)
                while (++slot < a.pool_slots) to[(int64_t)slot * N2] = 0.f;
        }
        if (n < n_last) __syncthreads();
    }
}

template <int K, int K2, int N2, int WPS, int FILTER>
hipError_t launch_chain(const NetChain &a, hipStream_t st) {
    const int lds = ChainLds<K, K2, N2>::bytes(a.N, FILTER);
    hipLaunchKernelGGL((k_net_chain<K, K2, N2, WPS, FILTER>), dim3(xcd_grid(a.tiles)), dim3(kThreads), lds, st, a);
    return hipGetLastError();
}

}  // namespace

// Whether the two convolutions are one launch: with the spatial branch and the filter in front of it, as
// networks have it, that pays from few tiles on.  us for a whole network, as separate launches / as one: 64 channels, 98
// tiles (4 x 224 x 224) 375 / 371, 147 411 / 404, 49 337 / 342; 128 channels, 98 tiles (16 x 224 x 224) 505 / 523, 128 516 / 525,
// 147 586 / 582.  Where 256 channels follow, two workgroups run side by side on a compute unit and a second
// round of them may be half full, which the launches that are saved make up for: 128 x 28 x 28 x 128 -> 512 -> 256 with
// what is in front of it 103 / 84 us, the network 1653 / 1622.
bool net_chain_covers(int64_t M, int64_t K, int64_t side, int64_t N, int64_t N2) {
    if (N % kChunk || N < kChunk || N > kMaxWide || M > INT32_MAX - 256) return false;
    const int64_t tiles = cdiv(M, kChainRows);
    if (tiles < (K == 64 ? 96 : 144)) return false;
    if (side) return K == 64 && side == 64 && N2 == 64;
    return (K == 64 && (N2 == 64 || N2 == 128)) || (K == 128 && (N2 == 128 || N2 == 256));
}

// (runs of four pixels; rows of 4096 pixels keep a tile's neighbours within 2.2 MB, far from where 32-bit offsets end.
// No size was found where the two launches are faster.  The instances without a filter serve ddf_hip_net_conv_chain; a
// network, whose rows are whole runs, takes one only for images wider than 16384.)
bool net_chain_filters(int64_t W, int64_t K) { return W % kRun == 0 && W <= 4096 && (K == 64 || K == 128); }

int net_chain_pool_slots(int64_t M, int npix) {
    const int start = M > npix ? kChainRows - std::gcd(kChainRows, npix) : 0;
    return (start + npix - 1) / kChainRows + 1;
}

// (the waves per SIMD are what registers and LDS leave room for)
hipError_t net_chain(NetChain a, hipStream_t st) {
    if (a.M == 0) return hipSuccess;
    if (!net_chain_covers(a.M, a.K, a.side_K, a.N, a.N2)) return hipErrorNotSupported;
    if (a.cf && !net_chain_filters(a.W, a.K)) return hipErrorNotSupported;
    a.tiles = (int)cdiv(a.M, kChainRows);
    a.pool_slots = net_chain_pool_slots(a.M, a.npix);
    if (a.cf) {
        a.row = Divisor::make(a.W, a.M);
        a.rows = Divisor::make(a.npix / a.W, a.M / a.W);
    }
#define DDF_CHAIN(K_, SIDE_, N2_, WPS_, FWPS_) \
    if (a.K == K_ && a.side_K == SIDE_ && a.N2 == N2_) {                                            \
        if (!a.cf) return launch_chain<K_, SIDE_, N2_, WPS_, kNoFilter>(a, st);                     \
        return a.mul ? launch_chain<K_, SIDE_, N2_, FWPS_, kFilterMul>(a, st) : launch_chain<K_, SIDE_, N2_, FWPS_, kFilterAdd>(a, st); \
    }
    DDF_CHAIN(64, 64, 64, 3, 3)
    DDF_CHAIN(64, 0, 64, 4, 3)
    DDF_CHAIN(64, 0, 128, 3, 3)
    DDF_CHAIN(128, 0, 128, 2, 2)
    DDF_CHAIN(128, 0, 256, 2, 2)
#undef DDF_CHAIN
    return hipErrorNotSupported;
}

}  // namespace ddf

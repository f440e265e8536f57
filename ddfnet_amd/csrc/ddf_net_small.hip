// 1x1 convolutions of a network in small tiles (DDF-ResNet inference, fp16, channels-last; ddf_resnet.py:34-111 of the
// reference composes them).
#include <type_traits>

#include "ddf_net_device.h"

namespace ddf {
namespace {
using namespace net;
constexpr int kSmallDepth = 4;    // blocks on their way

// What k_net_conv computes, in tiles of T pixels x T channels: the four waves of a workgroup take a quarter of the summed dimension
// each (of a pair's two products, one behind the other) and bring it in themselves, 64 values of the T rows of x and of w at a time, straight
// to a ring of LDS of their own: D blocks on their way, nobody waits for another wave until the sums meet.  What such a launch takes
// is what one compute unit's operands take on their way in, and a unit takes rows' segments of 128 bytes at 133 bytes/ns where
// the 64 that a stage of k_net_conv has there come at 88: this beats tiles of 64 as long as the smaller tiles do not bring
// in too much (conv_tile has the figures).  Written straight to LDS it also beats a tile of 16 x 16 whose operands come to registers, a
// lane's 32 bytes at a time (us, registers / this: 49 x 2048 -> 512 6.1 / 4.3, 196 x 1024 -> 256 4.4 / 3.6, 1 x 2048 -> 1000 4.5 / 3.7).
template <int T, bool PAIR, bool POOL, bool RES>
__global__ __launch_bounds__(kThreads, 1) void k_net_conv_small(NetConv a, NetConv first, TileCut cut) {
    constexpr int D = kSmallDepth, WAVES = kThreads / kWave, V = T * T / kThreads, PER = T / V;    // a thread's results: V channels of a pixel
    constexpr int NL = 2 * T * 8 / kWave;              // loads of a block: eight rows each
    constexpr int BLOCK = 2 * T * 64, PITCH = T + 4;   // halves; floats
    constexpr int P = PAIR ? 2 : 1;
    static_assert((T == 16 || T == 32) && !(RES && PAIR));
    typedef _Float16 lane_t __attribute__((ext_vector_type(V)));
    typedef float sums_t __attribute__((ext_vector_type(V)));
    extern __shared__ __align__(16) _Float16 small_smem[];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    at_once(a.x, a.w, a.M, a.N, a.K, a.stride, cut.tiles_n.by, cut.tiles_n.magic);
    at_once(a.norm.weight, a.norm.bias, a.norm.mean, a.norm.var, a.norm.conv_bias, a.out, a.res, a.relu);
    if constexpr (PAIR) at_once(first.x, first.w, first.K, first.stride, first.H, first.W, first.norm.var, first.norm.weight);
    // (an XCD has some pixels' tiles or some channels': the smaller operand comes to every L2, the larger one to one)
    const int block = a.M > a.N ? xcd_block(blockIdx.x, cut.tiles) : (int)blockIdx.x;
    if (block >= cut.tiles) return;
    const int tm = (int)cut.tiles_n.of(block), tn = block - tm * (int)cut.tiles_n.by;
    const int64_t m0 = (int64_t)tm * T;
    const int n0 = tn * T;
    const int rows = (int)min((int64_t)T, a.M - m0);

    // Row r of a block (the pixels', then the channels') is eight chunks of 16 bytes, chunk q in place q ^ turn(r): the sixteen lanes
    // that LDS serves at once meet all of its banks (see k_net_conv).
    auto turn = [](int r) { return T == 32 ? (r >> 1) & 7 : r & 7; };
    const char *xp[P][NL / 2], *wb[P];
    int wo[P][NL / 2];
    auto aim = [&](const NetConv &c, int which) __attribute__((always_inline)) {
        int64_t sample = 0;
        int at = 0;
        if (c.stride > 1) {
            sample = m0 >> 32 == 0 ? (uint32_t)m0 / (uint32_t)c.npix : m0 / c.npix;
            at = (int)(m0 - sample * c.npix);
        }
        wb[which] = static_cast<const char *>(c.w) + (int64_t)n0 * c.K * 2;
#pragma unroll
        for (int i = 0; i < NL / 2; ++i) {
            const int r = i * 8 + lane / 8, q = ((lane & 7) ^ turn(r)) * 16;
            int64_t row = m0 + min(r, rows - 1);
            if (c.stride > 1) {
                const uint32_t pix = (uint32_t)(at + min(r, rows - 1)), n = cut.npix.of(pix), p = pix - n * c.npix, y = cut.Wo.of(p), xx = p - y * c.Wo;
                row = ((sample + n) * c.H + y * c.stride) * c.W + xx * c.stride;
            }
            xp[which][i] = static_cast<const char *>(c.x) + row * c.K * 2 + q;
            wo[which][i] = min(r, a.N - 1 - n0) * (c.K * 2) + q;
        }
    };
    const int nb0 = PAIR ? first.K / 64 : 0, blocks = nb0 + a.K / 64, per = (blocks + WAVES - 1) / WAVES;
    const int b0 = wave * per, count = max(min(per, blocks - b0), 0);
    const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) _Float16 *)small_smem + (uint32_t)(wave * D * BLOCK * 2);
    auto request = [&](int b) __attribute__((always_inline)) {
        const int k = b0 + b, which = PAIR && k >= nb0 ? 1 : 0, at = (k - (which ? nb0 : 0)) * 128;
        const uint32_t to = ring + (uint32_t)((b % D) * (BLOCK * 2));
#pragma unroll
        for (int i = 0; i < NL / 2; ++i) load_to_lds(to + i * 1024, (PAIR && which ? xp[P - 1][i] : xp[0][i]) + at);
#pragma unroll
        for (int i = 0; i < NL / 2; ++i) load_to_lds(to + (NL / 2 + i) * 1024, (PAIR && which ? wb[P - 1] : wb[0]) + at, PAIR && which ? wo[P - 1][i] : wo[0][i]);
    };
    if constexpr (PAIR) aim(first, 0);
    aim(a, P - 1);
#pragma unroll
    for (int b = 0; b < D; ++b)
        if (b < count) request(b);
    // what the results meet on their way out
    const int p = tid / PER, c = n0 + (tid % PER) * V;
    const bool ok = c < a.N && p < rows;
    Affine<V> aff, side_aff;
    aff.request(a.norm, c < a.N ? c : 0);
    if constexpr (PAIR) side_aff.request(first.norm, c < a.N ? c : 0);
    lane_t rv;
    if constexpr (RES) {
        const _Float16 *from = static_cast<const _Float16 *>(a.res) + (ok ? (m0 + p) * a.N + c : 0);
        __builtin_memcpy(&rv, from, sizeof(rv));
    }
    typedef typename std::conditional<T == 32, float16_t, float4_t>::type acc_t;
    constexpr int ACC = T == 32 ? 16 : 4;
    acc_t acc[P];
#pragma unroll
    for (int w = 0; w < P; ++w)
#pragma unroll
        for (int e = 0; e < ACC; ++e) acc[w][e] = 0.f;
    // (lane's row of the operands, its chunk of a step's)
    const int row = T == 32 ? lane & 31 : lane & 15, piece = T == 32 ? lane >> 5 : lane >> 4;
    constexpr int STEPS = T == 32 ? 4 : 2, CH = 8 / STEPS;
    auto multiply = [&](int b, acc_t &sum) __attribute__((always_inline)) {
        const _Float16 *s = small_smem + wave * D * BLOCK + (b % D) * BLOCK + row * 64;
        half8_t xv[STEPS], wv[STEPS];
#pragma unroll
        for (int k = 0; k < STEPS; ++k) {
            const int at = ((k * CH + piece) ^ turn(row)) * 8;
            xv[k] = *reinterpret_cast<const half8_t *>(s + at);
            wv[k] = *reinterpret_cast<const half8_t *>(s + T * 64 + at);
        }
#pragma unroll
        for (int k = 0; k < STEPS; ++k) {
            if constexpr (T == 32) sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(wv[k], xv[k], sum, 0, 0, 0);
            else sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[k], xv[k], sum, 0, 0, 0);
        }
    };
    for (int b = 0; b < count; ++b) {
        const int behind = min(D - 1, count - 1 - b);    // blocks that may be on their way still
        if (D > 3 && behind >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * NL) : "memory");
        else if (D > 2 && behind == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NL) : "memory");
        else if (behind == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (PAIR && b0 + b >= nb0) multiply(b, acc[P - 1]);
        else multiply(b, acc[0]);
        // (its operands have been read: the products wait for them)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (b + D < count) request(b + D);
    }
    __syncthreads();
    // the waves' sums, [product][wave][pixel][channel]
    float *const red = reinterpret_cast<float *>(small_smem);
#pragma unroll
    for (int w = 0; w < P; ++w) {
        float *to = red + (w * WAVES + wave) * (T * PITCH) + row * PITCH;
#pragma unroll
        for (int g = 0; g < ACC / 4; ++g)
            *reinterpret_cast<float4_t *>(to + 8 * g + 4 * piece) = float4_t{acc[w][4 * g], acc[w][4 * g + 1], acc[w][4 * g + 2], acc[w][4 * g + 3]};
    }
    float sc[V], sh[V], side_sc[V], side_sh[V];
    aff.finish(a.norm, sc, sh);
    if constexpr (PAIR) side_aff.finish(first.norm, side_sc, side_sh);
    __syncthreads();
    auto total = [&](int w) __attribute__((always_inline)) {
        sums_t q[WAVES];
#pragma unroll
        for (int k = 0; k < WAVES; ++k) q[k] = *reinterpret_cast<const sums_t *>(red + (w * WAVES + k) * (T * PITCH) + p * PITCH + (tid % PER) * V);
        return (q[0] + q[1]) + (q[2] + q[3]);
    };
    const sums_t sum = total(P - 1);
    sums_t side;
    if constexpr (PAIR) side = total(0);
    lane_t v;
    // (under a BatchNorm the sum is rounded first, as a convolution's result is; without one a bias is part of it, of a pair's sums too,
    // which k_net_conv rounds first)
    auto under = [](const NetNorm &n, float x) { return n.var ? (float)(_Float16)x : x; };
#pragma unroll
    for (int e = 0; e < V; ++e) {
        float f = fmaf(under(a.norm, sum[e]), sc[e], sh[e]);
        if constexpr (RES) f += (float)rv[e];
        if constexpr (PAIR) f += (float)(_Float16)fmaf(under(first.norm, side[e]), side_sc[e], side_sh[e]);
        asm volatile("" : "+v"(f));    // (rounded to fp32 first in every instance)
        v[e] = (_Float16)(a.relu ? relu(f) : f);
    }
    if (ok) *reinterpret_cast<lane_t *>(static_cast<_Float16 *>(a.out) + (m0 + p) * a.N + c) = v;
    if constexpr (POOL) {
        // Sums over the tile's pixels of each sample it touches (see k_net_conv), a channel's by one thread
        __syncthreads();
#pragma unroll
        for (int e = 0; e < V; ++e) red[p * PITCH + (tid % PER) * V + e] = ok ? (float)v[e] : 0.f;
        __syncthreads();
        if (tid >= T || n0 + tid >= a.N) return;
        const int begin = (int)m0, end = begin + rows, n_last = (int)cut.npix.of(end - 1);
        float x[T];
#pragma unroll
        for (int r = 0; r < T; ++r) x[r] = red[r * PITCH + tid];
        for (int n = (int)cut.npix.of(begin); n <= n_last; ++n) {
            const int lo = n * a.npix - begin, hi = lo + a.npix;
            float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < T; ++r) s[r & 3] += r >= lo && r < hi ? x[r] : 0.f;
            float *to = a.pool + (int64_t)n * a.pool_slots * a.N + n0 + tid;
            int slot = tm - (int)((int64_t)n * a.npix / T);
            to[(int64_t)slot * a.N] = (s[0] + s[1]) + (s[2] + s[3]);
            if (hi <= end - begin)
                while (++slot < a.pool_slots) to[(int64_t)slot * a.N] = 0.f;
        }
    }
}

template <int T>
hipError_t launch_small(const NetConv &a, const NetConv *first, hipStream_t st) {
    const int64_t tiles_n = cdiv(a.N, T), tiles = cdiv(a.M, T) * tiles_n;
    if (tiles > (1 << 30)) return hipErrorInvalidConfiguration;
    const NetConv &x = first ? *first : a;
    const TileCut cut{(int)tiles, Divisor::make(tiles_n, tiles), Divisor::make(x.npix, a.pool ? a.M : x.npix + (int64_t)T), Divisor::make(x.Wo, x.npix)};
    constexpr int kRing = kThreads / kWave * kSmallDepth * 2 * T * 64 * 2, kSums = 2 * (kThreads / kWave) * T * (T + 4) * 4;
    constexpr int lds = kRing > kSums ? kRing : kSums;
    const dim3 grid(a.M > a.N ? xcd_grid(tiles) : (unsigned)tiles);
    if (first) hipLaunchKernelGGL((k_net_conv_small<T, true, false, false>), grid, dim3(kThreads), lds, st, a, *first, cut);
    else if (a.pool) hipLaunchKernelGGL((k_net_conv_small<T, false, true, false>), grid, dim3(kThreads), lds, st, a, a, cut);
    else if (a.res) hipLaunchKernelGGL((k_net_conv_small<T, false, false, true>), grid, dim3(kThreads), lds, st, a, a, cut);
    else hipLaunchKernelGGL((k_net_conv_small<T, false, false, false>), grid, dim3(kThreads), lds, st, a, a, cut);
    return hipGetLastError();
}

}  // namespace

hipError_t net_conv_small(int rows, const NetConv &a, const NetConv *first, hipStream_t st) {
    return rows == 16 ? launch_small<16>(a, first, st) : launch_small<32>(a, first, st);
}

}  // namespace ddf

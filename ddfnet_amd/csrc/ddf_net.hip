// DDF-ResNet inference in fp16 with channels-last activations (gfx950).
//
// Between the image and the logits a network is its own world: its activations have no
// layout anybody else sees.  Here they are (N, H, W, C): a 1x1 convolution is then a
// product of two row-major matrices whose summed dimension is contiguous in both, which is
// what the matrix cores read; a lane of the dynamic filter owns eight channels of a pixel
// and its neighbours are whole vectors, whatever the row length; and BatchNorm, ReLU and
// the residual addition ride on the kernel that produces the values.  A bottleneck is
// four launches, each activation is written once:
//   k_net_conv      1x1 convolution (+ BatchNorm, residual, ReLU), sums over its pixels on the way
//   k_net_branches  spatial and channel filter branch
//   k_net_filter    dynamic filter + BatchNorm + ReLU
//   k_net_conv
// (with many pixels all but the channel branch are one with the next one's first, k_net_chain of
// ddf_net_chain.hip)
// and k_net_stem is the 7x7 convolution, BatchNorm, ReLU and max-pool in one.
// At batch 128 the network took 8.85 ms as torch modules around the operator: 3.2 ms of
// BatchNorm, 1.6 ms of ReLU and additions, 3 ms of convolutions (ddf_resnet.py:34-111 of
// the reference is the same composition).  Sums are fp32; what is stored is rounded to
// fp16 where the modules round it, and less often (not between convolution and BatchNorm's
// ReLU).
#include <algorithm>
#include <numeric>
#include <type_traits>

#include "ddf_channel.h"
#include "ddf_common.h"
#include "ddf_net_device.h"
#include "ddf_rows.h"

namespace ddf {
namespace {
using namespace net;
using rows::from_left;
using rows::kOutside;
using rows::load_words;
using rows::plane_rsrc;

// ---- 1x1 convolution ----------------------------------------------------------
// out[m, o] = act(affine(sum_k x[row(m), k] w[o, k]) (+ res[m, o])), row(m) the sampled
// pixel under a stride.  Tiles of BM pixels x BN channels; 2 x WN waves over the tile,
// each in 32x32x16 steps.  W is the A operand, so a lane ends with runs of four channels of
// one pixel; the tile goes through LDS once more and leaves as whole 16-byte vectors.
// K comes in stages of KST that go from memory straight into a ring of ST LDS buffers, ST - 1
// of them in flight: no registers hold what is on its way, so WG = 2 to 3 workgroups share a
// compute unit (staged through registers, the 128 x 128 tile took 230 of them).  One barrier
// per stage: a wave waits for its own loads of stage k and for its reads of stage k - 1, then
// the buffer of stage k - 1 is free for k + ST - 1.
// A stage is rows of KST / 8 16-byte chunks without padding (the loads write LDS in lane
// order), chunk c of row r in place c ^ turn(r): the sixteen lanes that a 16-byte LDS read
// serves at once are rows {0-3, 12-15, 20-27} or {4-11, 16-19, 28-31} of 32, and with these
// turns they meet all sixteen places of the 256 bytes the banks span (r & 7, the turn before,
// had every second read conflict: 1.76 M conflict cycles at 25088 x 1024 x 256, now 0.15 M).
// Rate at batch 128, us staged through registers / through the ring: 56 x 56 x 64 -> 256 82 / 65, 28 x 28 x
// 512 -> 1024 under stride 2 54 / 47, 14 x 14 x 1024 -> 256 28 / 24 (545 TFLOP/s); deeper rings,
// larger tiles and a K order turned per tile change nothing there; the matrix cores are busy a
// third of the time, and 98 tiles for an XCD's 96 places cost 125 -> 128 images 10 %.  The wide
// results of the 56 x 56 layers run at copy rate.
// On the way out the vector ALU counts as much as memory (half of its time at 56 x 56): all of a
// thread's vectors come from LDS at once, and eight results take 24 instructions instead of 57 -
// fp16 operands inside the multiply-adds, ReLU two at a time after the rounding.  Batch 128, us:
// 56 x 56 x 64 -> 256 with a residual 91.9 -> 85.0, 28 x 28 x 128 -> 512 54.4 -> 48.3, 14 x 14 x
// 256 -> 1024 38.4 -> 34.2; pairs 95 -> 81 (28 x 28 x 128 + 256 -> 512), 80 -> 67 (7 x 7).
//
// What a launch of few tiles takes besides its products is its way to the first load and from the last product to the stores:
// arguments at once, tiles and pixels by multiplications, the first stages in front of the norm's parameters, scale and
// shift by a thread per channel.  First loads out / end, us inside the launch: 14 x 14 x 256 -> 1024 with a residual 1.00 / 2.90
// -> 0.44 / 2.32, 56 x 56 x 256 -> 64 1.06 / 3.44 -> 0.48 / 2.73; networks of 1, 8, 32 and 128 images of 224 x 224 310.4 -> 299.3, 415
// -> 402, 670 -> 662, 1634 -> 1614 us, 48 of 256 x 256 889 -> 876.
//
// With PAIR the tile is act(affine(x w) + affine'(x' w')) of two products, a bottleneck's last
// convolution and its projection: x' w' goes first, its affine result stays in registers as
// the fp16 values that a projection of its own would have stored.
template <int BM, int BN, int KST, int ST, int WAVES>
constexpr int conv_lds_halves() {
    // (behind the tile: the waves' sums over its pixels)
    const int ring = (BM + BN) * KST * ST, tile = BM * (BN + 8) + WAVES * BN * 2;
    return ring > tile ? ring : tile;
}

// ALONE: a stage's loads in front of its products instead of between them (see launch_conv).
template <int BM, int BN, int KST, int ST, int WN, int WG, bool PAIR, bool POOL, bool RES, bool ALONE = false>
__global__ __launch_bounds__(2 * WN * kWave, WG * WN / 2) void k_net_conv(NetConv a, NetConv first, TileCut cut) {
    constexpr int WAVES = 2 * WN, T = WAVES * kWave, CH = KST / 8, STAGE = (BM + BN) * KST;
    constexpr int RX = BM * CH / T, RW = BN * CH / T;
    constexpr int TM = BM / 64, TN = BN / 32 / WN;      // 32-wide tiles per wave: pixels, channels
    constexpr int PITCH = BN + 8;
    static_assert((ST == 2 || ST == 3) && (CH == 4 || CH == 8) && RX > 0 && RW > 0 && !(RES && PAIR));
    extern __shared__ __align__(16) _Float16 net_smem[];
    __shared__ __align__(16) float affine[PAIR ? 4 : 2][BN];    // scale, shift; of the first product, too
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    at_once(a.x, a.w, a.M, a.N, a.K, cut.tiles, cut.tiles_n.by, cut.tiles_n.magic);
    at_once(a.norm.weight, a.norm.bias, a.norm.mean, a.norm.var, a.norm.conv_bias, a.out, a.res, a.relu);
    if constexpr (PAIR) at_once(first.x, first.w, first.K, first.stride, first.H, first.W, first.norm.var, first.norm.weight);
    const int block = xcd_block(blockIdx.x, cut.tiles);
    if (block >= cut.tiles) return;
    const int tm = (int)cut.tiles_n.of(block), tn = block - tm * (int)cut.tiles_n.by;
    const int64_t m0 = (int64_t)tm * BM;
    const int n0 = tn * BN;
    const int rows = (int)min((int64_t)BM, a.M - m0);    // pixels of the tile
    auto turn = [](int r) { return CH == 8 ? (r >> 1) & 7 : (r >> 2) & 3; };

    const _Float16 *xp[RX], *wp[RW];
    auto aim = [&](const NetConv &c) __attribute__((always_inline)) {
        const _Float16 *x = static_cast<const _Float16 *>(c.x), *w = static_cast<const _Float16 *>(c.w) + (int64_t)n0 * c.K;
        if (c.stride > 1) {
            const int64_t sample = m0 >> 32 == 0 ? (uint32_t)m0 / (uint32_t)c.npix : m0 / c.npix;
            const int at = (int)(m0 - sample * c.npix);
#pragma unroll
            for (int i = 0; i < RX; ++i) {
                const int q = tid + i * T, r = q / CH, ch = (q % CH) ^ turn(r);
                const unsigned pix = (unsigned)(at + min(r, rows - 1)), n = cut.npix.of(pix), p = pix - n * c.npix;
                const unsigned y = cut.Wo.of(p), xx = p - y * c.Wo;
                xp[i] = x + (((sample + n) * c.H + y * c.stride) * c.W + xx * c.stride) * c.K + ch * 8;
            }
        } else {
            x += m0 * c.K;
#pragma unroll
            for (int i = 0; i < RX; ++i) {
                const int q = tid + i * T, r = q / CH, ch = (q % CH) ^ turn(r);
                xp[i] = x + ((int64_t)min(r, rows - 1) * c.K + ch * 8);
            }
        }
#pragma unroll
        for (int i = 0; i < RW; ++i) {
            const int q = tid + i * T, r = q / CH, ch = (q % CH) ^ turn(r);
            wp[i] = w + ((int64_t)min(r, a.N - 1 - n0) * c.K + ch * 8);
        }
    };
    const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) _Float16 *)net_smem;
    // (load i of a stage; first those of x)
    auto load_one = [&](int i, int buf) __attribute__((always_inline)) {
        const uint32_t at = ring + (uint32_t)(buf * STAGE) * 2 + (uint32_t)wave * (kWave * 16);
        const _Float16 *&p = i < RX ? xp[i < RX ? i : 0] : wp[i < RX ? 0 : i - RX];
        load_to_lds(at + (i < RX ? i * T * 16 : BM * KST * 2 + (i - RX) * T * 16), p);
        p += KST;
    };
    const int wm = wave & 1, wn = wave >> 1;
    const int l32 = lane & 31, hi = lane >> 5;
    // Lane column of a 32x32 step's D = pixel l32, rows (channels) 8 * g + 4 * hi + 0..3 in
    // registers 4g .. 4g+3.
    auto channel = [&](int j, int g) { return wn * (BN / WN) + j * 32 + 8 * g + 4 * hi; };
    float16_t acc[TM][TN];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    };
    clear();
    // Without a BatchNorm (the classifier) a bias is part of the sum, which is rounded once, as
    // nn.Linear has it.  Elsewhere, and in a pair, the sum is rounded first, as a convolution's
    // result is.  (A bias in a pair's accumulators had the 128 x 128 tiles spill: 86 -> 117 us; the rounding left out where there is no BatchNorm
    // takes 14 to 17 registers of a pair's and spills 33 of those in short stages.  A pair without one in the small tiles of ddf_net_small.hip, which have room,
    // and as the two launches it once was, is rounded once less.)
    const bool bias_in_sum = !PAIR && !a.norm.var && a.norm.conv_bias;
    // `meanwhile`: what goes out behind the products of a step, the stage's loads spread over its steps.  The
    // next step's operands are asked for in front of a step's products: left to itself the compiler keeps one set of
    // registers for operands, and every step waits out LDS.  Batch 128, us before / now: 14 x 14 x 1024 -> 256 24.2 / 22.5,
    // -> 512 43.5 / 38.0, 7 x 7 x 512 -> 2048 25.5 / 23.1, 2048 -> 512 30.4 / 29.4, 28 x 28 x 512 -> 256 42.2 / 41.0.  (All loads
    // behind the first step 23.1 and 41.3; a raised priority around the products 23.9 and 42.2.)
    constexpr int STEPS = KST / 16;
    auto multiply = [&](int buf, auto meanwhile) __attribute__((always_inline)) {
        const _Float16 *s = net_smem + buf * STAGE;
        half8_t xv[2][TM], wv[2][TN];
        auto operands = [&](int kk) __attribute__((always_inline)) {
            const int ch = kk * 2 + hi;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int r = wn * (BN / WN) + j * 32 + l32;
                wv[kk & 1][j] = *reinterpret_cast<const half8_t *>(s + BM * KST + r * KST + (ch ^ turn(r)) * 8);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int r = wm * (BM / 2) + i * 32 + l32;
                xv[kk & 1][i] = *reinterpret_cast<const half8_t *>(s + r * KST + (ch ^ turn(r)) * 8);
            }
        };
        operands(0);
#pragma unroll
        for (int kk = 0; kk < STEPS; ++kk) {
            if (kk + 1 < STEPS) operands(kk + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wv[kk & 1][j], xv[kk & 1][i], acc[i][j], 0, 0, 0);
            meanwhile(kk);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // what the tile's results meet on their way out: this thread's eight channels, and the
    // residual of its pixels
    constexpr int CPR = BN / 8;                     // vectors per pixel
    constexpr int RO = BM * CPR / T, STEP = T / CPR;
    const int cq = tid % CPR, r0 = tid / CPR, c = n0 + cq * 8;
    const bool cok = c < a.N;
    half8_t rv[RES ? RO : 1];
    auto residual = [&]() __attribute__((always_inline)) {
        if constexpr (RES) {
            const _Float16 *res = static_cast<const _Float16 *>(a.res) + m0 * a.N + (cok ? c : 0);
#pragma unroll
            for (int i = 0; i < RO; ++i)
                rv[i] = *reinterpret_cast<const half8_t *>(res + (int64_t)min(r0 + i * STEP, rows - 1) * a.N);
        }
    };
    // ReLU of rounded results, which a NaN passes: the larger of them and this
    const _Float16 least = a.relu ? (_Float16)0.f : -(_Float16)__builtin_inff();
    half4_t side[PAIR ? TM : 1][PAIR ? TN : 1][PAIR ? 4 : 1];
    auto affine_of = [&](int which, int i, int j, int g, float (&f)[4]) __attribute__((always_inline)) {
        const float4_t sc = *reinterpret_cast<const float4_t *>(&affine[which][channel(j, g)]);
        const float4_t sh = *reinterpret_cast<const float4_t *>(&affine[which + 1][channel(j, g)]);
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = fmaf((float)(_Float16)acc[i][j][4 * g + e], sc[e], sh[e]);
    };

    const int nk0 = PAIR ? first.K / KST : 0, nk = nk0 + a.K / KST;
    // (the first stages go out before anything else is asked for)
    aim(PAIR ? first : a);
    auto load_stage = [&](int k, int buf) __attribute__((always_inline)) {
        if (PAIR && k == nk0) aim(a);
#pragma unroll
        for (int i = 0; i < RX + RW; ++i) load_one(i, buf);
    };
#pragma unroll
    for (int s = 0; s < ST - 1; ++s)
        if (s < nk) load_stage(s, s);
    // (scale and shift by a thread per channel: worked out by every thread for its own eight, they were half of the way out
    // of a small launch)
    Affine<1> of[PAIR ? 2 : 1];
    if (tid < BN) {
        of[0].request(a.norm, min(n0 + tid, a.N - 1), PAIR || !bias_in_sum);
        if constexpr (PAIR) of[1].request(first.norm, min(n0 + tid, a.N - 1));
    }
    auto put_affine = [&](int which, const NetNorm &n) __attribute__((always_inline)) {
        float sc[1], sh[1];
        of[which].finish(n, sc, sh);
        affine[2 * which][tid] = sc[0];
        affine[2 * which + 1][tid] = sh[0];
    };
    if (bias_in_sum) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int o = n0 + channel(j, g);    // (rows are whole vectors of 8)
                half4_t b = {0, 0, 0, 0};
                if (o < a.N) __builtin_memcpy(&b, static_cast<const _Float16 *>(a.norm.conv_bias) + o, sizeof(b));
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][4 * g + e] = (float)b[e];
            }
    }
    if constexpr (PAIR) {
        if (tid < BN) {
            put_affine(0, a.norm);
            put_affine(1, first.norm);
        }
    }
    int buf = 0;
    auto nothing = [](int) __attribute__((always_inline)) {};
    auto loads_to = [&](int to) __attribute__((always_inline)) {
        return [&, to](int kk) __attribute__((always_inline)) {
#pragma unroll
            for (int i = kk * (RX + RW) / STEPS; i < (kk + 1) * (RX + RW) / STEPS; ++i) load_one(i, to);
        };
    };
    auto multiply_stage = [&](int k, auto meanwhile) __attribute__((always_inline)) {
        multiply(buf, meanwhile);
        buf = buf == ST - 1 ? 0 : buf + 1;
        if constexpr (PAIR) {
            if (k == nk0 - 1) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            float f[4];
                            affine_of(2, i, j, g, f);
#pragma unroll
                            for (int e = 0; e < 4; ++e) side[i][j][g][e] = (_Float16)f[e];
                        }
                clear();
            }
        }
    };
    // A stage's loads are followed by those of the ST - 2 after it, the last stage's by the
    // residual's RO, which are asked for a stage earlier than they were and in one go (a branch for
    // each and a wait between them took a memory latency per tile).  No load moves across arrive().
    if constexpr (PAIR) {
        int k = 0;
        if constexpr (STEPS > 2) {
            for (; k < nk - (ST - 1); ++k) {
                arrive<(ST - 2) * (RX + RW)>();
                if (k + ST - 1 == nk0) aim(a);
                multiply_stage(k, loads_to(buf == 0 ? ST - 1 : buf - 1));
            }
        }
        // (short stages, three workgroups a unit: 75 us where the loads between the steps take 78, 128 x 28 x 28 x
        // 128 + 256 -> 512)
        for (; k < nk; ++k) {
            if (k + 1 < nk) arrive<(ST - 2) * (RX + RW)>();
            else arrive<0>();
            if (STEPS <= 2 && k + ST - 1 < nk) load_stage(k + ST - 1, buf == 0 ? ST - 1 : buf - 1);
            multiply_stage(k, nothing);
        }
    } else {
        int k = 0;
        for (; k < nk - 2; ++k) {
            arrive<(ST - 2) * (RX + RW)>();
            const int to = buf == 0 ? ST - 1 : buf - 1;
            if constexpr (ALONE) load_stage(k + ST - 1, to);
            if constexpr (ALONE) multiply_stage(k, nothing);
            else multiply_stage(k, loads_to(to));
        }
        if (nk > 1) {
            arrive<(ST - 2) * (RX + RW)>();
            if (ST == 2) load_stage(k + 1, buf ^ 1);
        } else {
            arrive<0>();
        }
        residual();
        if (nk > 1) {
            multiply_stage(k, nothing);
            arrive<RES ? RO : 0>();
        }
        if (tid < BN) put_affine(0, a.norm);
        multiply_stage(nk - 1, nothing);
    }
    __syncthreads();
    float one = 1.f;
    asm volatile("" : "+v"(one));    // (value * one + f: a conversion less than value + f)

    // The tile through LDS as [pixel][channel]: a single product's sums rounded to fp16, a
    // pair's results.
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                half4_t v;
                if constexpr (PAIR) {
                    float f[4];
                    affine_of(0, i, j, g, f);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        f[e] = fmaf((float)side[i][j][g][e], one, f[e]);
                        asm volatile("" : "+v"(f[e]));
                        v[e] = (_Float16)f[e];
                    }
                    v = __builtin_elementwise_maximum(v, half4_t{least, least, least, least});
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = (_Float16)acc[i][j][4 * g + e];
                }
                const int px = wm * (BM / 2) + i * 32 + l32;
                *reinterpret_cast<half4_t *>(net_smem + px * PITCH + channel(j, g)) = v;
            }
    __syncthreads();
    half8_t results[RO];
#pragma unroll
    for (int i = 0; i < RO; ++i)
        results[i] = *reinterpret_cast<const half8_t *>(net_smem + (r0 + i * STEP) * PITCH + cq * 8);
    if constexpr (!PAIR) {
        float sc[8], sh[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4_t s4 = *reinterpret_cast<const float4_t *>(&affine[0][cq * 8 + h * 4]);
            const float4_t o4 = *reinterpret_cast<const float4_t *>(&affine[1][cq * 8 + h * 4]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sc[4 * h + e] = s4[e];
                sh[4 * h + e] = o4[e];
            }
        }
#pragma unroll
        for (int i = 0; i < RO; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float f = fmaf((float)results[i][e], sc[e], sh[e]);
                if constexpr (RES) f = fmaf((float)rv[i][e], one, f);
                asm volatile("" : "+v"(f));    // (rounded to fp32 first in every instance)
                results[i][e] = (_Float16)f;
            }
            results[i] = __builtin_elementwise_maximum(results[i], half8_t{least, least, least, least, least, least, least, least});
        }
    }
    _Float16 *out = static_cast<_Float16 *>(a.out) + (m0 * a.N + (int64_t)r0 * a.N + c);
#pragma unroll
    for (int i = 0; i < RO; ++i, out += (int64_t)STEP * a.N)
        if (cok && r0 + i * STEP < rows) *reinterpret_cast<half8_t *>(out) = results[i];
    if constexpr (POOL) {
        // Sums over the tile's pixels of each sample it touches, to the sample's slot for this
        // tile; the tile with a sample's last pixel clears the slots that sample does not use.
        float *red = reinterpret_cast<float *>(net_smem + BM * PITCH);    // [waves][BN]
        const int first = (int)m0, end = (int)min(m0 + BM, a.M);
        const int n_last = (int)cut.npix.of(end - 1);
        for (int n = (int)cut.npix.of(first); n <= n_last; ++n) {
            const int lo = n * a.npix - first, hi = lo + a.npix;
            float sum[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) sum[e] = 0.f;
            auto add = [&](auto whole) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < RO; ++i) {
                    const int r = r0 + i * STEP;
                    rows_u4 v = __builtin_bit_cast(rows_u4, results[i]);
                    if (!decltype(whole)::value && (r < lo || r >= hi)) v = rows_u4{0, 0, 0, 0};
                    const half8_t f = __builtin_bit_cast(half8_t, v);
#pragma unroll
                    for (int e = 0; e < 8; ++e) sum[e] = fmaf((float)f[e], one, sum[e]);
                }
            };
            if (lo <= 0 && hi >= BM) add(std::true_type{});
            else add(std::false_type{});
            // over the lanes that share this one's channels: from eight sums to the two of
            // channels 2 * row of lanes + 0..1
            if constexpr (CPR == 8) {
#pragma unroll
                for (int e = 0; e < 8; ++e) sum[e] = add_permuted<0x128 /* row_ror:8 */>(sum[e]);
            }
            float half[4], pair[2];
#pragma unroll
            for (int e = 0; e < 4; ++e) half[e] = add_swapped32(sum[e], sum[e + 4]);
#pragma unroll
            for (int e = 0; e < 2; ++e) pair[e] = add_swapped16(half[e], half[e + 2]);
            if (CPR == 16 || !(lane & 8)) {
                typedef float float2_t __attribute__((ext_vector_type(2)));
                *reinterpret_cast<float2_t *>(red + wave * BN + (lane % CPR) * 8 + (lane >> 4) * 2) = float2_t{pair[0], pair[1]};
            }
            __syncthreads();
            if (tid < BN && n0 + tid < a.N) {
                float *to = a.pool + (int64_t)n * a.pool_slots * a.N + n0 + tid;
                int slot = tm - (int)((int64_t)n * a.npix / BM);
                float total = (red[tid] + red[BN + tid]) + (red[2 * BN + tid] + red[3 * BN + tid]);
                if constexpr (WAVES == 8) total += (red[4 * BN + tid] + red[5 * BN + tid]) + (red[6 * BN + tid] + red[7 * BN + tid]);
                to[(int64_t)slot * a.N] = total;
                if (hi <= end - first)
                    while (++slot < a.pool_slots) to[(int64_t)slot * a.N] = 0.f;
            }
            if (n < n_last) __syncthreads();
        }
    }
}

// ---- stem: 7x7 convolution of stride 2, BatchNorm, ReLU, 3x3 max-pool of stride 2 ----
// A workgroup produces 8 x 8 pooled pixels x 64 channels at a time: 17 x 17 convolution
// results from 39 x 39 image pixels.  The image tile sits in LDS as [row][column][4
// channels, the last one zero]: for a filter row the eight columns under a result are 32
// contiguous values, one step of the 16x16x32 matrix instruction: the column left of the seven
// and those (the fourth channel, zeros, and that column, cleared after the read lest an infinity
// in it make a NaN, meet zero weights), so that a tile starts at an even column and comes in as
// pairs of columns.  The weights stay in registers over the tiles a workgroup walks.
// Convolution results never leave LDS (205 MB at batch 128).  The vector ALU (46 % of the clocks) and the matrix cores (44 %) bound
// it, with two waves per SIMD that wait for one another's barriers: a round's products go out between the instructions that
// finish the round before, results outside the image are left out by the pooling's addresses instead of masked one by
// one, and the pooling's lanes are laid over LDS without conflicts (8.5 -> 4.9 M clocks of them).  us, 128, 32, 8 and one image of
// 224 x 224 75.0 / 66.7, 27.6 / 25.8, 14.3 / 13.2, 10.3 / 9.0, 64 of 192 x 192 34.3 / 31.0 (128 of 224 x 224: 26 at the matrix cores' rate, 17
// for the bytes).  The first tile and the norm's parameters asked for in front of the weights: no faster.
constexpr int kPoolTile = 8, kConvTile = 2 * kPoolTile + 1, kImgRows = 2 * (kConvTile - 1) + 7, kImgCols = kImgRows + 1;
constexpr int kConvPitch = 64 + 8, kStemOut = 64;
constexpr int kStemPixels = kConvTile * kConvTile, kStemTiles = (kStemPixels + 15) / 16,
              kStemRounds = (kStemTiles + kThreads / kWave - 1) / (kThreads / kWave);

__global__ __launch_bounds__(kThreads, 2) void k_net_stem(const _Float16 *__restrict__ img,
                                                          const _Float16 *__restrict__ w, NetNorm norm,
                                                          _Float16 *__restrict__ out, int N, int H, int W, int tiles_x,
                                                          int tiles_y) {
    __shared__ __align__(16) _Float16 tile[kImgRows * kImgCols * 4];
    __shared__ __align__(16) _Float16 conv[kStemPixels * kConvPitch];
    static_assert(kStemOut * 7 * 32 <= kStemPixels * kConvPitch, "the weights pass through the results' space");
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int row = lane & 15, quad = lane >> 4;
    const int Hp = H / 4, Wp = W / 4;
    const uint32_t first_column = quad == 0 ? 0u : ~0u;   // (columns 2 * quad and 2 * quad + 1 of eight)
    // weights to LDS as [output][filter row][column * 4 + channel], then to registers
    {
        constexpr int COUNT = kStemOut * 147, R = (COUNT + kThreads - 1) / kThreads;
        _Float16 wr[R];
#pragma unroll
        for (int i = 0; i < R; ++i) wr[i] = w[min(tid + i * kThreads, COUNT - 1)];
        for (int i = tid; i < kStemOut * 7 * 32 / 8; i += kThreads)
            *reinterpret_cast<half8_t *>(conv + i * 8) = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
        __syncthreads();
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int e = tid + i * kThreads;
            const int o = e / 147, r = e - o * 147, ch = r / 49, q = r - ch * 49, ky = q / 7, kx = q - ky * 7;
            if (e < COUNT) conv[(o * 7 + ky) * 32 + (kx + 1) * 4 + ch] = wr[i];
        }
    }
    __syncthreads();
    half8_t wv[4][7];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int ky = 0; ky < 7; ++ky)
            wv[ct][ky] = *reinterpret_cast<const half8_t *>(conv + ((ct * 16 + row) * 7 + ky) * 32 + quad * 8);
    float sc[4][4], sh[4][4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
        Affine<4> aff;
        aff.request(norm, ct * 16 + quad * 4);
        aff.finish(norm, sc[ct], sh[ct]);
    }

    const int per_image = tiles_x * tiles_y, total = N * per_image;
    // The image part of a tile, two pixels of three channels per item (the width is even, so both
    // are in the image or neither): requested a tile ahead, while the matrix cores work on the one
    // before.
    constexpr int kPairs = kImgCols / 2, RI = (kImgRows * kPairs + kThreads - 1) / kThreads;
    static_assert(kImgCols % 2 == 0, "pairs of columns");
    const uint32_t plane_b = (uint32_t)(H * W) * 2;
    uint32_t pix[RI][3];
    int item_row[RI], item_col[RI];
#pragma unroll
    for (int k = 0; k < RI; ++k) {
        const int i = tid + k * kThreads;
        item_row[k] = i / kPairs;
        item_col[k] = 2 * (i - item_row[k] * kPairs);
    }
    auto request = [&](int t) {
        const int n = t / per_image, r = t - n * per_image, ty = r / tiles_x, tx = r - ty * tiles_x;
        const int iy0 = 4 * ty * kPoolTile - 5, ix0 = 4 * tx * kPoolTile - 6;   // first image pixel
        const __amdgpu_buffer_rsrc_t in = plane_rsrc(img + (int64_t)n * 3 * H * W, 3 * plane_b);
#pragma unroll
        for (int k = 0; k < RI; ++k) {
            const int yy = iy0 + item_row[k], xx = ix0 + item_col[k];
            const uint32_t off = (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W ? (uint32_t)(yy * W + xx) * 2 : kOutside;
#pragma unroll
            for (int ch = 0; ch < 3; ++ch)
                pix[k][ch] = __builtin_amdgcn_raw_buffer_load_b32(in, (int)off, (int)(ch * plane_b), 0);
        }
    };
    // Pooled pixel of a row and eight channels of a lane, a wave a row.  A pixel's neighbour is 18 places of 16 bytes further on, so
    // pixels x and x + 4 fill the sixteen places that an LDS read serves at once (lanes 0-3, 12-15, 20-27 and 4-11, 16-19,
    // 28-31 of 32).
    const int part = (lane >> 2) & 7;
    const int pool_x = ((part ^ (part >> 1) ^ (part >> 2)) & 1) + (part >> 2) * 4 + (lane >> 5) * 2;
    const int pool_c = (lane & 3) + ((part >> 1) & 1) * 4;
    if ((int)blockIdx.x < total) request(blockIdx.x);
    for (int t = blockIdx.x; t < total; t += gridDim.x) {
        const int n = t / per_image, r = t - n * per_image, ty = r / tiles_x, tx = r - ty * tiles_x;
#pragma unroll
        for (int k = 0; k < RI; ++k) {
            const int i = tid + k * kThreads;
            const rows_u4 v = {__builtin_amdgcn_perm(pix[k][1], pix[k][0], 0x05040100u), pix[k][2] & 0xffffu,
                               __builtin_amdgcn_perm(pix[k][1], pix[k][0], 0x07060302u), pix[k][2] >> 16};
            if (i < kImgRows * kPairs) *reinterpret_cast<rows_u4 *>(tile + i * 8) = v;
        }
        if (t + (int)gridDim.x < total) request(t + gridDim.x);
        __syncthreads();   // (also: the weights, or the last tile's results, have been read)
        // Sixteen results per wave and round.  A round's products go out between the instructions that finish the
        // round before: 28 of 16 clocks in the matrix cores, beside some 120 in the vector ALU.
        float4_t acc[2][4];
        int pixel[2];
        rows::static_for<0, kStemRounds + 1>([&](auto round) __attribute__((always_inline)) {
            constexpr int I = decltype(round)::value;
            if constexpr (I < kStemRounds) {
                // (past the last: the last one again, the same bits to the same place)
                const int pc = min((I * (kThreads / kWave) + wave) * 16 + row, kStemPixels - 1);
                const int cy = pc / kConvTile, cx = pc - cy * kConvTile;
                const _Float16 *src = tile + (2 * cy * kImgCols + 2 * cx + quad * 2) * 4;
                pixel[I & 1] = pc;
#pragma unroll
                for (int ct = 0; ct < 4; ++ct) acc[I & 1][ct] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ky = 0; ky < 7; ++ky) {
                    rows_u4 words = *reinterpret_cast<const rows_u4 *>(src + ky * kImgCols * 4);
                    words[0] &= first_column;
                    words[1] &= first_column;
                    const half8_t b = __builtin_bit_cast(half8_t, words);
#pragma unroll
                    for (int ct = 0; ct < 4; ++ct)
                        acc[I & 1][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[ct][ky], b, acc[I & 1][ct], 0, 0, 0);
                }
            }
            if constexpr (I > 0) {
                // (results outside the image are whatever the zeros there give: no maximum reads them)
                constexpr int P = (I - 1) & 1;
                _Float16 *const to = conv + pixel[P] * kConvPitch + quad * 4;
#pragma unroll
                for (int ct = 0; ct < 4; ++ct) {
                    half4_t v;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
                        // (two sums rounded by one instruction)
                        uint32_t sums = __builtin_bit_cast(uint32_t, half2_t{(_Float16)acc[P][ct][2 * h], (_Float16)acc[P][ct][2 * h + 1]});
                        asm volatile("" : "+v"(sums));
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            float f = fmaf((float)__builtin_bit_cast(half2_t, sums)[e], sc[ct][2 * h + e], sh[ct][2 * h + e]);
                            asm volatile("" : "+v"(f));
                            v[2 * h + e] = (_Float16)f;
                        }
                    }
                    *reinterpret_cast<half4_t *>(to + ct * 16) = __builtin_elementwise_maximum(v, half4_t{0, 0, 0, 0});
                }
            }
            if constexpr (I > 0 && I < kStemRounds) {
                __builtin_amdgcn_sched_group_barrier(0x100 /* LDS reads */, 7, 0);
                rows::static_for<0, 28>([&](auto) __attribute__((always_inline)) {
                    __builtin_amdgcn_sched_group_barrier(0x2 /* vector ALU */, 4, 0);
                    __builtin_amdgcn_sched_group_barrier(0x8 /* a product */, 1, 0);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPoolTile * kWave / kThreads; ++k) {
            const int py = wave + k * (kThreads / kWave);
            const int oy = ty * kPoolTile + py, ox = tx * kPoolTile + pool_x;
            // (the row above and the column left of the image: the next ones, which a maximum takes in any case.
            // Those past its other edges belong to pixels that are not stored)
            const int up = 2 * py + (oy == 0), left = 2 * pool_x + (ox == 0);
            half8_t m = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                for (int dx = 0; dx < 3; ++dx) {
                    const half8_t v = *reinterpret_cast<const half8_t *>(
                        conv + ((dy ? 2 * py + dy : up) * kConvTile + (dx ? 2 * pool_x + dx : left)) * kConvPitch + pool_c * 8);
                    m = __builtin_elementwise_maximum(m, v);
                }
            if (oy < Hp && ox < Wp)
                *reinterpret_cast<half8_t *>(out + (((int64_t)n * Hp + oy) * Wp + ox) * kStemOut + pool_c * 8) = m;
        }
        // (the next tile's image part does not touch `conv`, and its barrier comes before
        // the next results do)
    }
}

// ---- filter branches --------------------------------------------------------------
// Both branches depend on the first convolution only - the spatial one on its results, the
// channel one on their sums, which the convolution leaves - so one launch has them both: its first
// workgroups are the channel branch (ddf_channel.h), a chain of round trips, the others the
// spatial one.  A wave of the spatial branch takes
// tiles of sixteen pixels, as many at a time as make eight loads, its weights in registers; under
// stride 2 only the sampled pixels are read.  us for both branches, as two launches with the pooling
// in the spatial one (which then read every pixel under stride 2, too) / now, batch 128: 56 x 56 x 64
// 21.0 / 20.5, 28 x 28 x 128 16.8 / 14.0, from 56 x 56 under stride 2 31.5 / 12.9, 14 x 14 x 256
// 17.0 / 7.6, from 14 x 14 x 512 under stride 2 28.5 / 13.6; one image, 56 x 56 x 64 10.5 / 5.3,
// 14 x 14 x 256 13.4 / 5.8, 7 x 7 x 512 16.2 / 6.9.  (The spatial taps in the first convolution,
// where its tile has all channels: 8 us more there, 8 less here, and a slower filter, whose
// operands this launch leaves in the caches.)
struct NetTaps {
    const _Float16 *x, *w, *bias;
    _Float16 *sf;
    int W, Wo, npix, plane, pixels, tiles;    // npix, plane: results, pixels of a sample; pixels: results of all
    float gain;
    Divisor sample, row;    // by npix, by Wo
};

template <int KS, int S, int U>
__device__ __forceinline__ void net_taps(const NetTaps &a, int wave, int waves) {
    constexpr int C = KS * 32;
    const int lane = threadIdx.x & (kWave - 1), col = lane & 15, quad = lane >> 4;
    TapWeights<KS> weights;
    weights.request(a.w, a.bias, lane);
    for (int t0 = wave * U; t0 < a.tiles; t0 += waves * U) {
        half8_t v[U][KS];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int p = min((t0 + u) * 16 + col, a.pixels - 1);    // (past the last: not stored)
            int64_t at = p;
            if constexpr (S == 2) {
                const int n = (int)a.sample.of(p), q = p - n * a.npix, y = (int)a.row.of(q), xx = q - y * a.Wo;
                at = (int64_t)n * a.plane + 2 * y * a.W + 2 * xx;
            }
            const _Float16 *src = a.x + at * C + quad * 8;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) v[u][ks] = *reinterpret_cast<const half8_t *>(src + ks * 32);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int p = (t0 + u) * 16 + col;
            weights.taps(v[u], a.gain, p < a.pixels, a.sf, p, lane);
        }
    }
}

// Workgroups of the channel branch in front of those of the spatial one.
enum { kNoChannels, kChannelsRows, kChannelsMma };
template <int CH> struct ChannelArgs { };
template <> struct ChannelArgs<kChannelsRows> { ChannelRows<__half> a; };
template <> struct ChannelArgs<kChannelsMma> { ChannelMma a; };
constexpr int branch_threads(int ch) { return ch == kChannelsRows ? kRowsThreads : kMmaThreads; }

template <int KS, int S, int U, int CH>
__global__ __launch_bounds__(branch_threads(CH)) void k_net_branches(NetTaps taps, ChannelArgs<CH> channels, int blocks_x,
                                                                     int blocks) {
    extern __shared__ __align__(16) unsigned char branch_smem[];
    at_once(taps.x, taps.w, taps.bias, taps.sf, taps.W, taps.Wo, taps.npix, taps.plane, taps.pixels, taps.tiles, blocks, blocks_x);
    const int block = blockIdx.x;
    if constexpr (CH != kNoChannels) {
        if (block < blocks) {
            const int by = block / blocks_x, bx = block - by * blocks_x;
            const ToFilter<__half, 9> sink{channels.a.cf, channels.a.C};
            if constexpr (CH == kChannelsRows) {
                channel_rows<__half, false>(channels.a, bx, by, branch_smem, Nothing(), Nothing(), Nothing(), sink);
            } else {
                const int n0 = by * kMmaSamples;
                channel_mma<9, false>(channels.a, bx, n0, min(kMmaSamples, channels.a.N - n0), branch_smem, Nothing(), Nothing(), Nothing(), sink);
            }
            return;
        }
    }
    constexpr int WAVES = branch_threads(CH) / kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    net_taps<KS, S, U>(taps, (block - blocks) * WAVES + wave, (gridDim.x - blocks) * WAVES);
}

// ---- dynamic filter + BatchNorm + ReLU ---------------------------------------------
// C / 8 lanes own a pixel, eight channels each, and walk along a row: the window slides, so
// a step loads one new column (three 16-byte vectors; two columns under stride 2), a step
// ahead of use.  The channel taps of the lane's channels stay in registers; a pixel's nine spatial
// taps come with it.  comb(CF, SF) is one packed fp16 operation for two (rounded like the
// operands), the sums are fp32.  Filter rows 0 and 1 of a channel are a pair, so the two-element
// dot product takes both (a column's eight words are paired once for the three results it is
// under); row 2 goes two channels at a time.  With ReLU on rounded pairs a result takes 140 vector
// instructions where it took 175: 56 x 56 x 64 at batch 128 26.2 -> 25.3 us, 28 x 28 x 128 17.5 ->
// 16.4; what is left is the latency of a column, at two to three waves per SIMD.  WIDE: comb in
// fp32 - for rows of an odd length, where the operator's own kernels have it so.  A row outside the
// image, a column past its ends and a walk past the last pixel read zeros through the buffer
// descriptor.
template <int LP, int S, bool MUL, bool WIDE>
__global__ __launch_bounds__(kThreads) void k_net_filter(const _Float16 *__restrict__ x,
                                                         const _Float16 *__restrict__ cf,
                                                         const _Float16 *__restrict__ sf, NetNorm norm,
                                                         _Float16 *__restrict__ out, int H, int W, int Ho, int Wo,
                                                         Divisor runs, Divisor rows, int run, int units, int blocks,
                                                         uint32_t x_bytes, uint32_t out_bytes, uint32_t tap_bytes) {
    constexpr int C = LP * 8, SLOTS = kWave / LP, KK = 9;
    at_once(x, cf, sf, out, H, W, Wo, run, units, blocks, x_bytes, tap_bytes);
    at_once(runs.by, runs.magic, rows.by, rows.magic);
    const int block = xcd_block(blockIdx.x, blocks);
    if (block >= blocks) return;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int cl = lane % LP;
    const int unit = (block * (kThreads / kWave) + wave) * SLOTS + lane / LP;
    const bool live = unit < units;
    const int u = live ? unit : units - 1;
    const int row = (int)runs.of(u), r = u - row * (int)runs.by;
    const int n = (int)rows.of(row), y = row - n * Ho;
    const int x0 = r * run;
    const int x1 = live ? min(x0 + run, Wo) : x0;
    // (lanes of a wave may belong to different samples: one descriptor over all of them)
    const __amdgpu_buffer_rsrc_t xr = plane_rsrc(x, x_bytes);
    const __amdgpu_buffer_rsrc_t tr = plane_rsrc(sf, tap_bytes);
    const uint32_t tap_row = (uint32_t)((n * Ho + y) * Wo) * (kTapPitch * 2);
    const __amdgpu_buffer_rsrc_t orr = plane_rsrc(out, out_bytes);
    const uint32_t oo = (uint32_t)(((n * Ho + y) * Wo) * C + cl * 8) * 2;

    Affine<8> aff;
    aff.request(norm, cl * 8);
    uint32_t cfa[3][8], cfb[3][4];
    channel_taps(cf + ((int64_t)n * C + cl * 8) * KK, cfa, cfb);
    uint32_t rowo[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int yy = y * S - 1 + i;
        rowo[i] = (live && yy >= 0 && yy < H) ? (uint32_t)(((n * H + yy) * W) * C + cl * 8) * 2 : kOutside;
    }
    float sc[8], sh[8];
    // Columns in rings of registers, all indices constants (as structures handed around they
    // were parked in LDS, and every step waited for its own loads: 60 us where this takes 25
    // at 128 x 56 x 56 x 64).
    constexpr int RING = S == 1 ? 4 : 6;
    uint32_t col[RING][3][4], tap[2][6];
    auto column = [&](auto slot, int xx) __attribute__((always_inline)) {
        constexpr int J = decltype(slot)::value % RING;
        // (a column outside, a row outside or both: past the descriptor's end and short of 2^32)
        const uint32_t at = (unsigned)xx < (unsigned)W ? (uint32_t)xx * C * 2 : kOutside - 16;
#pragma unroll
        for (int i = 0; i < 3; ++i) load_words<4>(xr, rowo[i] + at, col[J][i]);
    };
    auto taps = [&](auto slot, int xx) __attribute__((always_inline)) {
        constexpr int J = decltype(slot)::value % 2;
        const uint32_t at = tap_row + (uint32_t)min(xx, Wo - 1) * (kTapPitch * 2);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            uint32_t q[2];
            load_words<2>(tr, at + i * 8, q);
            tap[J][2 * i] = q[0];
            tap[J][2 * i + 1] = q[1];
        }
    };
    auto pair_rows = [&](auto slot) __attribute__((always_inline)) { pair_column(col[decltype(slot)::value % RING]); };
    // result xx from the columns in slots A, A + 1 and A + 2 and the taps in slot J
    auto emit = [&](auto first, auto slot, int xx) __attribute__((always_inline)) {
        constexpr int A = decltype(first)::value, J = decltype(slot)::value % 2;
        float acc[8];
        filter_sums<MUL, WIDE>(cfa, cfb, col[A % RING], col[(A + 1) % RING], col[(A + 2) % RING], tap[J], acc);
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            // (the complete sum is rounded as the operator's result is)
            float f = fmaf((float)(_Float16)acc[e], sc[e], sh[e]);
            asm volatile("" : "+v"(f));
            o[e] = (_Float16)f;
        }
        o = __builtin_elementwise_maximum(o, half8_t{0, 0, 0, 0, 0, 0, 0, 0});
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(rows_u4, o), orr,
                                               (int)(xx < x1 ? oo + (uint32_t)xx * C * 2 : kOutside), 0, 0);
    };
#define DDF_I(v) std::integral_constant<int, (v)>{}
    if constexpr (S == 1) {
        column(DDF_I(0), x0 - 1);
        column(DDF_I(1), x0);
        column(DDF_I(2), x0 + 1);
        taps(DDF_I(0), x0);
        aff.finish(norm, sc, sh);
        pair_rows(DDF_I(0));
        pair_rows(DDF_I(1));
        for (int j = 0; j < run; j += 4) {
            rows::static_for<0, 4>([&](auto q) __attribute__((always_inline)) {
                constexpr int Q = decltype(q)::value;
                const int xx = x0 + j + Q;
                column(DDF_I(Q + 3), xx + 2);
                taps(DDF_I(Q + 1), xx + 1);
                __builtin_amdgcn_sched_barrier(0);
                pair_rows(DDF_I(Q + 2));
                emit(DDF_I(Q), q, xx);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
    } else {
        // (three pairs of columns: slots 2q - 1, 2q and 2q + 1 are under result q)
        column(DDF_I(5), 2 * x0 - 1);
        column(DDF_I(0), 2 * x0);
        column(DDF_I(1), 2 * x0 + 1);
        taps(DDF_I(0), x0);
        aff.finish(norm, sc, sh);
        pair_rows(DDF_I(5));
        for (int j = 0; j < run; j += 6) {
            rows::static_for<0, 6>([&](auto q) __attribute__((always_inline)) {
                constexpr int Q = decltype(q)::value;
                const int xx = x0 + j + Q;
                column(DDF_I(2 * Q + 2), 2 * xx + 2);
                column(DDF_I(2 * Q + 3), 2 * xx + 3);
                taps(DDF_I(Q + 1), xx + 1);
                __builtin_amdgcn_sched_barrier(0);
                pair_rows(DDF_I(2 * Q));
                pair_rows(DDF_I(2 * Q + 1));
                emit(DDF_I(2 * Q + 5), q, xx);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
    }
#undef DDF_I
}

// ---- branches and dynamic filter in one launch, few pixels ---------------------------------
// Where the two launches are latency, a workgroup computes sixteen channels' taps, the spatial
// taps of `rows` result rows and those rows' results of its channels: every workgroup of a sample
// recomputes the hidden vector, every one of a row its spatial taps, and neither goes through
// memory.  The rows it reads (and zeros around them) come into LDS as [pixel][16 channels] while
// the channel branch waits for its weights, the spatial taps are computed meanwhile; then every
// thread takes four (of sixteen waves, two) channels of a pixel.  Rounding is k_net_filter's.  us, two
// launches / this: one image 56 x 56 x 64 10.3 / 6.2, 28 x 28 x 128 10.4 / 5.9, 14 x 14 x 256 10.6 /
// 6.1, 7 x 7 x 512 11.9 / 7.9; most of it is the channel branch's chain and the instructions in front
// of the first barrier (divisions by runtime values there cost 1 us).  Weights go out in front of everything else; a
// conversion that the compiler does where its operand is asked for was a trip to memory in front of a barrier, and eight
// channels to half of the threads 0.4 us: 7.4, 7.0, 6.7 and 8.1 us a launch with those.
struct NetFew {
    const _Float16 *x, *tap_w, *tap_bias;
    _Float16 *out;
    NetNorm norm;
    int H, W, Ho, Wo, rows;
    int per_row;                               // 64 vectors of a row of W + 2 pixels
    uint32_t per_row_magic;                    // 2^16 / per_row, rounded up
    uint32_t wo_magic;                         // 2^20 / Wo, rounded up
    float tap_gain;
    int sf, tile, channels;                    // where in LDS (bytes): spatial taps, rows, the channel branch's
};
constexpr int kFewItems = 3;
// One workgroup per compute unit, of up to this many pixels: with more of them the launch takes longer than the two it
// replaces (ResNet-50, us, at most 256 or 512 / at most 128 / two launches: 1 image 342 / 340 / 385, 8 471 / 458 /
// 468, 16 596 / 573 / 570).
constexpr int kFewBlocks = 256, kFewPixels = 128;
constexpr int kFewCf = 9 * kMmaChannels * 2;   // the channels' taps [tap][channel], at LDS 0

template <int KS, int S, bool MUL, bool WIDE, int CH>
__global__ __launch_bounds__(branch_threads(CH)) void k_net_filter_few(NetFew a, ChannelArgs<CH> channels) {
    constexpr int C = KS * 32, KK = 9, GROUPS = C / kMmaChannels, THREADS = branch_threads(CH), WAVES = THREADS / kWave;
    constexpr int ITEMS = kFewItems;           // 16-byte vectors of the rows per thread at most
    constexpr int V = kMmaChannels * kFewPixels / THREADS, PER = kMmaChannels / V;    // channels of a thread, threads of a pixel
    typedef _Float16 lane_t __attribute__((ext_vector_type(V)));
    extern __shared__ __align__(16) unsigned char few_smem[];
    _Float16 *cfs = reinterpret_cast<_Float16 *>(few_smem), *sfs = reinterpret_cast<_Float16 *>(few_smem + a.sf);
    rows_u4 *tile = reinterpret_cast<rows_u4 *>(few_smem + a.tile);
    at_once(a.x, a.H, a.W, a.Ho, a.Wo, a.rows, a.per_row, a.per_row_magic, a.wo_magic, a.sf, a.tile, a.channels);
    at_once(a.norm.weight, a.norm.bias, a.norm.mean, a.norm.var);
    const int g = blockIdx.x % GROUPS, chunk = blockIdx.x / GROUPS, n = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int y0 = chunk * a.rows, rows = min(a.rows, a.Ho - y0), pixels = rows * a.Wo;
    const uint32_t sample_bytes = (uint32_t)(a.H * a.W) * C * 2;
    const _Float16 *xn = a.x + (int64_t)n * a.H * a.W * C;

    // Rows S * y0 - 1 .. S * (y0 + rows - 1) + 1, columns -1 .. W, both halves of a pixel: a wave
    // takes 64 vectors of a row at a time (no division per lane: with sixteen waves that alone was
    // 1 us).
    const int pitch = a.W + 2, waves_of = (S * (rows - 1) + 3) * a.per_row;
    const __amdgpu_buffer_rsrc_t xr = plane_rsrc(xn, sample_bytes);
    rows_u4 part[ITEMS];
    int to[ITEMS];
    // (row of a result pixel of the workgroup: below 512, as Wo is)
    auto row_of = [&](int q) __attribute__((always_inline)) { return (int)(((uint32_t)q * a.wo_magic) >> 20); };
    const int o = tid % PER, p = tid / PER;
    const int c = g * kMmaChannels + o * V;
    Affine<V> aff;
    // Spatial taps by the last waves first, which have nothing to do when the hidden values are
    // made: the pixels of a wave's first tile are requested early, its taps are worked out then.
    TapWeights<KS> weights;
    half8_t v[KS];
    auto pixels_of = [&](int t) __attribute__((always_inline)) {
        const int q = min(t * 16 + (lane & 15), pixels - 1), y = row_of(q), x = q - y * a.Wo;
        const _Float16 *src = xn + (int64_t)(S * (y0 + y) * a.W + S * x) * C + (lane >> 4) * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) v[ks] = *reinterpret_cast<const half8_t *>(src + ks * 32);
    };
    const int t_first = WAVES - 1 - wave;
    constexpr bool kEarly = KS <= 8;           // (512 channels: no registers for that)
    // (a wave that fetches weights asks for these behind them: it waits for all of it)
    auto early = [&]() __attribute__((always_inline)) {
        aff.request(a.norm, c);
        if (kEarly && t_first * 16 < pixels) {
            pixels_of(t_first);
            weights.request(a.tap_w, a.tap_bias, lane);
        }
    };
    auto begin = [&](bool loader) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            to[k] = -1;
            if (wave + k * WAVES >= waves_of) continue;
            const int i = wave + k * WAVES, yy = (int)((uint32_t)i * a.per_row_magic >> 16), at = (i - yy * a.per_row) * kWave + lane;
            const int y = S * y0 - 1 + yy, x = (at >> 1) - 1;
            to[k] = at < 2 * pitch ? yy * 2 * pitch + at : -1;
            const bool in = to[k] >= 0 && y >= 0 && y < a.H && x >= 0 && x < a.W;
            part[k] = __builtin_bit_cast(rows_u4, __builtin_amdgcn_raw_buffer_load_b128(
                xr, in ? ((y * a.W + x) * C + g * kMmaChannels + (at & 1) * 8) * 2 : (int)kOutside, 0, 0));
        }
        if (loader) early();
    };
    auto meanwhile = [&](bool loader) __attribute__((always_inline)) {
        if (!loader) early();
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (to[k] >= 0) tile[to[k]] = part[k];
    };
    float sc[V], sh[V];
    auto after = [&]() __attribute__((always_inline)) {
        aff.finish(a.norm, sc, sh);
        weights.hold();
        for (int t = t_first; t * 16 < pixels; t += WAVES) {
            if (!kEarly || t != t_first) pixels_of(t);
            if (!kEarly) weights.request(a.tap_w, a.tap_bias, lane);
            weights.taps(v, a.tap_gain, t * 16 + (lane & 15) < pixels, sfs, t * 16 + (lane & 15), lane);
        }
    };
    auto sink = [&](int64_t, int c, const float (&u)[KK]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < KK; ++t) cfs[t * kMmaChannels + (c & (kMmaChannels - 1))] = (_Float16)u[t];
    };
    if constexpr (CH == kChannelsRows) channel_rows<__half, false>(channels.a, g, n, few_smem + a.channels, begin, meanwhile, after, sink);
    else channel_mma<KK, false>(channels.a, g, n, 1, few_smem + a.channels, begin, meanwhile, after, sink);
    __syncthreads();
    if (p >= pixels) return;
    const int y = row_of(p), x = p - y * a.Wo;
    uint32_t tap[6];
    __builtin_memcpy(tap, __builtin_assume_aligned(sfs + p * kTapPitch, 8), sizeof(tap));
    float acc[V];
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] = 0.f;
    const lane_t *const xs = reinterpret_cast<const lane_t *>(tile) + o, *const cs = reinterpret_cast<const lane_t *>(cfs) + o;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int t = i * 3 + j;
            const half2_t sp = __builtin_bit_cast(half2_t, tap[t / 2]);
            const half2_t sv = {sp[t & 1], sp[t & 1]};
            const lane_t xw = xs[((S * y + i) * pitch + S * x + j) * PER], cw = cs[t * PER];
#pragma unroll
            for (int k = 0; k < V / 2; ++k)
                filter_pair<MUL, WIDE>(half2_t{cw[2 * k], cw[2 * k + 1]}, sv, half2_t{xw[2 * k], xw[2 * k + 1]}, acc[2 * k], acc[2 * k + 1]);
        }
    lane_t r;
#pragma unroll
    for (int e = 0; e < V; ++e) r[e] = (_Float16)relu(fmaf((float)(_Float16)acc[e], sc[e], sh[e]));
    *reinterpret_cast<lane_t *>(a.out + (((int64_t)n * a.Ho + y0 + y) * a.Wo + x) * C + c) = r;
}

// ---- mean (fp16) or sum (fp32) over the pixels ---------------------------------------------
template <typename O>
__global__ __launch_bounds__(kThreads) void k_net_pool(const _Float16 *__restrict__ x, O *__restrict__ out,
                                                       int plane, int C) {
    constexpr int LANES = 32, GROUPS = kThreads / LANES;
    __shared__ float red[GROUPS][LANES * 8];
    const int l = threadIdx.x % LANES, grp = threadIdx.x / LANES;
    const int n = blockIdx.y, c = blockIdx.x * LANES * 8 + l * 8;
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    if (c < C) {
        const _Float16 *p = x + (int64_t)n * plane * C + c;
#pragma unroll 4
        for (int i = grp; i < plane; i += GROUPS) {
            const half8_t v = *reinterpret_cast<const half8_t *>(p + (int64_t)i * C);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] += (float)v[e];
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) red[grp][l * 8 + e] = acc[e];
    __syncthreads();
    const int i = threadIdx.x, cc = blockIdx.x * LANES * 8 + i;
    if (cc >= C) return;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < GROUPS; ++k) s += red[k][i];
    if constexpr (sizeof(O) == 2) out[(int64_t)n * C + cc] = (O)(s / (float)plane);
    else out[(int64_t)n * C + cc] = s;
}

template <int BM, int BN, int KST, int ST, int WN, int WG>
hipError_t launch_conv(const NetConv &a, const NetConv *first, hipStream_t st) {
    const int tiles_n = (int)cdiv(a.N, BN);
    const int64_t tiles = cdiv(a.M, BM) * tiles_n;
    if (tiles > (1 << 30)) return hipErrorInvalidConfiguration;
    const int lds = conv_lds_halves<BM, BN, KST, ST, 2 * WN>() * (int)sizeof(_Float16);
    // (a strided product's pixels are counted from a sample's first: below npix + BM; a pooled one's from the first)
    const NetConv &x = first ? *first : a;
    const TileCut cut{(int)tiles, Divisor::make(tiles_n, tiles), Divisor::make(x.npix, a.pool ? a.M : x.npix + (int64_t)BM), Divisor::make(x.Wo, x.npix)};
    // A workgroup that has its unit to itself waits for its next stages: their loads go out in front of the products.  us, between / in
    // front, 640 x 2048 -> 1000, 160 tiles, 11.7 / 11.0, 400 x 2048 -> 1000, 112, 10.8 / 10.0; networks of 14 to 27 images of 96 x 96
    // or 64 x 128 0.5 to 1 % less.  With more tiles other workgroups fill the waits, and in front is the slower order (a network of 56 images of
    // 224 x 224 867 / 875, of 10 of 288 x 288 514 / 521).
    constexpr bool kSmall = BM * BN <= 64 * 64;
    const bool alone = kSmall && tiles <= 256;
#define DDF_NET_CONV(POOL_, RES_)                                                                   \
    do {                                                                                            \
        if (alone)                                                                                  \
            hipLaunchKernelGGL((k_net_conv<BM, BN, KST, ST, WN, WG, false, POOL_, RES_, kSmall>), dim3(xcd_grid(tiles)), \
                               dim3(2 * WN * kWave), lds, st, a, a, cut);                 \
        else                                                                                        \
            hipLaunchKernelGGL((k_net_conv<BM, BN, KST, ST, WN, WG, false, POOL_, RES_>), dim3(xcd_grid(tiles)), \
                               dim3(2 * WN * kWave), lds, st, a, a, cut);                 \
    } while (0)
    if (first)
        hipLaunchKernelGGL((k_net_conv<BM, BN, KST, ST, WN, WG, true, false, false>), dim3(xcd_grid(tiles)), dim3(2 * WN * kWave), lds, st, a,
                           *first, cut);
    else if (a.pool) DDF_NET_CONV(true, false);
    else if (a.res) DDF_NET_CONV(false, true);
    else DDF_NET_CONV(false, false);
#undef DDF_NET_CONV
    return hipGetLastError();
}

// Tiles of 128 x 128, two workgroups of eight waves per compute unit, wherever they leave more than one workgroup per unit.  Four waves per SIMD
// cover one another's LDS and barriers better than two or three (four waves per workgroup: 132 to 203 registers), whatever the stages.
// us, four waves of three short stages / of two long ones / eight of two long ones: 25088 pixels 1024 -> 256 with sums over the pixels 24.1 / 21.9 / 21.7, 256 -> 1024
// with a residual 27.9 / 27.8 / 27.1, 50176 512 -> 256 25.5 / 22.9 / 22.6, pairs 128 + 256 -> 512 of 12544, 25088 and 50176 pixels 14.5 / 13.8 / 13.4, 25.9 / 24.2 /
// 22.7, 40.2 / 41.8 / 38.9, 256 + 512 -> 1024 of 25088 64.9 / 62.8 / 60.0.  With many tiles of short sums memory counts more, and three
// workgroups of four waves in short stages are ahead: a product of less than 768 from 1024 tiles on, with a residual from 2048, a pair of less than 1024 from 2048.  us, eight waves /
// short stages, operands of the call before in cache | others': with sums over the pixels 100352 pixels, 1568 tiles, 64 -> 256 16.0 / 15.3 | 21.5 / 20.1, 256 -> 256
// 31.2 / 26.8 | 37.2 / 32.6, 512 -> 256 45.4 / 41.9 | 54.2 / 50.4, 640 -> 256 52.9 / 52.1 | 66.3 / 62.4, 768 -> 256 61.1 / 61.1 | 73.9 / 70.2, 1024 -> 256 76.2 / 80.2 | 91.3 /
// 91.1, 2048 -> 256 171.7 / 171.8 | 169.5 / 172.1; 25088 512 -> 1024 40.0 / 41.5 | 49.7 / 45.7, 768 -> 1024 55.1 / 60.2 | 66.8 / 64.7; with a residual
// 50176 256 -> 512 28.9 / 27.6 | 36.5 / 34.1, 1024 -> 512 71.7 / 77.3 | 88.7 / 87.7; below 1024 tiles 760 of 256 20.6 / 18.8 and 1018 23.5 / 23.8 (not in cache); pairs
// 128 + 256 -> 512 1300 tiles 32.0 / 32.9 | 36.4 / 37.3, 1960 43.4 / 44.6 | 51.1 / 50.6, 3136 68.9 / 69.8 | 82.0 / 79.4, 256 + 512 -> 1024 1300 48.4 / 52.7 | 54.9 / 55.7, 3136 110 /
// 119 | 130 / 128, 512 + 1024 -> 2048 3136 191 / 221 | 214 / 228.  (In a network, whose other products of
// these sizes are in chains, five of 25088 256 -> 1024 with a residual, 1568 tiles, by eight waves are 2 us less of 1534, of 104 images 3 of 1351.)
// Up to one workgroup per unit the stages themselves are the time, and a third one in flight is what helps: us, tiles of 64 x 64 / 128 x 128 in two
// stages / in three, 12544 pixels 1024 -> 256, 196 tiles, 16.9 / 16.1 / 13.2, 6272 2048 -> 512 28.4 / 28.8 / 22.1, pairs 256 + 512 -> 1024 of 3136 14.8 /
// 13.2 / 11.9, 512 + 1024 -> 2048 of 1568 24.3 / 23.5 / 18.4, 148 tiles of K = 2048 21.7 / 27.5 / 20.9.  Fewer than that fill the chip better in
// tiles of 64: 100 of K = 2048 16.0 / 26.0 / 19.5, of 1024 9.8 / 13.8 / 11.5; 160 of 512 8.1 / 8.9 / 8.3; 152 of 256 5.7 / 6.1 / 6.2.
// Where the last round of two per unit would be nearly empty, 128 x 64, three workgroups per unit: us, 128 x 128 / 128 x 64, 294 tiles
// of 18816 1024 -> 256 20.4 / 20.0, 304 of 2048 19.6 / 18.5, 304 of a pair 27.6 / 26.8; 588 of 75264 512 -> 128 22.0 / 20.5, 592 of 512 -> 2048 19.6 / 18.5, of
// pairs 27.8 / 26.9 and 49.2 / 46.3; 344 tiles 20.2 / 20.1, 688 50.2 / 51.1 (operands in cache, 60 sizes of 520 to 608 tiles 1 to 12 % less; from memory 3 to 9 %
// less for 256 channels, up to 14 more for 2048).  Of fewer than 128 channels 128 x 64 in short stages from 1024 tiles on, in long
// ones from 448.
// In small tiles (ddf_net_small.hip), whose workgroups bring in a quarter of K per wave, what leaves most of the chip idle in tiles
// of 64: 16 x 16 up to two workgroups per compute unit, 32 x 32 of a K that is worth four waves up to one.  us, tiles of 64 / 16 x 16 / 32 x 32:
// 64 -> 64 of 1024 pixels, 256 tiles of 16, 2.95 / 2.88, 392 2.96 / 3.18 (a K of 64 is one wave's); 512 -> 128 784 pixels, 392, 4.28 / 3.58,
// 1568 pixels, 784 and 196 of 32, 4.35 / 5.52 / 4.29; 256 -> 128 512 tiles 3.65 / 3.32, 784 and 196 3.69 / 4.96 / 3.95; 1024 -> 256 196
// pixels 4.35 / 3.60, 400 5.70 / 4.27 / 5.05, 784 6.19 / 6.72 / 5.21, 1568, 392 of 32, 6.67 / 11.3 / 9.14; 2048 -> 512 49 6.09 / 4.26, 400
// 10.2 / 10.1 / 7.1; 512 -> 2048 with a residual 49 pixels 4.21 / 3.14; pairs 256 + 512 -> 1024 49 7.06 / 3.68, 196 6.53 / 6.83 / 5.34, 512 +
// 1024 -> 2048 49, 512 tiles, 8.95 / 5.86, 98 9.73 / 9.64 / 7.42; 2048 -> 1000 of 1, 49 and 128 rows 4.51 / 3.71, 6.53 / 5.23, 9.5 / 7.3 / 5.9.
enum ConvTile { kSmall16, kSmall32, kTile128, kTile128Short, kTile128Deep, kTile128x64, kTile128x64Long, kTile64 };
ConvTile conv_tile(const NetConv &a, const NetConv *first) {
    const bool pair = first;
    const int64_t K = (int64_t)a.K + (pair ? first->K : 0);
    auto count = [&](int bm, int bn) { return cdiv(a.M, bm) * cdiv(a.N, bn); };
    constexpr int kMany = 1024;
    if (a.N % 8 != 0 || count(16, 16) <= (K > 64 ? 512 : 256)) return kSmall16;
    if (K > 256 && count(32, 32) <= 256) return kSmall32;
    if (a.N >= 128) {
        const int64_t tiles = count(128, 128);
        if (tiles <= 256 && tiles > (K >= 1024 ? 128 : 160)) return kTile128Deep;
        if (tiles >= (pair || a.res ? 2048 : 1024) && K < (pair ? 1024 : 768)) return kTile128Short;
        if (tiles >= 320 && (tiles <= 512 || tiles > 608)) return kTile128;
    } else if (count(128, 64) >= kMany) {
        return kTile128x64;
    }
    if (count(128, 64) >= 448) return kTile128x64Long;
    return kTile64;
}
int tile_rows(ConvTile t) { return t == kSmall16 ? 16 : t == kSmall32 ? 32 : t == kTile64 ? 64 : 128; }

hipError_t conv_tiles(ConvTile tile, const NetConv &a, const NetConv *first, hipStream_t st) {
    switch (tile) {
        case kSmall16: return net_conv_small(16, a, first, st);
        case kSmall32: return net_conv_small(32, a, first, st);
        case kTile128: return launch_conv<128, 128, 64, 2, 4, 2>(a, first, st);
        case kTile128Short: return launch_conv<128, 128, 32, 3, 2, 3>(a, first, st);
        case kTile128Deep: return launch_conv<128, 128, 64, 3, 4, 1>(a, first, st);
        case kTile128x64: return launch_conv<128, 64, 32, 3, 2, 4>(a, first, st);
        case kTile128x64Long: return launch_conv<128, 64, 64, 2, 2, 3>(a, first, st);
        default: return launch_conv<64, 64, 64, 3, 2, 3>(a, first, st);
    }
}

}  // namespace

bool net_conv_supported(const NetConv &a) { return a.K % 64 == 0 && a.K > 0 && a.N > 0; }

// Slots of a sample in a convolution's sums over its pixels: one per tile of rows that a sample
// can touch (samples start at multiples of the common divisor of their pixels and the tile).
int net_conv_pool_slots(const NetConv &a) {
    const int rows = tile_rows(conv_tile(a, nullptr)), start = a.M > a.npix ? rows - std::gcd(rows, a.npix) : 0;
    return (start + a.npix - 1) / rows + 1;
}

hipError_t net_conv(const NetConv &a, hipStream_t st) {
    if (a.M == 0) return hipSuccess;
    if (!net_conv_supported(a) || (a.pool && a.M > INT32_MAX - 256)) return hipErrorNotSupported;
    return conv_tiles(conv_tile(a, nullptr), a, nullptr, st);
}

hipError_t net_conv_pair(const NetConv &a, const NetConv &first, hipStream_t st) {
    if (a.M == 0) return hipSuccess;
    if (!net_conv_supported(a) || !net_conv_supported(first)) return hipErrorNotSupported;
    return conv_tiles(conv_tile(a, &first), a, &first, st);
}

hipError_t net_stem(const void *img, const void *w, const NetNorm &norm, void *out, int64_t N, int64_t H, int64_t W,
                    hipStream_t st) {
    if (H % 4 != 0 || W % 4 != 0 || H * W >= (1 << 27)) return hipErrorNotSupported;
    const int tx = (int)cdiv(W / 4, kPoolTile), ty = (int)cdiv(H / 4, kPoolTile);
    const int64_t tiles = N * tx * ty;
    if (tiles == 0) return hipSuccess;
    if (tiles > (1 << 30)) return hipErrorInvalidConfiguration;
    // (two workgroups per compute unit, each walking as many tiles as it takes)
    hipLaunchKernelGGL(k_net_stem, dim3((unsigned)std::min<int64_t>(tiles, 512)), dim3(kThreads), 0, st,
                       (const _Float16 *)img, (const _Float16 *)w, norm, (_Float16 *)out, (int)N, (int)H, (int)W, tx, ty);
    return hipGetLastError();
}

// Waves of the spatial branch at most: the weights a wave loads first are paid for once per walk.
constexpr int kMaxTapWaves = 8192;
// Several tiles at a time from this many waves on (us, one / several: 8 x 56 x 56 x 64, 392 waves,
// 5.7 / 7.5; 40 x 28 x 28 x 128, 980, 8.6 / 7.6).
constexpr int kManyTapWaves = 512;

// Which of the channel branch's device functions has these sizes (both would: the same one as in
// a launch of its own); its arguments but for the split over LDS.
int channel_kind(const NetChannel &c, int64_t N, int64_t H, int64_t W, int64_t C, ChannelMma *mma, ChannelRows<__half> *rows) {
    auto half = [](const void *p) { return static_cast<const __half *>(p); };
    auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const float scale = 1.f / (float)(H * W);
    *rows = {nullptr, half(c.w1), half(c.b1), half(c.w2), half(c.b2), (__half *)c.cf, (int)N, (int)C, (int)c.mid,
             (float)c.gain, half(c.gain_vec), half(c.offset_vec), c.parts, c.n_parts, scale, ChannelSave()};
    *mma = {nullptr, half(c.w1), half(c.b1), half(c.w2), half(c.b2), (__half *)c.cf, (int)N, (int)C, (int)c.mid,
            (float)c.gain, half(c.gain_vec), half(c.offset_vec), c.parts, c.n_parts, scale, ChannelSave()};
    if (!aligned(c.w1) || !aligned(c.w2) || !aligned(c.parts) || N > 65535) return kNoChannels;
    if (C >= 256 && channel_mma_covers(C, c.mid, 9)) return kChannelsMma;
    return C <= 128 && c.mid < kMmaStep ? kChannelsRows : kNoChannels;
}

// The spatial branch, and before it in the same launch the channel branch where `channel` is
// given and its kernels cover it; else in a launch of its own.
hipError_t net_branches(const void *x, const void *w, const void *bias, void *sf, double gain, const NetChannel *channel,
                        int64_t N, int64_t H, int64_t W, int64_t C, int stride, hipStream_t st) {
    if ((stride != 1 && stride != 2) || (stride == 2 && (H % 2 || W % 2)) || N * H * W >= (1ll << 31) - 256)
        return hipErrorNotSupported;
    const int64_t pixels = N * (H / stride) * (W / stride);
    const NetTaps taps{(const _Float16 *)x, (const _Float16 *)w, (const _Float16 *)bias, (_Float16 *)sf, (int)W,
                       (int)(W / stride), (int)((H / stride) * (W / stride)), (int)(H * W), (int)pixels,
                       (int)cdiv(pixels, 16), (float)gain,
                       Divisor::make((H / stride) * (W / stride), pixels), Divisor::make(W / stride, (H / stride) * (W / stride))};
    ChannelArgs<kChannelsMma> mma{};
    ChannelArgs<kChannelsRows> rows{};
    int kind = kNoChannels, blocks_x = 1, blocks = 0, lds = 0;
    if (channel) {
        kind = channel_kind(*channel, N, H, W, C, &mma.a, &rows.a);
        if (kind == kChannelsMma) {
            blocks_x = (int)(C / kMmaChannels);
            blocks = blocks_x * (int)cdiv(N, kMmaSamples);
            // (a channel block on every compute unit: half of the LDS, so that there is room for
            // spatial ones beside it.  128 x 7 x 7 x 512 16.1 -> 13.4 us, w1 by 48 rows.)
            mma.a.lds = channel_mma_lds(C, channel->mid, 9, blocks > 128 ? kMmaLds / 2 : kMmaLds);
            if (mma.a.lds.chunk == 0) mma.a.lds = channel_mma_lds(C, channel->mid, 9);
            lds = mma.a.lds.total;
        } else if (kind == kChannelsRows && channel_rows_plan(rows.a)) {
            blocks_x = (int)cdiv(C, rows.a.block);
            blocks = blocks_x * (int)N;
            lds = rows.a.total;
        } else {
            kind = kNoChannels;
            const ChannelRows<__half> &c = rows.a;
            const hipError_t err = channel_branch<__half>(nullptr, c.w1, c.b1, c.w2, c.b2, c.cf, N, C, c.mid, 3, c.gain,
                                                          c.gain_vec, c.offset_vec, st, c.parts, c.nparts, c.scale);
            if (err != hipSuccess) return err;
        }
    }
    bool done = false;
#define DDF_NET_BRANCHES(KS_, S_, U_, CH_, ARGS_)                                                                   \
    if (!done && C == KS_ * 32 && stride == S_ && kind == CH_ && (U_ == 1 || cdiv(taps.tiles, U_) >= kManyTapWaves)) { \
        constexpr int kWaves = branch_threads(CH_) / kWave;                                                         \
        const int64_t most = kMaxTapWaves / kWaves;                                                                 \
        const unsigned grid = (unsigned)(blocks + std::min(cdiv(cdiv(taps.tiles, U_), kWaves), most));              \
        hipLaunchKernelGGL((k_net_branches<KS_, S_, U_, CH_>), dim3(grid), dim3(branch_threads(CH_)), lds, st, taps, \
                           ARGS_, blocks_x, blocks);                                                                \
        done = true;                                                                                                \
    }
#define DDF_NET_BRANCHES_S(KS_, U_, CH_, ARGS_) \
    DDF_NET_BRANCHES(KS_, 1, U_, CH_, ARGS_) DDF_NET_BRANCHES(KS_, 2, U_, CH_, ARGS_)
    const ChannelArgs<kNoChannels> none{};
    DDF_NET_BRANCHES_S(2, 4, kChannelsRows, rows) DDF_NET_BRANCHES_S(2, 1, kChannelsRows, rows)
    DDF_NET_BRANCHES_S(4, 2, kChannelsRows, rows) DDF_NET_BRANCHES_S(4, 1, kChannelsRows, rows)
    DDF_NET_BRANCHES_S(8, 1, kChannelsMma, mma) DDF_NET_BRANCHES_S(16, 1, kChannelsMma, mma)
    DDF_NET_BRANCHES_S(2, 1, kNoChannels, none) DDF_NET_BRANCHES_S(4, 1, kNoChannels, none)
    DDF_NET_BRANCHES_S(8, 1, kNoChannels, none) DDF_NET_BRANCHES_S(16, 1, kNoChannels, none)
#undef DDF_NET_BRANCHES_S
#undef DDF_NET_BRANCHES
    return done ? hipGetLastError() : hipErrorNotSupported;
}

// The spatial branch alone, and the planes' sums.
hipError_t net_spatial(const void *x, const void *w, const void *bias, void *sf, float *parts, int *n_parts, int64_t N,
                       int64_t H, int64_t W, int64_t C, int stride, double gain, hipStream_t st) {
    if (N > 65535) return hipErrorNotSupported;
    const hipError_t err = net_branches(x, w, bias, sf, gain, nullptr, N, H, W, C, stride, st);
    if (err != hipSuccess) return err;
    *n_parts = 1;
    hipLaunchKernelGGL((k_net_pool<float>), dim3((unsigned)cdiv(C, 256), (unsigned)N), dim3(kThreads), 0, st,
                       (const _Float16 *)x, parts, (int)(H * W), (int)C);
    return hipGetLastError();
}

hipError_t net_filter(const void *x, const void *cf, const void *sf, const NetNorm &norm, void *out, int64_t N,
                      int64_t H, int64_t W, int64_t C, int stride, bool mul, hipStream_t st) {
    const int64_t Ho = H / stride, Wo = W / stride;
    if (N * Ho * Wo == 0) return hipSuccess;
    const int step = stride == 1 ? 4 : 6;
    if (C < 8 || C > kWave * 8) return hipErrorNotSupported;
    const int slots = (int)(kWave * 8 / C);
    // (32-bit offsets: as many samples at a time as stay below 2 GiB; a pixel is 16 bytes or more)
    const int64_t sample = H * W * C * 2, most = ((1ll << 31) - 16) / sample;
    if (most < 1) return hipErrorNotSupported;
    for (int64_t n0 = 0; n0 < N; n0 += most) {
        const int64_t cnt = std::min(most, N - n0);
        // The walk: whole rounds of the kernel's unrolled steps; the length that takes the
        // fewest steps over the rounds of resident waves it makes (three per SIMD), each walk
        // paying for its channel taps, its BatchNorm and two columns it does not produce.
        constexpr int kResident = 3072, kEntry = 6;
        int run = step;
        int64_t best = 0;
        for (int cand = step; ; cand += step) {
            const int64_t waves = cdiv(cnt * Ho * cdiv(Wo, cand), slots);
            const int64_t cost = cdiv(waves, kResident) * (cand + kEntry);
            if (best == 0 || cost < best) { best = cost; run = cand; }
            if (cand >= Wo) break;
        }
        const int64_t runs = cdiv(Wo, run);
        const int64_t units = cnt * Ho * runs, blocks = cdiv(units, slots * (kThreads / kWave));
        if (units > (1 << 30)) return hipErrorInvalidConfiguration;
        const _Float16 *xn = (const _Float16 *)x + n0 * H * W * C, *cn = (const _Float16 *)cf + n0 * C * 9,
                       *sn = (const _Float16 *)sf + n0 * Ho * Wo * kTapPitch;
        _Float16 *on = (_Float16 *)out + n0 * Ho * Wo * C;
        const bool wide = Wo % 2 != 0;    // (128 x 7 x 7 x 512 under BatchNorm 7.9 us packed, 8.6 wide)
        bool done = false;
#define DDF_NET_FILTER_LAUNCH(LP_, S_, MUL_, WIDE_)                                                         \
    hipLaunchKernelGGL((k_net_filter<LP_, S_, MUL_, WIDE_>), dim3(xcd_grid(blocks)), dim3(kThreads), 0, st, \
                       xn, cn, sn, norm, on, (int)H, (int)W, (int)Ho, (int)Wo, Divisor::make(runs, units),  \
                       Divisor::make(Ho, cnt * Ho), run, (int)units, (int)blocks, (uint32_t)(cnt * sample), (uint32_t)(cnt * Ho * Wo * C * 2),        \
                       (uint32_t)(cnt * Ho * Wo * kTapPitch * 2))
#define DDF_NET_FILTER(LP_, S_)                                     \
    if (C == LP_ * 8 && stride == S_) {                             \
        if (wide && mul) DDF_NET_FILTER_LAUNCH(LP_, S_, true, true); \
        else if (wide) DDF_NET_FILTER_LAUNCH(LP_, S_, false, true); \
        else if (mul) DDF_NET_FILTER_LAUNCH(LP_, S_, true, false);  \
        else DDF_NET_FILTER_LAUNCH(LP_, S_, false, false);          \
        done = true;                                                \
    }
        DDF_NET_FILTER(8, 1) DDF_NET_FILTER(16, 1) DDF_NET_FILTER(32, 1) DDF_NET_FILTER(64, 1)
        DDF_NET_FILTER(8, 2) DDF_NET_FILTER(16, 2) DDF_NET_FILTER(32, 2) DDF_NET_FILTER(64, 2)
#undef DDF_NET_FILTER
#undef DDF_NET_FILTER_LAUNCH
        if (!done) return hipErrorNotSupported;
    }
    return hipGetLastError();
}

// Both branches and the filter behind them: one launch where a compute unit has one workgroup of
// sixteen channels of some rows at most; else two.
hipError_t net_ddf(const void *x, const void *w, const void *bias, void *sf, double gain, const NetChannel &channel,
                   const NetNorm &norm, void *out, int64_t N, int64_t H, int64_t W, int64_t C, int stride, bool mul,
                   hipStream_t st) {
    const int64_t Ho = H / stride, Wo = W / stride;
    ChannelArgs<kChannelsMma> mma{};
    ChannelArgs<kChannelsRows> rows{};
    const int kind = channel_kind(channel, N, H, W, C, &mma.a, &rows.a);
    const int threads = branch_threads(kind);
    const int64_t groups = C / kMmaChannels, most = kFewBlocks / std::max<int64_t>(groups * N, 1);    // chunks of a sample
    const int64_t per = most > 0 ? cdiv(Ho, most) : Ho;
    const int64_t tile = (stride * (per - 1) + 3) * (W + 2) * 2, per_row = cdiv(2 * (W + 2), kWave);
    bool few = kind != kNoChannels && (stride == 1 || (stride == 2 && H % 2 == 0 && W % 2 == 0)) && most > 0 &&
               per * Wo <= kFewPixels && per_row * (stride * (per - 1) + 3) <= kFewItems * (threads / kWave) && H * W * C * 2 < (1ll << 31);
    if (few) {
        NetFew a{(const _Float16 *)x, (const _Float16 *)w, (const _Float16 *)bias, (_Float16 *)out, norm, (int)H, (int)W,
                 (int)Ho, (int)Wo, (int)per, (int)per_row, (uint32_t)cdiv(1 << 16, per_row), (uint32_t)cdiv(1 << 20, Wo),
                 (float)gain, kFewCf, 0, 0};
        const dim3 grid((unsigned)(groups * cdiv(Ho, per)), (unsigned)N);
        a.tile = mma_round(a.sf + per * Wo * kTapPitch * 2);
        a.channels = a.tile + (int)tile * 16;
        int lds = 0;
        if (kind == kChannelsMma) {
            mma.a.lds = channel_mma_lds(C, channel.mid, 9, kMmaLds - a.channels);
            few = mma.a.lds.chunk > 0;
            lds = a.channels + mma.a.lds.total;
        } else {
            few = channel_rows_lds(rows.a, kMmaChannels);
            lds = a.channels + rows.a.total;
        }
        few = few && lds <= kMmaLds;
        if (few) {
            const bool wide = Wo % 2 != 0;
            bool done = false;
#define DDF_NET_FEW_LAUNCH(KS_, S_, MUL_, WIDE_, CH_, ARGS_)                                                          \
    hipLaunchKernelGGL((k_net_filter_few<KS_, S_, MUL_, WIDE_, CH_>), grid, dim3(threads), lds, st, a, ARGS_)
#define DDF_NET_FEW(KS_, S_, CH_, ARGS_)                                         \
    if (C == KS_ * 32 && stride == S_) {                                         \
        if (wide && mul) DDF_NET_FEW_LAUNCH(KS_, S_, true, true, CH_, ARGS_);    \
        else if (wide) DDF_NET_FEW_LAUNCH(KS_, S_, false, true, CH_, ARGS_);     \
        else if (mul) DDF_NET_FEW_LAUNCH(KS_, S_, true, false, CH_, ARGS_);      \
        else DDF_NET_FEW_LAUNCH(KS_, S_, false, false, CH_, ARGS_);              \
        done = true;                                                             \
    }
            if (kind == kChannelsRows) {
                DDF_NET_FEW(2, 1, kChannelsRows, rows) DDF_NET_FEW(4, 1, kChannelsRows, rows)
                DDF_NET_FEW(2, 2, kChannelsRows, rows) DDF_NET_FEW(4, 2, kChannelsRows, rows)
            } else {
                DDF_NET_FEW(8, 1, kChannelsMma, mma) DDF_NET_FEW(16, 1, kChannelsMma, mma)
                DDF_NET_FEW(8, 2, kChannelsMma, mma) DDF_NET_FEW(16, 2, kChannelsMma, mma)
            }
#undef DDF_NET_FEW
#undef DDF_NET_FEW_LAUNCH
            if (done) return hipGetLastError();
        }
    }
    const hipError_t err = net_branches(x, w, bias, sf, gain, &channel, N, H, W, C, stride, st);
    return err == hipSuccess ? net_filter(x, channel.cf, sf, norm, out, N, H, W, C, stride, mul, st) : err;
}

hipError_t net_pool(const void *x, void *out, int64_t N, int64_t plane, int64_t C, hipStream_t st) {
    if (N * plane * C == 0) return hipSuccess;
    if (N > 65535 || C % 8 != 0) return hipErrorNotSupported;
    hipLaunchKernelGGL((k_net_pool<_Float16>), dim3((unsigned)cdiv(C, 256), (unsigned)N), dim3(kThreads), 0, st,
                       (const _Float16 *)x, (_Float16 *)out, (int)plane, (int)C);
    return hipGetLastError();
}

}  // namespace ddf

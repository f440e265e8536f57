// What the kernels of a network's inference share (ddf_net.hip, ddf_net_chain.hip).
#pragma once

#include "ddf_channel.h"
#include "ddf_common.h"
#include "ddf_rows.h"

namespace ddf {
namespace net {

typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t rows_u4 __attribute__((ext_vector_type(4)));
using rows::half2_t;

constexpr int kThreads = 256;
constexpr int kXcd = 8;

// Workgroups are handed to the XCDs round-robin: consecutive logical blocks share one.
__device__ __forceinline__ int xcd_block(int block, int blocks) {
    const int per = (blocks + kXcd - 1) / kXcd;
    return (block % kXcd) * per + block / kXcd;   // (may be >= blocks: nothing to do then)
}
inline unsigned xcd_grid(int64_t blocks) { return (unsigned)(cdiv(blocks, kXcd) * kXcd); }

// The tiles of a product, row by row; of a pair's first product, the pixels it samples.
struct TileCut {
    int tiles;
    Divisor tiles_n, npix, Wo;
};

// y = scale * x + shift of the convolution's bias and the BatchNorm behind it, for V
// consecutive channels: requested as vectors early, worked out where they are needed.  (Read
// channel by channel at the end of a kernel they cost more than small kernels do.)  A parameter that is not there is asked
// for behind a descriptor that holds nothing: no branches, which the loads behind them wait for.
template <int V>
struct Affine {
    typedef _Float16 vec __attribute__((ext_vector_type(V)));
    vec w, b, m, v, cb;
    // bias: the convolution's is part of it.
    __device__ __forceinline__ void request(const NetNorm &n, int c, bool bias = true) {
        auto get = [&](const void *p) __attribute__((always_inline)) {
            const __amdgpu_buffer_rsrc_t r = rows::plane_rsrc(p, p ? 0x7fffffffu : 0u);
            if constexpr (V == 1) {
                return __builtin_bit_cast(vec, (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, c * 2, 0, 0));
            } else {
                uint32_t q[V / 2];
                rows::load_words<V / 2>(r, (uint32_t)c * 2, q);
                return __builtin_bit_cast(vec, q);
            }
        };
        const bool bn = n.var;
        w = get(bn ? n.weight : nullptr);
        b = get(bn ? n.bias : nullptr);
        m = get(bn ? n.mean : nullptr);
        v = get(n.var);
        cb = get(bias ? n.conv_bias : nullptr);
    }
    __device__ __forceinline__ void finish(const NetNorm &n, float (&scale)[V], float (&shift)[V]) const {
        const bool bn = n.var;
        const float eps = bn ? n.eps : 1.f;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            scale[e] = (bn && n.weight ? (float)w[e] : 1.f) * rsqrtf((float)v[e] + eps);
            shift[e] = (float)b[e] + ((float)cb[e] - (float)m[e]) * scale[e];
        }
    }
};

// Lanes of the lower half of the wave: a over both halves; of the upper half: b.
__device__ __forceinline__ float add_swapped32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Lanes of even rows of sixteen: a over the row and the next; of odd rows: b over the row before, too.
__device__ __forceinline__ float add_swapped16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

constexpr int kTapPitch = 12;    // a pixel's spatial taps: nine and padding

// ---- spatial filter branch of sixteen pixels ------------------------------------------
// Pixels are the columns, the nine taps nine of the sixteen rows of 16x16x32 steps over the
// channels; both operands contiguous.  A pixel's taps end up on four lanes, which normalise them
// across the wave's rows; they are stored as (pixel, kTapPitch), nine taps and padding.

template <int KS>
struct TapWeights {
    static constexpr int KK = 9;
    half8_t w[KS];
    uint32_t b[4];
    // (rows past the ninth, and a bias that is not there, lie outside their buffers: zeros)
    __device__ __forceinline__ void request(const _Float16 *weight, const _Float16 *bias, int lane) {
        const int col = lane & 15, quad = lane >> 4;
        const __amdgpu_buffer_rsrc_t wr = rows::plane_rsrc(weight, KK * KS * 64), br = rows::plane_rsrc(bias, bias ? KK * 2 : 0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            w[ks] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(wr, col * KS * 64 + quad * 16, ks * 64, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = __builtin_amdgcn_raw_buffer_load_b16(br, (quad * 4 + e) * 2, 0, 0);
    }
    // The bias is converted behind this: the compiler has it done, and waited for, where it is asked for.
    __device__ __forceinline__ void hold() {
#pragma unroll
        for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(b[e]));
    }
    // v: channels ks * 32 + quad * 8 .. + 7 of the lane's pixel; `at`: where its taps go
    __device__ __forceinline__ void taps(const half8_t (&v)[KS], float gain, bool there, _Float16 *sf, int64_t at, int lane) const {
        const int quad = lane >> 4;
        float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[ks], v[ks], acc, 0, 0, 0);
        // taps 4 * quad + e of the pixel (rows past the ninth: zero weights, zero bias)
        float f[4], s = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f[e] = acc[e] + (float)__builtin_bit_cast(_Float16, (uint16_t)b[e]);
            s += f[e];
        }
        const float mean = rows_total(s) / (float)KK;
        float sq = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f[e] -= mean;
            if (quad * 4 + e < KK) sq = fmaf(f[e], f[e], sq);
        }
        const float inv = gain / (sqrtf(rows_total(sq) / (float)(KK - 1)) + 1e-10f);
        half4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float tap = f[e] * inv;
            asm volatile("" : "+v"(tap));    // (rounded to fp32 first in every instance)
            o[e] = (_Float16)tap;
        }
        if (there && quad < 3) *reinterpret_cast<half4_t *>(sf + at * kTapPitch + quad * 4) = o;
    }
};

// The dynamic filter of eight channels of a pixel (k_net_filter's comment has the reasons).
template <bool MUL, bool WIDE>
__device__ __forceinline__ void filter_pair(half2_t cv, half2_t sv, half2_t xv, float &a0, float &a1) {
    if constexpr (WIDE) {
        const float c0 = (float)cv[0], c1 = (float)cv[1], s0 = (float)sv[0], s1 = (float)sv[1];
        a0 = fmaf((float)xv[0], MUL ? c0 * s0 : c0 + s0, a0);
        a1 = fmaf((float)xv[1], MUL ? c1 * s1 : c1 + s1, a1);
    } else {
        const half2_t cb = MUL ? cv * sv : cv + sv;
        a0 = fmaf((float)xv[0], (float)cb[0], a0);
        a1 = fmaf((float)xv[1], (float)cb[1], a1);
    }
}

// The channel taps of eight channels: of filter rows 0 and 1 as a channel's pair, of row 2 as two channels'.
__device__ __forceinline__ void channel_taps(const _Float16 *cf, uint32_t (&cfa)[3][8], uint32_t (&cfb)[3][4]) {
    const uint4 *src = reinterpret_cast<const uint4 *>(cf);
    uint32_t wd[36];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const uint4 q = src[i];
        wd[4 * i] = q.x; wd[4 * i + 1] = q.y; wd[4 * i + 2] = q.z; wd[4 * i + 3] = q.w;
    }
    auto half_at = [&](int i) { return (i & 1) ? wd[i / 2] >> 16 : wd[i / 2] & 0xffffu; };
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
        for (int e = 0; e < 8; ++e) cfa[j][e] = half_at(9 * e + j) | (half_at(9 * e + 3 + j) << 16);
#pragma unroll
        for (int k = 0; k < 4; ++k) cfb[j][k] = half_at(18 * k + 6 + j) | (half_at(18 * k + 15 + j) << 16);
    }
}

// Rows 0 and 1 of a column as a channel's pair each, once for the three results it is under.
__device__ __forceinline__ void pair_column(uint32_t (&col)[3][4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t top = col[0][k], low = col[1][k];
        col[0][k] = __builtin_amdgcn_perm(low, top, 0x05040100);
        col[1][k] = __builtin_amdgcn_perm(low, top, 0x07060302);
    }
}

// The sums of a result from its three (paired) columns and the pixel's taps.
template <bool MUL, bool WIDE>
__device__ __forceinline__ void filter_sums(const uint32_t (&cfa)[3][8], const uint32_t (&cfb)[3][4], const uint32_t (&c0)[3][4],
                                            const uint32_t (&c1)[3][4], const uint32_t (&c2)[3][4], const uint32_t (&tp)[6],
                                            float (&acc)[8]) {
    // spatial taps j and 3 + j
    const uint32_t sa[3] = {__builtin_amdgcn_perm(tp[1], tp[0], 0x07060100), __builtin_amdgcn_perm(tp[2], tp[0], 0x05040302),
                            __builtin_amdgcn_perm(tp[2], tp[1], 0x07060100)};
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    // (all indices constants: a loop over j was unrolled too late in larger kernels, its taps went through memory)
    rows::static_for<0, 3>([&](auto column) __attribute__((always_inline)) {
        constexpr int j = decltype(column)::value;
        const uint32_t(&at)[3][4] = j == 0 ? c0 : j == 1 ? c1 : c2;
        const half2_t sp = __builtin_bit_cast(half2_t, sa[j]);
        const half2_t sb = __builtin_bit_cast(half2_t, tp[(6 + j) / 2]);
        const half2_t sv = {sb[j & 1], sb[j & 1]};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const half2_t xv = __builtin_bit_cast(half2_t, at[e & 1][e / 2]), cv = __builtin_bit_cast(half2_t, cfa[j][e]);
            if constexpr (WIDE) {
                const float f0 = (float)cv[0], f1 = (float)cv[1], s0 = (float)sp[0], s1 = (float)sp[1];
                acc[e] = fmaf((float)xv[0], MUL ? f0 * s0 : f0 + s0, acc[e]);
                acc[e] = fmaf((float)xv[1], MUL ? f1 * s1 : f1 + s1, acc[e]);
            } else {
                acc[e] = __builtin_amdgcn_fdot2(xv, MUL ? cv * sp : cv + sp, acc[e], false);
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            filter_pair<MUL, WIDE>(__builtin_bit_cast(half2_t, cfb[j][k]), sv, __builtin_bit_cast(half2_t, at[2][k]),
                                   acc[2 * k], acc[2 * k + 1]);
    });
}

// This wave's loads but the last N have arrived and its LDS reads are done; then all waves'.
template <int N>
__device__ __forceinline__ void arrive() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

}  // namespace net

// A convolution (two with `first`) in the tiles of ddf_net_small.hip: 16 x 16 or 32 x 32.
hipError_t net_conv_small(int rows, const NetConv &a, const NetConv *first, hipStream_t st);
}  // namespace ddf

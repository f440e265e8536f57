// What the kernels of a network's inference share (ddf_net.hip, ddf_net_chain.hip).
#pragma once

#include "ddf_channel.h"
#include "ddf_common.h"
#include "ddf_rows.h"

namespace ddf {
namespace net {

typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t rows_u4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kXcd = 8;

// Workgroups are handed to the XCDs round-robin: consecutive logical blocks share one.
__device__ __forceinline__ int xcd_block(int block, int blocks) {
    const int per = (blocks + kXcd - 1) / kXcd;
    return (block % kXcd) * per + block / kXcd;   // (may be >= blocks: nothing to do then)
}
inline unsigned xcd_grid(int64_t blocks) { return (unsigned)(cdiv(blocks, kXcd) * kXcd); }

// y = scale * x + shift of the convolution's bias and the BatchNorm behind it, for V
// consecutive channels: requested as vectors early, worked out where they are needed.  (Read
// channel by channel at the end of a kernel they cost more than small kernels do.)
template <int V>
struct Affine {
    typedef _Float16 vec __attribute__((ext_vector_type(V)));
    vec w, b, m, v, cb;
    // bias: the convolution's is part of it.
    __device__ __forceinline__ void request(const NetNorm &n, int c, bool bias = true) {
        auto get = [&](const void *p, _Float16 other) {
            vec r;
            if (p) __builtin_memcpy(&r, static_cast<const _Float16 *>(p) + c, sizeof(vec));
            else
#pragma unroll
                for (int e = 0; e < V; ++e) r[e] = other;
            return r;
        };
        w = get(n.var ? n.weight : nullptr, (_Float16)1);
        b = get(n.var ? n.bias : nullptr, (_Float16)0);
        m = get(n.var ? n.mean : nullptr, (_Float16)0);
        v = get(n.var, (_Float16)1);
        cb = get(bias ? n.conv_bias : nullptr, (_Float16)0);
    }
    __device__ __forceinline__ void finish(const NetNorm &n, float (&scale)[V], float (&shift)[V]) const {
        const float eps = n.var ? n.eps : 0.f;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            scale[e] = (float)w[e] * rsqrtf((float)v[e] + eps);
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

// This wave's loads but the last N have arrived and its LDS reads are done; then all waves'.
template <int N>
__device__ __forceinline__ void arrive() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

}  // namespace net
}  // namespace ddf

// Shared declarations of the DDF HIP library (gfx950 only, wave64).
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ddf_hip.h"

namespace ddf {

constexpr int kWave = 64;

// Problem description handed to every launcher.  Ho/Wo use floor division
// (ddf/ddf.py:56 of the reference), r is the tap radius in taps.
struct Problem {
    int64_t N, C, H, W, Ho, Wo;
    int k, d, s, r, kk;
    bool mul;
};

inline Problem make_problem(int64_t N, int64_t C, int64_t H, int64_t W, int k,
                            int d, int s, int combine) {
    Problem p;
    p.N = N; p.C = C; p.H = H; p.W = W;
    p.Ho = H / s; p.Wo = W / s;
    p.k = k; p.d = d; p.s = s; p.r = (k - 1) / 2; p.kk = k * k;
    p.mul = (combine == DDF_MUL);
    return p;
}

// Accumulator type: fp16 and fp32 storage accumulate in fp32, fp64 in fp64.
template <typename T> struct Acc { using type = float; };
template <> struct Acc<double> { using type = double; };

__device__ __forceinline__ float ld(const __half *p) { return __half2float(*p); }
__device__ __forceinline__ float ld(const float *p) { return *p; }
__device__ __forceinline__ double ld(const double *p) { return *p; }
__device__ __forceinline__ void st(__half *p, float v) { *p = __float2half(v); }
__device__ __forceinline__ void st(float *p, float v) { *p = v; }
__device__ __forceinline__ void st(double *p, double v) { *p = v; }

template <bool MUL, typename A>
__device__ __forceinline__ A comb(A a, A b) { return MUL ? a * b : a + b; }

// (NaN stays NaN, as torch's ReLU has it)
__device__ __forceinline__ float relu(float f) { return f < 0.f ? 0.f : f; }

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The spatial filter normalisation behind the spatial-filter gradient (FilterNorm
// of the spatial branch, ddf/ddf.py:146-157 of the reference: the operator's
// spatial filter is gain * standardised(raw) over the k*k taps of a pixel).  A
// backward pass that is handed one pushes dSF through the normalisation's
// Jacobian in the pass that adds up its partial sums and writes d_raw instead;
// `applied` tells the caller whether that happened (else dSF is complete where
// the pass was told to put it, and the caller runs filter_norm_backward).
template <typename T>
struct NormTail {
    const T *raw;          // (N, k*k, Ho, Wo), before the normalisation
    T *d_raw;              // gradient with respect to raw
    T *terms;              // nullable: dSF * standardised(raw), summed by the caller into the gain_vec gradient
    const T *gain_vec;     // nullable: (groups, k*k); sample n uses group n % groups
    int groups;
    double gain;           // used when gain_vec is null
    bool applied;
};

// Launchers.  Each returns a hipError_t from the launch (hipSuccess when the
// tensor is empty and nothing was launched).  `supported` queries tell the
// API layer whether the tiled family covers a problem.
template <typename T>
hipError_t generic_forward(const Problem &p, const T *x, const T *cf, const T *sf,
                           T *out, hipStream_t st);
template <typename T>
hipError_t generic_backward(const Problem &p, const T *go, const T *x, const T *cf,
                            const T *sf, T *dx, T *dcf, T *dsf, unsigned need,
                            hipStream_t st);

// y = gain * standardised(x) + offset over the `taps` axis of an
// (outer, groups, taps, inner) tensor; gain_vec / offset_vec are (groups, taps)
// or null (then the scalar `gain` / no offset).
template <typename T>
hipError_t filter_norm(const T *x, T *y, int64_t outer, int64_t groups, int taps, int64_t inner,
                       double gain, const T *gain_vec, const T *offset_vec, hipStream_t st);

// Gradient of filter_norm with respect to x; `terms` (nullable) receives
// dy * standardised(x), whose sum over (outer, inner) is the gain_vec gradient.
template <typename T>
hipError_t filter_norm_backward(const T *dy, const T *x, T *dx, T *terms, int64_t outer,
                                int64_t groups, int taps, int64_t inner, double gain,
                                const T *gain_vec, hipStream_t st);

// The filter branches of DDFPack, one launch each (ddf_branches.hip): 1x1
// convolution (stride as the operator's) + spatial filter normalisation, and
// bottleneck MLP on the pooled features + channel filter normalisation.
// hipErrorNotSupported: kernel size or sizes not covered, nothing launched.
bool branch_kernel_size_built(int k);
// What the channel branch leaves for its gradient (each may be null), fp32: the pooled
// vectors (N, C), the hidden vectors behind the ReLU (N, mid) and the taps in front of the
// normalisation (N, C * k*k), as the forward pass used them.
struct ChannelSave { float *pooled = nullptr, *hidden = nullptr, *taps = nullptr; };
// raw (may be null; with pool_part only): the taps in front of the normalisation.
template <typename T>
// pool_part (may be null): the launch also leaves the sums of the feature map over
// the pixels of each of *pool_parts parts of a plane, fp32, [(n * parts + p) * C + c]; at most
// pool_capacity floats.  hipErrorNotSupported where no kernel does that.
hipError_t spatial_branch(const T *x, const T *w, const T *bias, T *sf, int64_t N, int64_t C,
                          int64_t H, int64_t W, int head, int k, int stride, double gain,
                          const T *gain_vec, const T *offset_vec, hipStream_t st,
                          float *pool_part = nullptr, int64_t pool_capacity = 0,
                          int *pool_parts = nullptr, T *raw = nullptr);
// parts (may be null): the pooled vectors are scale * the sums of nparts such partial
// sums instead of `pooled`.
template <typename T>
hipError_t channel_branch(const T *pooled, const T *w1, const T *b1, const T *w2, const T *b2,
                          T *cf, int64_t N, int64_t C, int64_t mid, int k, double gain,
                          const T *gain_vec, const T *offset_vec, hipStream_t st,
                          const float *parts = nullptr, int nparts = 0, double scale = 1.0,
                          ChannelSave save = ChannelSave());
// Partial sums of the pooled vectors ([sample][part][channel]) to totals; more of them than the
// second says (3 x 3 taps) are better added up before the channel branch (channel_parts_left).
hipError_t collapse_parts(const float *parts, int nparts, float *totals, int64_t N, int64_t C, hipStream_t st);
int64_t parts_left(int64_t N, int64_t C, int64_t mid, int esz);

// Gradients of both branches (ddf_pack_backward.hip; 3 x 3 taps): from dcf and draw (the
// gradients of the channel filter and of the un-normalised spatial taps) and what the
// forward pass saved, to every parameter's gradient (dbs, db1, db2 and dgain may be null)
// and, unless dx is null, added to the operator's own feature gradient in dx.
template <typename T>
struct PackBackward {
    const T *x, *dcf, *draw;
    const float *pooled, *hidden, *taps;   // ChannelSave
    const T *ws, *w1, *w2, *gain_vec;      // gain_vec null: the scalar gain
    double gain;
    T *dx, *dws, *dbs, *dw1, *db1, *dw2, *db2, *dgain;
};
// (sizes both halves cover: the forward launches that save for it, and pack_backward)
bool pack_backward_supported(int64_t N, int64_t C, int64_t mid, int64_t H, int64_t W, int head, int k,
                             int stride, int dtype);
size_t pack_backward_workspace(int64_t N, int64_t C, int64_t mid, int64_t H, int64_t W, int head, int stride,
                               int dtype);
template <typename T>
hipError_t pack_backward(const PackBackward<T> &b, int64_t N, int64_t C, int64_t H, int64_t W, int64_t mid,
                         int head, int stride, void *ws, hipStream_t st);

#ifdef __HIPCC__
// A kernel's arguments, all in front of its first instruction: they are read from memory, and read where each is needed a
// launch of a few microseconds waits for them two or three times (0.2 us each).
template <typename A, typename B, typename C, typename D>
__device__ __forceinline__ void at_once(A a, B b, C c, D d) {
    asm volatile("" ::"s"(a), "s"(b), "s"(c), "s"(d));
}
template <typename A, typename B, typename C, typename D, typename... More>
__device__ __forceinline__ void at_once(A a, B b, C c, D d, More... more) {
    asm volatile("" ::"s"(a), "s"(b), "s"(c), "s"(d));
    at_once(more...);
}
#endif  // __HIPCC__

// Division by a number that the host knows: by a multiplication where that is exact (0: it is not).
struct Divisor {
    uint32_t by, magic;
    // of numbers below `most`
    static Divisor make(int64_t by, int64_t most) {
        return {(uint32_t)by, by > 1 && by * most < (1ll << 32) ? (uint32_t)(((1ull << 32) + by - 1) / by) : 0u};
    }
#ifdef __HIPCC__
    __device__ __forceinline__ uint32_t of(uint32_t n) const { return by == 1 ? n : magic ? __umulhi(n, magic) : n / by; }
#endif
};

// Channels-last fp16 kernels of the DDF-ResNets' inference (ddf_net.hip).
// The per-channel affine map behind a convolution: its bias and the BatchNorm (eval mode)
// that follows; null pointers: absent (var null: no BatchNorm).
struct NetNorm {
    const void *weight, *bias, *mean, *var, *conv_bias;
    float eps;
};
// out (M, N) = act(norm(x (rows of K) . w (N, K)) + res (M, N)); stride > 1: row m of x is the
// pixel of an (n, H, W) batch that result m = (n, y, x) of npix = Ho * Wo samples.
struct NetConv {
    const void *x, *w, *res;
    void *out;
    NetNorm norm;
    int64_t M;
    int N, K, relu, stride, H, W, Wo, npix;
    // nullable: also the results' sums over the pixels of each sample, fp32, in parts:
    // [(sample * pool_slots + slot) * N + channel]
    float *pool;
    int pool_slots;
};
bool net_conv_supported(const NetConv &a);
int net_conv_pool_slots(const NetConv &a);    // as many as the launch leaves
hipError_t net_conv(const NetConv &a, hipStream_t st);
// act(affine(a) + affine'(first)): same pixels and channels, activation and output a's
hipError_t net_conv_pair(const NetConv &a, const NetConv &first, hipStream_t st);
// out (M, N) = relu(norm(x (M, K) . w (N, K)) + res), with side_K > 0 relu(norm(..) + side_norm(side (M, side_K)
// . side_w (N, side_K))); next (M, N2) = relu(norm2(out . w2 (N2, N))) and its sums over the pixels of
// each sample (npix), in net_chain_pool_slots parts.  With cf, x holds the features of images W wide and what is
// multiplied is relu(filter_norm(the operator)) with the filters cf and the spatial branch's (tap_w, tap_bias,
// tap_gain), as net_branches and net_filter make it.
struct NetChain {
    const void *x, *w, *res, *side, *side_w, *w2;
    void *out, *next;
    float *pool;
    NetNorm norm, side_norm, norm2;
    int64_t M;
    int K, side_K, N, N2, npix;
    const void *cf, *tap_w, *tap_bias;
    float tap_gain;
    NetNorm filter_norm;
    int W, mul;
    // net_chain's own
    int tiles, pool_slots;
    Divisor row, rows;        // pixels of a row, rows of an image
};
bool net_chain_covers(int64_t M, int64_t K, int64_t side_K, int64_t N, int64_t N2);
// whether the spatial branch and the filter are made in front of it by the same launch
bool net_chain_filters(int64_t W, int64_t K);
int net_chain_pool_slots(int64_t M, int npix);
hipError_t net_chain(NetChain a, hipStream_t st);
hipError_t net_stem(const void *img, const void *w, const NetNorm &norm, void *out, int64_t N, int64_t H, int64_t W,
                    hipStream_t st);
// Both filter branches (channel null: the spatial one), the channel one from the pooled vectors'
// partial sums.
struct NetChannel {
    const float *parts;
    int n_parts;
    const void *w1, *b1, *w2, *b2, *gain_vec, *offset_vec;
    void *cf;
    int64_t mid;
    double gain;
};
hipError_t net_branches(const void *x, const void *w, const void *bias, void *sf, double gain, const NetChannel *channel,
                        int64_t N, int64_t H, int64_t W, int64_t C, int stride, hipStream_t st);
hipError_t net_spatial(const void *x, const void *w, const void *bias, void *sf, float *parts, int *n_parts, int64_t N,
                       int64_t H, int64_t W, int64_t C, int stride, double gain, hipStream_t st);
hipError_t net_filter(const void *x, const void *cf, const void *sf, const NetNorm &norm, void *out, int64_t N,
                      int64_t H, int64_t W, int64_t C, int stride, bool mul, hipStream_t st);
hipError_t net_ddf(const void *x, const void *w, const void *bias, void *sf, double gain, const NetChannel &channel,
                   const NetNorm &norm, void *out, int64_t N, int64_t H, int64_t W, int64_t C, int stride, bool mul,
                   hipStream_t st);
hipError_t net_pool(const void *x, void *out, int64_t N, int64_t plane, int64_t C, hipStream_t st);

// All scale*scale sub-pixel branches of an up-sampling DDF in one launch,
// written into the pixel-shuffled (N, C, H*scale, W*scale) result; cf / sf are
// host arrays of scale*scale device pointers.
bool up_forward_supported(int64_t H, int64_t W, int k, int d, int scale);
template <typename T>
hipError_t up_forward(int64_t N, int64_t C, int64_t H, int64_t W, int k, int d, int scale,
                      bool mul, const T *x, const void *const *cf, const void *const *sf, T *out,
                      hipStream_t st);

// What a filter-gradient launch leaves in its workspace where the caller adds it up itself: partial sums
// of dSF over csplit channel splits, of dCF over nstrips strips (null: the result is complete).
template <typename T>
struct FilterParts {
    const typename Acc<T>::type *sf = nullptr, *cf = nullptr;
    int csplit = 1, nstrips = 1;
};

// Helpers of the up-sampling backward: the gradient of the pixel shuffle (dO
// split into its scale*scale sub-pixel lattices, stored back to back) and, with cf_all, the branches'
// filters copied back to back (cf / sf: host arrays of device pointers); the
// sum of `parts` equally sized tensors stored back to back.
template <typename T>
hipError_t up_prepare(const T *go, T *lat, int64_t planes, int64_t H, int64_t W, int scale, const void *const *cf,
                      const void *const *sf, T *cf_all, T *sf_all, int64_t n_cf, int64_t n_sf, hipStream_t st);
template <typename T>
hipError_t up_sum_parts(const T *in, T *out, int64_t count, int parts, hipStream_t st);
// After the backward pass of all branches as one batch: dX summed from the branches' parts (parts may be
// null), and the batch's filter gradients (complete where `left` names no partial sums of them) to
// the branches' tensors (null destinations are skipped; dcf_all / dsf_all null: not asked for).
template <typename T>
hipError_t up_finish(const T *parts, T *dx, int64_t n_x, int branches, const T *dcf_all, const T *dsf_all,
                     const FilterParts<T> &left, void *const *dcfs, void *const *dsfs, int64_t N, int64_t C, int64_t kk,
                     int64_t plane, hipStream_t st);

// Tiny planes (H*W <= 64), 3x3, stride 1: forward (backward = false: x -> out)
// and feature gradient (backward = true: dO -> dX), G = 256 / (H*W) channel
// planes per workgroup pass.
bool small_supported(const Problem &p);
template <typename T>
hipError_t small_launch(const Problem &p, bool backward, const T *x, const T *cf, const T *sf,
                        T *out, hipStream_t st);

// Row-register kernels (stride 1; rows that are a whole number of vectors):
// forward (backward = false: x -> out) or feature gradient (backward = true:
// dO -> dX).  hipErrorNotSupported when the family does not cover the problem
// or a pointer is not aligned to its vectors; nothing was launched then.
template <typename T>
hipError_t rows_launch(const Problem &p, bool backward, const T *x, const T *cf, const T *sf,
                       T *out, hipStream_t st);

// Filter gradients (dCF, dSF) on the row-register kernel; same conventions.
// With dx != nullptr the launch also writes the feature gradient (the whole
// backward pass in one kernel, 3x3 without dilation).  The workspace
// (rows_filters_workspace bytes, 256-byte aligned) holds the partial sums over
// channel splits and strips.
size_t rows_filters_workspace(const Problem &p, int dtype, unsigned need);
// The row-register kernels cover the feature gradient and, in a launch of its
// own, the filter gradients of this problem (pointer alignment assumed).
bool rows_cover_backward(const Problem &p, int dtype);
// Stride 2: the row-register kernels cover the filter gradients.
bool rows_cover_stride2_filters(const Problem &p, int dtype);
// x_mod != 0: the batch p.N is several groups of x_mod samples sharing one set
// of features x (x_mod samples long); everything else is indexed by the sample.
// left != null: partial sums are not added up but named there.
template <typename T>
hipError_t rows_filters_launch(const Problem &p, const T *go, const T *x, const T *cf, const T *sf,
                               T *dx, T *dcf, T *dsf, void *ws, unsigned need, hipStream_t st,
                               int x_mod = 0, NormTail<T> *norm = nullptr, FilterParts<T> *left = nullptr);
// The whole backward pass of such a batch on the row-register kernels, or
// hipErrorNotSupported before anything is launched (shape or alignment not
// covered).  `ws`: rows_filters_workspace(p) bytes.
template <typename T>
hipError_t rows_backward_shared_features(const Problem &p, int x_mod, const T *go, const T *x,
                                         const T *cf, const T *sf, T *dx, T *dcf, T *dsf, void *ws,
                                         unsigned need, hipStream_t st, FilterParts<T> *left);

// Names of the kernels a forward / backward call on the tiled families would
// launch, written into buf (at most len bytes); returns snprintf's count.
int describe_forward(const Problem &p, int dtype, char *buf, int len);
int describe_backward(const Problem &p, int dtype, unsigned need, char *buf, int len);

bool tiled_forward_supported(const Problem &p, int dtype);
template <typename T>
hipError_t tiled_forward(const Problem &p, const T *x, const T *cf, const T *sf,
                         T *out, hipStream_t st);

bool tiled_backward_supported(const Problem &p, int dtype);
size_t tiled_backward_workspace(const Problem &p, int dtype, unsigned need);
template <typename T>
hipError_t tiled_backward(const Problem &p, const T *go, const T *x, const T *cf,
                          const T *sf, T *dx, T *dcf, T *dsf, void *ws,
                          unsigned need, hipStream_t st, NormTail<T> *norm = nullptr);

}  // namespace ddf

// Filter gradients with the tap rows dealt out to waves (gfx950, stride 1):
// same lane layout as ddf_rows.h.
//
// K consecutive work items walk the same channels of the same strip of the
// same sample; item i handles the K taps of filter row i.  For those a wave
// needs one feature row per result row only (the one (i - K/2) * D rows away),
// K spatial taps per pixel and K accumulators per pixel, so a 5 x 5 filter
// costs a wave the registers of five taps, not of twenty-five.  The waves
// share nothing: each stores the dSF planes of its own taps and parks its own
// dCF partials in its own LDS rows, which one lane per (channel, tap) then adds
// up (see ddf_rows_filters.h).  No workgroup barrier, no atomics.  A workgroup
// is g.wpb such independent waves, one per SIMD (the K of a pixel strip mostly
// share a compute unit and its L1, where they read the same dO rows).
// Partial sums over channel splits (dSF) and strips (dCF) go to the workspace.
// Reference kernels computing the same sums:
// ddf/src/cuda/ddf_mul_cuda_kernel.cu:293-355 (spatial filter), :358-420
// (channel filter).
#pragma once

#include "ddf_rows_filters.h"

namespace ddf {
namespace rows {

// Channels whose dCF partials are parked before one lane per (channel, tap of
// the wave's row) adds them up: as many as 64 lanes serve, a power of two.
template <int K>
constexpr int taprow_flush_channels() { return K <= 4 ? 16 : 8; }

constexpr int kTaprowWaves = 4;   // independent waves per workgroup

template <int K>
constexpr int taprow_lds_bytes(int asz) {
    return kTaprowWaves * taprow_flush_channels<K>() * K * kRedPitch * asz;
}

// What k_rows_taprow_backward is built for, X(D, VXF, VX, PAD, TAIL): the one list that its plan and its launcher go by.
// (Taps two apart reach two pixels into a lane's neighbours: no vectors of two.  TAIL 2: an odd tail of fp16.)
#define DDF_BACKWARD5_EXACT(X, D, VXF, VX) X(D, VXF, VX, false, 0) X(D, VXF, VX, true, 0)
#define DDF_BACKWARD5_BOTH_TYPES(X)                                                             \
    DDF_BACKWARD5_EXACT(X, 1, 2, 4) DDF_BACKWARD5_EXACT(X, 1, 4, 4) DDF_BACKWARD5_EXACT(X, 2, 4, 4) \
    X(1, 4, 4, true, 1) X(2, 4, 4, true, 1)
#define DDF_BACKWARD5_F16(X)                                                                    \
    X(1, 4, 4, true, 2) X(2, 4, 4, true, 2)                                                     \
    DDF_BACKWARD5_EXACT(X, 1, 4, 8) DDF_BACKWARD5_EXACT(X, 2, 4, 8)                             \
    DDF_BACKWARD5_EXACT(X, 1, 8, 8) DDF_BACKWARD5_EXACT(X, 2, 8, 8)                             \
    X(1, 8, 8, true, 1) X(2, 8, 8, true, 1) X(1, 8, 8, true, 2) X(2, 8, 8, true, 2)

inline int taprow_backward_tail(const RowsGeom &g) { return g.tail == 0 ? 0 : g.shift ? 2 : 1; }
inline bool taprow_backward_pad(const RowsGeom &g) { return g.tail > 0 || rows_shift_in_as_is(g); }
inline bool taprow_backward_built(int esz, int d, int vxf, int vx, bool pad, int tail) {
#define DDF_BACKWARD5_IS(D_, VXF_, VX_, PAD_, TAIL_) || (d == D_ && vxf == VXF_ && vx == VX_ && pad == PAD_ && tail == TAIL_)
    return (false DDF_BACKWARD5_BOTH_TYPES(DDF_BACKWARD5_IS)) || (esz == 2 && (false DDF_BACKWARD5_F16(DDF_BACKWARD5_IS)));
#undef DDF_BACKWARD5_IS
}

#ifdef __HIPCC__

template <typename T, int K, int D, bool MUL, int VX, int R, bool PAD, int NST, int TAIL = 0>
__device__ __forceinline__ void taprow_walk(
    const RowsGeom &g, int block, const T *__restrict__ go, const T *__restrict__ x, const T *__restrict__ cf,
    const T *__restrict__ sf, T *__restrict__ dcf, T *__restrict__ dsf,
    typename Acc<T>::type *__restrict__ ws_sf, typename Acc<T>::type *__restrict__ ws_cf,
    unsigned need, int x_mod) {
    using A = typename Acc<T>::type;
    constexpr int KK = K * K, RAD = K / 2, HX = RAD * D;
    constexpr int NW = VX * sizeof(T) / 4;
    constexpr int G = taprow_flush_channels<K>();
    using Row = ExtRow<T, VX, HX, PAD>;
    static_assert(G * K <= kWave, "one lane per (channel, tap) of a flush group");
    extern __shared__ __align__(16) unsigned char smem[];

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int item = Work::item_of(g, block, wave);
    if (item < 0) return;
    const int trow = item % K;   // filter row of this wave
    Work wk;
    wk.decode(g, item / K);
    const bool want_cf = need & DDF_NEED_DCF, want_sf = need & DDF_NEED_DSF;
    const int c0 = wk.c_begin;
    const int nch = wk.c_end - c0;
    const int64_t plane = (int64_t)g.H * g.W;
    const uint32_t plane_bytes = (uint32_t)plane * (uint32_t)sizeof(T);
    Lane<R, 0, VX, (TAIL > 0)> ln;
    ln.init(g, wk.strip, lane, (trow - RAD) * D);
    static_assert(TAIL == 0 || PAD, "ragged rows: padded");
    Ragged<T, VX, TAIL> rag;
    rag.init(g, ln.ragged);

    const int64_t xn = x_mod ? wk.n % x_mod : wk.n;   // (see k_rows_filters)
    const T *xs = x + (xn * g.C + c0) * plane;
    const T *gs = go + (wk.n * g.C + c0) * plane;
    uint32_t xb[R], ob[R], lob[R];   // (lob: where the lane's own vectors are loaded)
#pragma unroll
    for (int r = 0; r < R; ++r) {
        xb[r] = ln.xoff[r] < 0 ? kOutside : (uint32_t)ln.xoff[r] * (uint32_t)sizeof(T);
        ob[r] = ln.ooff[r] < 0 ? kOutside : (uint32_t)ln.ooff[r] * (uint32_t)sizeof(T);
        lob[r] = rag.load_at(ob[r]);
    }
    const int tl = lane < K ? lane : K - 1;
    const T *cfs = cf + (wk.n * g.C + c0) * KK + trow * K;   // the wave's K taps of a channel

    // Feature rows, dO rows and channel taps of channel ci, stage ST.  A channel
    // past the last one reads zeros (empty descriptors) and so adds nothing.
    constexpr bool kScalarTaps = sizeof(T) >= 4;   // (see k_rows)
    uint32_t xw[NST][R][NW], gw[NST][R][NW];
    T cfl[NST];
    A cfu[NST][kScalarTaps && MUL ? K : 1];
    // One descriptor per tensor for the whole walk: channel ci is reached through the
    // uniform offset ci * plane_bytes, the per-lane offset stays inside one plane.
    // spatial taps of the lane's pixels (needed for dCF under 'mul' only)
    uint32_t sfw[MUL ? R : 1][K][NW];
    if constexpr (MUL) {
        const T *sfn = sf + (wk.n * KK + trow * K) * plane;
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const __amdgpu_buffer_rsrc_t sr = plane_rsrc(sfn + j * plane, plane_bytes);
#pragma unroll
            for (int r = 0; r < R; ++r) load_words<NW>(sr, lob[r], sfw[r][j]);
        }
    }
    // A channel past the last one gets an empty descriptor: it reads zeros and so
    // adds nothing.  (Channels are issued in order: xs and gs run ahead plane by plane.)
    auto issue = [&](auto st_tag, int ci) __attribute__((always_inline)) {
        constexpr int ST = decltype(st_tag)::value;
        const bool live = ci < nch;
        const uint32_t bytes = live ? plane_bytes : 0u;
        const __amdgpu_buffer_rsrc_t pr = plane_rsrc(xs, bytes);
        const __amdgpu_buffer_rsrc_t gr = plane_rsrc(gs, bytes);
        xs += plane;
        gs += plane;
#pragma unroll
        for (int r = 0; r < R; ++r) load_words<NW>(pr, xb[r], xw[ST][r]);
#pragma unroll
        for (int r = 0; r < R; ++r) load_words<NW>(gr, lob[r], gw[ST][r]);
        if constexpr (MUL) {
            const int cc = live ? ci : nch - 1;
            if constexpr (kScalarTaps) {
#pragma unroll
                for (int j = 0; j < K; ++j) cfu[ST][j] = cfs[(int64_t)cc * KK + j];
            } else {
                cfl[ST] = cfs[(int64_t)cc * KK + tl];
            }
        }
    };
    static_for<0, NST - 1>([&](auto s) { issue(s, decltype(s)::value); });
    if constexpr (MUL) {
        // The taps were requested before the first channels: wait for them here, not
        // inside the walk (a wait there would drain the channel pipeline every round).
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int j = 0; j < K; ++j)
#pragma unroll
                for (int k = 0; k < NW; ++k) asm volatile("" : "+v"(sfw[r][j][k]));
        if constexpr (TAIL) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int j = 0; j < K; ++j) rag.fix(sfw[r][j]);
        }
    }

    A acc_sf[R][K][VX];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < K; ++j)
#pragma unroll
            for (int e = 0; e < VX; ++e) acc_sf[r][j][e] = 0;
    A *red = reinterpret_cast<A *>(smem) + (size_t)wave * (G * K * kRedPitch);

    // Where the dCF sums of the walk go: the wave's channels of dCF itself, or (more
    // than one strip per plane) of the per-strip partial sums.  Lane slot * K + j
    // serves tap j of the wave's row for channel `slot` of a flush group.
    const bool cf_direct = g.nstrips == 1;
    const uint32_t cf_pitch = cf_direct ? KK * (uint32_t)sizeof(T)                   // bytes per channel
                                        : (uint32_t)g.nstrips * KK * (uint32_t)sizeof(A);
    const __amdgpu_buffer_rsrc_t cf_out =
        cf_direct ? plane_rsrc(dcf + (wk.n * g.C + c0) * KK, (uint32_t)nch * cf_pitch)
                  : plane_rsrc(ws_cf + ((wk.n * g.C + c0) * g.nstrips + wk.strip) * KK,
                               // (the last channel's row ends with this strip's taps)
                               (uint32_t)(nch - 1) * cf_pitch + KK * (uint32_t)sizeof(A));
    const int fl_slot = lane / K, fl_tap = trow * K + (lane - fl_slot * K);
    const uint32_t cf_lane = (uint32_t)fl_slot * cf_pitch +
                             (uint32_t)fl_tap * (cf_direct ? (uint32_t)sizeof(T) : (uint32_t)sizeof(A));

    // Adds up the 64 lane partials of each (channel, tap) of a flush group of
    // `cnt` channels starting at channel `cbase` of the walk, and stores them.
    auto flush = [&](int cbase, int cnt) __attribute__((always_inline)) {
        wave_sync();
        if (lane < cnt * K) {
            const A *rowp = red + lane * kRedPitch;
            A tot[4] = {0, 0, 0, 0};
#pragma nounroll
            for (int k0 = 0; k0 < kWave / 4; k0 += 4) {
                typedef A vec4 __attribute__((ext_vector_type(4)));
                vec4 v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const vec4 *>(rowp + 4 * (k0 + k));
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int q = 0; q < 4; ++q) tot[q] += v[k][q];
            }
            const A sum = (tot[0] + tot[1]) + (tot[2] + tot[3]);
            if (cf_direct) store_value<T>(cf_out, cf_lane + (uint32_t)cbase * cf_pitch, sum);
            else store_value<A>(cf_out, cf_lane + (uint32_t)cbase * cf_pitch, sum);
        }
        wave_sync();
    };

    auto compute = [&](auto st_tag, auto slot_tag) __attribute__((always_inline)) {
        constexpr int ST = decltype(st_tag)::value, SLOT = decltype(slot_tag)::value;
        if constexpr (sizeof(T) == 2 && MUL) {
            // keep the packed taps packed (see k_rows)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int j = 0; j < K; ++j)
#pragma unroll
                    for (int k = 0; k < NW; ++k) asm volatile("" : "+v"(sfw[r][j][k]));
        }
        Row row[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int k = 0; k < NW; ++k) row[r].own[k] = xw[ST][r][k];
            if constexpr (TAIL) {
                rag.fix(row[r].own);
                rag.fix(gw[ST][r]);
            }
            row[r].sides(ln.first, ln.last);
        }
        A w[K];
        if constexpr (MUL) {
            if constexpr (kScalarTaps) {
#pragma unroll
                for (int j = 0; j < K; ++j) w[j] = cfu[ST][j];
            } else {
                const A cfa = (A)ld(&cfl[ST]);
#pragma unroll
                for (int j = 0; j < K; ++j) w[j] = lane_broadcast<A>(cfa, j);
            }
        }
        A pcf[K];
#pragma unroll
        for (int j = 0; j < K; ++j) pcf[j] = 0;
#pragma unroll
        for (int j = 0; j < K; ++j)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int e = 0; e < VX; ++e) {
                    const A gv = elem<T>(gw[ST][r], e), xv = row[r].at(e + j * D - HX);
                    if constexpr (MUL) {
                        const A gx = gv * xv;
                        acc_sf[r][j][e] = fma_(gx, w[j], acc_sf[r][j][e]);
                        pcf[j] = fma_(gx, elem<T>(sfw[r][j], e), pcf[j]);
                    } else {
                        // (two multiply-adds instead of a product and two additions)
                        acc_sf[r][j][e] = fma_(gv, xv, acc_sf[r][j][e]);
                        pcf[j] = fma_(gv, xv, pcf[j]);
                    }
                }
        // The accumulators are not read before the walk ends: without this the compiler
        // moves every update behind the flush branch and keeps (spills) the products.
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int j = 0; j < K; ++j)
#pragma unroll
                for (int e = 0; e < VX; ++e) asm volatile("" : "+v"(acc_sf[r][j][e]));
        // (a channel past the last one parks zeros; the flush does not read them)
#pragma unroll
        for (int j = 0; j < K; ++j) red[(SLOT * K + j) * kRedPitch + lane] = pcf[j];
    };

    // Groups of G channels, G a multiple of NST: the pipeline stage and the LDS
    // slot of every step are constants.  The walk covers whole groups; channels
    // past the last one read zeros.
    static_assert(G % NST == 0, "flush groups are whole pipeline rounds");
    for (int cb = 0; cb < nch; cb += G) {
        static_for<0, G>([&](auto s) {
            constexpr int S = decltype(s)::value;
            issue(std::integral_constant<int, (S + NST - 1) % NST>{}, cb + S + NST - 1);
            compute(std::integral_constant<int, S % NST>{}, s);
            // (one step at a time: interleaving the unrolled steps costs more registers
            // than the walk has)
            __builtin_amdgcn_sched_barrier(0);
        });
        if (want_cf) flush(cb, min(G, nch - cb));
    }

    if (!want_sf) return;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const int64_t t = trow * K + j;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (g.csplit == 1) {
                uint32_t ow[NW];
                pack<T, VX, A>(acc_sf[r][j], ow);
                rag.store(plane_rsrc(dsf + (wk.n * KK + t) * plane, plane_bytes), ob[r], ow);
            } else {
                // partial sums in the accumulator type, same plane shape
                constexpr int AW = VX * sizeof(A) / 4;
                constexpr int CH = AW < 4 ? AW : 4;
                const __amdgpu_buffer_rsrc_t wr =
                    plane_rsrc(ws_sf + ((wk.n * g.csplit + wk.cs) * KK + t) * plane,
                               (uint32_t)plane * (uint32_t)sizeof(A));
                const uint32_t off_a = ob[r] == kOutside ? kOutside
                                                         : ob[r] / (uint32_t)sizeof(T) * (uint32_t)sizeof(A);
                uint32_t aw[AW];
                pack<A, VX, A>(acc_sf[r][j], aw);
                if constexpr (TAIL) {
                    // (value by value: the last lane of a row has fewer)
#pragma unroll
                    for (int h = 0; h < AW; ++h) {
                        const uint32_t one[1] = {aw[h]};
                        store_words_nt<1>(wr, off_a == kOutside || (rag.last && h >= rag.tail) ? kOutside : off_a + h * 4,
                                          one);
                    }
                } else {
#pragma unroll
                    for (int h = 0; h < AW; h += CH) {
                        uint32_t part[CH];
#pragma unroll
                        for (int q = 0; q < CH; ++q) part[q] = aw[h + q];
                        store_words_nt<CH>(wr, off_a + h * 4, part);
                    }
                }
            }
        }
    }
}

template <typename T, int K, int D, bool MUL, int VX, int R, bool PAD, int NST, int WPE, int TAIL = 0>
__global__ __launch_bounds__(kWave * kTaprowWaves, WPE) void k_rows_taprow_filters(
    RowsGeom g, const T *__restrict__ go, const T *__restrict__ x, const T *__restrict__ cf,
    const T *__restrict__ sf, T *__restrict__ dcf, T *__restrict__ dsf,
    typename Acc<T>::type *__restrict__ ws_sf, typename Acc<T>::type *__restrict__ ws_cf,
    unsigned need, int x_mod) {
    taprow_walk<T, K, D, MUL, VX, R, PAD, NST, TAIL>(g, blockIdx.x, go, x, cf, sf, dcf, dsf, ws_sf, ws_cf, need, x_mod);
}

// All gradients in one launch: workgroups of filter gradients in front of those of the feature gradient (k_rows' walk,
// regrouped into as many waves).  The filter gradients are K waves per strip and sample, two and a fraction per SIMD: those with
// three of them keep their vector ALU busy to the end, the others idle for the last third, and the feature gradient, bound by the vector ALU as
// well, begins behind that.  Here its workgroups take the places that are left.  Kernel times of a whole step, us, two launches /
// this: fp32 32 x 128 x 56 x 56 taps two apart 133.9 / 108.3 (the gradients 102 / 77), one apart 128.6 / 105.6, 8 x 256 x 28 x 28 39.0 / 29.2, 3 x 256 x 100
// x 104 84.4 / 73.1, 5 x 33 x 200 x 190 81.7 / 73.0, 2 x 64 x 40 x 52 25.1 / 19.1; fp16 32 x 128 x 56 x 56 131.8 / 108.7, 'add' 107.8 / 91.0, 8 x 64 x 200
// x 200 184.9 / 179.6, 21 x 104 x 57 x 61 114.8 / 106.0, 1 x 512 x 50 x 75 51.1 / 41.3.  The gradients and their sums alone, even tails of
// fp16: 13 x 120 x 34 x 34 taps two apart 33.6 / 28.4, 6 x 76 x 9 x 66 20.8 / 13.9, 4 x 256 x 50 x 74 49.5 / 40.2, 16 x 64 x 90 x 90 65.6 / 55.4.  No size
// was found where two are faster.  Two remain for one half on its own, for operands that are not aligned to dX's vectors, and where the halves'
// layouts have no instance here in common (an eighth of fp16's sizes, a sixteenth of fp32's): filter gradients in vectors a quarter as long or half
// as long as ragged ones, or one half as a run, in segments or with idle lanes between rows and the other not.
template <typename T, int D, bool MUL, int VXF, int VX, bool PAD, int NST, int WPE, int TAIL>
__global__ __launch_bounds__(kWave * kTaprowWaves, WPE) void k_rows_taprow_backward(
    RowsGeom g, RowsGeom gx, int blocks, const T *__restrict__ go, const T *__restrict__ x, const T *__restrict__ cf,
    const T *__restrict__ sf, T *__restrict__ dx, T *__restrict__ dcf, T *__restrict__ dsf,
    typename Acc<T>::type *__restrict__ ws_sf, typename Acc<T>::type *__restrict__ ws_cf, unsigned need) {
    const int block = blockIdx.x;
    if (block < blocks) taprow_walk<T, 5, D, MUL, VXF, 1, PAD, NST, TAIL>(g, block, go, x, cf, sf, dcf, dsf, ws_sf, ws_cf, need, 0);
    else rows_walk<T, 5, D, MUL, true, VX, 1, PAD, 2, WPE, 1, TAIL>(gx, block - blocks, go, cf, sf, dx);
}

#endif  // __HIPCC__

}  // namespace rows

// Host-side geometry of k_rows_taprow_filters (ddf_rows_host.hip): a work item
// is a wave handling one filter row of one (sample, strip, channel range);
// g->nwork counts all K of each, g->csplit the ranges of g->cpb = g->cpw channels.
bool rows_taprow_geometry(const Problem &p, int dtype, RowsGeom *g, int *vx, int *r);
// What runs: that geometry or the one for ragged rows (see rows_plan).
bool rows_taprow_plan(const Problem &p, int dtype, RowsGeom *g, int *vx, int *r);
// Both of a 5 x 5 backward pass in one launch (k_rows_taprow_backward): the filter gradients' geometry and the
// feature gradient's, whose waves come in workgroups of as many here.
bool rows_taprow_backward_plan(const Problem &p, int dtype, RowsGeom *g, RowsGeom *gx, int *vxf, int *vx);

}  // namespace ddf

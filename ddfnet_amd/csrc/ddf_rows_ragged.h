// Launch code of the row-register kernels for rows that are no whole number of vectors
// (Ragged in ddf_rows.h), instantiated once per element type.  A row of 131 fp32 pixels takes
// 33 lanes of four pixels here where vectors that divide it are one pixel wide.
#pragma once

#include "ddf_rows_launch.h"

namespace ddf {
namespace rows {

template <typename T, int K, int D, int VX, int R, int TAIL>
hipError_t launch_ragged_kd(const Problem &p, const RowsGeom &g, bool backward, const T *x,
                            const T *cf, const T *sf, T *out, hipStream_t st) {
    const dim3 grid(g.xcd_per * kXcd), block(kWave * g.wpb);
#define DDF_ROWS_CASE(MUL_, BWD_)                                                               \
    hipLaunchKernelGGL((k_rows<T, K, D, MUL_, BWD_, VX, R, true, stages<K>(),                   \
                               waves_per_simd<T, K, VX, R, TAIL>(), 1, TAIL>),                  \
                       grid, block, 0, st, g, x, cf, sf, out)
    if (p.mul) {
        if (backward) DDF_ROWS_CASE(true, true);
        else DDF_ROWS_CASE(true, false);
    } else {
        if (backward) DDF_ROWS_CASE(false, true);
        else DDF_ROWS_CASE(false, false);
    }
#undef DDF_ROWS_CASE
    return hipGetLastError();
}

template <typename T, int VX, int TAIL>
hipError_t launch_ragged(const Problem &p, const RowsGeom &g, int r, bool backward, const T *x,
                         const T *cf, const T *sf, T *out, hipStream_t st) {
    if constexpr (VX * sizeof(T) == 16) {
        if (p.k == 3 && p.d == 1 && r == 2)
            return launch_ragged_kd<T, 3, 1, VX, 2, TAIL>(p, g, backward, x, cf, sf, out, st);
    }
    if (r != 1) return hipErrorNotSupported;
    if (p.k == 3 && p.d == 1) return launch_ragged_kd<T, 3, 1, VX, 1, TAIL>(p, g, backward, x, cf, sf, out, st);
    if (p.k == 3 && p.d == 2) return launch_ragged_kd<T, 3, 2, VX, 1, TAIL>(p, g, backward, x, cf, sf, out, st);
    if (p.k == 5 && p.d == 1) return launch_ragged_kd<T, 5, 1, VX, 1, TAIL>(p, g, backward, x, cf, sf, out, st);
    if (p.k == 5 && p.d == 2) return launch_ragged_kd<T, 5, 2, VX, 1, TAIL>(p, g, backward, x, cf, sf, out, st);
    return hipErrorNotSupported;
}

// Stride 2 (LaneStride2Ragged): forward or (BWD) the feature gradient.
template <typename T, bool BWD, int TAIL>
hipError_t launch_ragged_stride2(const Problem &p, const RowsGeom &g, const T *x, const T *cf,
                                 const T *sf, T *out, hipStream_t st) {
    const dim3 grid(g.xcd_per * kXcd), block(kWave * g.wpb);
    constexpr int VX = 8 / (int)sizeof(T);
    if (p.mul)
        hipLaunchKernelGGL((k_rows<T, 3, 1, true, BWD, VX, 1, true, kStages, 3, 2, TAIL>), grid, block, 0, st,
                           g, x, cf, sf, out);
    else
        hipLaunchKernelGGL((k_rows<T, 3, 1, false, BWD, VX, 1, true, kStages, 3, 2, TAIL>), grid, block, 0, st,
                           g, x, cf, sf, out);
    return hipGetLastError();
}

template <typename T, bool DX, int TAIL>
hipError_t launch_ragged_filters_stride2(const Problem &p, const RowsGeom &g, const T *go, const T *x,
                                         const T *cf, const T *sf, T *dx, T *dcf, T *dsf,
                                         typename Acc<T>::type *ws_sf, typename Acc<T>::type *ws_cf,
                                         unsigned need, hipStream_t st) {
    constexpr int VX = 8 / (int)sizeof(T), kStagesS2 = DX ? 2 : 4;   // (as launch_filters_stride2_v)
    const dim3 grid(g.xcd_per * kXcd), block(kWave * kFilterWaves);
    const int lds = filters_lds_bytes<9>((int)sizeof(typename Acc<T>::type), 1, VX);
    if (p.mul)
        hipLaunchKernelGGL((k_rows_filters<T, 3, 1, true, VX, 1, true, DX, kStagesS2, 2, 2, DX, TAIL>), grid,
                           block, lds, st, g, go, x, cf, sf, dx, dcf, dsf, ws_sf, ws_cf, need, 0);
    else
        hipLaunchKernelGGL((k_rows_filters<T, 3, 1, false, VX, 1, true, DX, kStagesS2, 2, 2, DX, TAIL>), grid,
                           block, lds, st, g, go, x, cf, sf, dx, dcf, dsf, ws_sf, ws_cf, need, 0);
    return hipGetLastError();
}

template <typename T, bool DX, int TAIL>
hipError_t launch_ragged_filters(const Problem &p, const RowsGeom &g, const T *go, const T *x,
                                 const T *cf, const T *sf, T *dx, T *dcf, T *dsf,
                                 typename Acc<T>::type *ws_sf, typename Acc<T>::type *ws_cf,
                                 unsigned need, int x_mod, hipStream_t st) {
    using A = typename Acc<T>::type;
    constexpr int kFilterStages = DX ? 2 : 4;   // (as launch_filters_v)
    const dim3 grid(g.xcd_per * kXcd), block(kWave * kFilterWaves);
    const int lds = filters_lds_bytes<9>((int)sizeof(A), 1, 4);
    if (p.k != 3 || (p.d != 1 && p.d != 2)) return hipErrorNotSupported;
#define DDF_ROWSF_CASE(D_, MUL_)                                                                 \
    hipLaunchKernelGGL((k_rows_filters<T, 3, D_, MUL_, 4, 1, true, DX, kFilterStages,            \
                                       MUL_ || DX ? 2 : 3, 1, DX, TAIL>),                        \
                       grid, block, lds, st, g, go, x, cf, sf, dx, dcf, dsf, ws_sf, ws_cf, need, x_mod)
    if (p.d == 1) {
        if (p.mul) DDF_ROWSF_CASE(1, true);
        else DDF_ROWSF_CASE(1, false);
    } else {
        if (p.mul) DDF_ROWSF_CASE(2, true);
        else DDF_ROWSF_CASE(2, false);
    }
#undef DDF_ROWSF_CASE
    return hipGetLastError();
}

template <typename T, int VX, int TAIL>
hipError_t launch_ragged_taprow(const Problem &p, const RowsGeom &g, const T *go, const T *x,
                                const T *cf, const T *sf, T *dcf, T *dsf,
                                typename Acc<T>::type *ws_sf, typename Acc<T>::type *ws_cf,
                                unsigned need, int x_mod, hipStream_t st) {
    using A = typename Acc<T>::type;
    const dim3 grid(g.xcd_per * kXcd), block(kWave * kTaprowWaves);
    const int lds = taprow_lds_bytes<5>((int)sizeof(A));
    if (p.k != 5 || (p.d != 1 && p.d != 2)) return hipErrorNotSupported;
#define DDF_TAPROW_CASE(D_, MUL_)                                                                \
    hipLaunchKernelGGL((k_rows_taprow_filters<T, 5, D_, MUL_, VX, 1, true, kTaprowStages,          \
                                              taprow_wpe<5, VX, MUL_>(), TAIL>), \
                       grid, block, lds, st, g, go, x, cf, sf, dcf, dsf, ws_sf, ws_cf, need, x_mod)
    if (p.d == 1) {
        if (p.mul) DDF_TAPROW_CASE(1, true);
        else DDF_TAPROW_CASE(1, false);
    } else {
        if (p.mul) DDF_TAPROW_CASE(2, true);
        else DDF_TAPROW_CASE(2, false);
    }
#undef DDF_TAPROW_CASE
    return hipGetLastError();
}

}  // namespace rows

template <typename T>
hipError_t rows_ragged_launch(const Problem &p, const RowsGeom &g, int vx, int r, bool backward,
                              const T *x, const T *cf, const T *sf, T *out, hipStream_t st) {
    if (p.s == 2) {
        if (vx * sizeof(T) != 8 || r != 1) return hipErrorNotSupported;
        if constexpr (sizeof(T) == 2) {
            if (g.shift)
                return backward ? rows::launch_ragged_stride2<T, true, 2>(p, g, x, cf, sf, out, st)
                                : rows::launch_ragged_stride2<T, false, 2>(p, g, x, cf, sf, out, st);
        }
        return backward ? rows::launch_ragged_stride2<T, true, 1>(p, g, x, cf, sf, out, st)
                        : rows::launch_ragged_stride2<T, false, 1>(p, g, x, cf, sf, out, st);
    }
    if constexpr (sizeof(T) == 2) {
        if (vx == 8)
            return g.shift ? rows::launch_ragged<T, 8, 2>(p, g, r, backward, x, cf, sf, out, st)
                           : rows::launch_ragged<T, 8, 1>(p, g, r, backward, x, cf, sf, out, st);
        if (vx == 4 && g.shift) return rows::launch_ragged<T, 4, 2>(p, g, r, backward, x, cf, sf, out, st);
    }
    if (vx == 4) return rows::launch_ragged<T, 4, 1>(p, g, r, backward, x, cf, sf, out, st);
    return hipErrorNotSupported;
}

template <typename T>
hipError_t rows_ragged_filters_launch(const Problem &p, const RowsGeom &g, const T *go, const T *x,
                                      const T *cf, const T *sf, T *dx, T *dcf, T *dsf,
                                      typename Acc<T>::type *ws_sf, typename Acc<T>::type *ws_cf,
                                      unsigned need, int x_mod, hipStream_t st) {
    if (p.s == 2) {
#define DDF_RAGGED_CASE(TAIL_)                                                                          \
    return dx ? rows::launch_ragged_filters_stride2<T, true, TAIL_>(p, g, go, x, cf, sf, dx, dcf, dsf,  \
                                                                    ws_sf, ws_cf, need, st)             \
              : rows::launch_ragged_filters_stride2<T, false, TAIL_>(p, g, go, x, cf, sf, dx, dcf, dsf, \
                                                                     ws_sf, ws_cf, need, st)
        if constexpr (sizeof(T) == 2) {
            if (g.shift) DDF_RAGGED_CASE(2);
        }
        DDF_RAGGED_CASE(1);
#undef DDF_RAGGED_CASE
    }
#define DDF_RAGGED_CASE(TAIL_)                                                                          \
    return dx ? rows::launch_ragged_filters<T, true, TAIL_>(p, g, go, x, cf, sf, dx, dcf, dsf, ws_sf,   \
                                                            ws_cf, need, x_mod, st)                     \
              : rows::launch_ragged_filters<T, false, TAIL_>(p, g, go, x, cf, sf, dx, dcf, dsf, ws_sf,  \
                                                             ws_cf, need, x_mod, st)
    if constexpr (sizeof(T) == 2) {
        if (g.shift) DDF_RAGGED_CASE(2);
    }
    DDF_RAGGED_CASE(1);
#undef DDF_RAGGED_CASE
}

template <typename T>
hipError_t rows_ragged_taprow_launch(const Problem &p, const RowsGeom &g, int vx, const T *go,
                                     const T *x, const T *cf, const T *sf, T *dcf, T *dsf,
                                     typename Acc<T>::type *ws_sf, typename Acc<T>::type *ws_cf,
                                     unsigned need, int x_mod, hipStream_t st) {
#define DDF_RAGGED_CASE(VX_, TAIL_)                                                              \
    return rows::launch_ragged_taprow<T, VX_, TAIL_>(p, g, go, x, cf, sf, dcf, dsf, ws_sf, ws_cf, need, x_mod, st)
    if constexpr (sizeof(T) == 2) {
        if (vx == 8 && g.shift) DDF_RAGGED_CASE(8, 2);
        if (vx == 8) DDF_RAGGED_CASE(8, 1);
        if (g.shift) DDF_RAGGED_CASE(4, 2);
    }
    if (vx == 4) DDF_RAGGED_CASE(4, 1);
    return hipErrorNotSupported;
#undef DDF_RAGGED_CASE
}

#define DDF_INSTANTIATE_RAGGED(T)                                                                  \
    template hipError_t rows_ragged_launch<T>(const Problem &, const RowsGeom &, int, int, bool,  \
                                              const T *, const T *, const T *, T *, hipStream_t); \
    template hipError_t rows_ragged_filters_launch<T>(const Problem &, const RowsGeom &, const T *, \
                                                      const T *, const T *, const T *, T *, T *,  \
                                                      T *, Acc<T>::type *, Acc<T>::type *,        \
                                                      unsigned, int, hipStream_t);                \
    template hipError_t rows_ragged_taprow_launch<T>(const Problem &, const RowsGeom &, int,      \
                                                     const T *, const T *, const T *, const T *,  \
                                                     T *, T *, Acc<T>::type *, Acc<T>::type *,    \
                                                     unsigned, int, hipStream_t);

}  // namespace ddf

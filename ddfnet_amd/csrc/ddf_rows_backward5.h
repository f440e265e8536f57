// All gradients of 5 x 5 filters in one launch (k_rows_taprow_backward), instantiated once per
// element type.
#pragma once

#include "ddf_rows_launch.h"

namespace ddf {
namespace rows {

// (both walks in the registers that the hungrier one has on its own)
template <typename T, int D, int VXF, int VX, bool PAD, int TAIL>
hipError_t launch_taprow_backward(const Problem &p, const RowsGeom &g, const RowsGeom &gx, const T *go, const T *x,
                                  const T *cf, const T *sf, T *dx, T *dcf, T *dsf, typename Acc<T>::type *ws_sf,
                                  typename Acc<T>::type *ws_cf, unsigned need, hipStream_t st) {
    const int blocks = (int)g.xcd_per * kXcd, lds = taprow_lds_bytes<5>((int)sizeof(typename Acc<T>::type));
    const dim3 grid(blocks + gx.xcd_per * kXcd), block(kWave * kTaprowWaves);
#define DDF_TAPROW_CASE(MUL_)                                                                                       \
    hipLaunchKernelGGL((k_rows_taprow_backward<T, D, MUL_, VXF, VX, PAD, kTaprowStages,                                  \
                                               std::min(taprow_wpe<5, VXF, MUL_>(), waves_per_simd<T, 5, VX, 1, TAIL>()), TAIL>), \
                       grid, block, lds, st, g, gx, blocks, go, x, cf, sf, dx, dcf, dsf, ws_sf, ws_cf, need)
    if (p.mul) DDF_TAPROW_CASE(true);
    else DDF_TAPROW_CASE(false);
#undef DDF_TAPROW_CASE
    return hipGetLastError();
}

}  // namespace rows

template <typename T>
hipError_t rows_taprow_backward_launch(const Problem &p, const RowsGeom &g, const RowsGeom &gx, int vxf, int vx, const T *go,
                                       const T *x, const T *cf, const T *sf, T *dx, T *dcf, T *dsf,
                                       typename Acc<T>::type *ws_sf, typename Acc<T>::type *ws_cf, unsigned need,
                                       hipStream_t st) {
    const int tail = rows::taprow_backward_tail(g);
    const bool pad = rows::taprow_backward_pad(g);
#define DDF_BACKWARD_CASE(D_, VXF_, VX_, PAD_, TAIL_)                                              \
    if (p.d == D_ && vxf == VXF_ && vx == VX_ && pad == PAD_ && tail == TAIL_)                     \
        return rows::launch_taprow_backward<T, D_, VXF_, VX_, PAD_, TAIL_>(p, g, gx, go, x, cf, sf, dx, dcf, dsf, ws_sf, ws_cf, need, st);
    DDF_BACKWARD5_BOTH_TYPES(DDF_BACKWARD_CASE)
    if constexpr (sizeof(T) == 2) {
        DDF_BACKWARD5_F16(DDF_BACKWARD_CASE)
    }
#undef DDF_BACKWARD_CASE
    return hipErrorNotSupported;
}

#define DDF_INSTANTIATE_BACKWARD5(T)                                                                                \
    template hipError_t rows_taprow_backward_launch<T>(const Problem &, const RowsGeom &, const RowsGeom &, int, int, \
                                                       const T *, const T *, const T *, const T *, T *, T *, T *,   \
                                                       Acc<T>::type *, Acc<T>::type *, unsigned, hipStream_t);

}  // namespace ddf

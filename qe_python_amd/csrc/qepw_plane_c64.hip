// The xy-plane stage in complex64 (qepw_plane.h).
#include "qepw_plane.h"

namespace qepw {

template <> const float2* plane_twiddles<float>(const Plan& p, int axis, bool square) {
  const int n = axis == 0 ? p.n1 : p.n2;
  return (square ? plane_square_table(n, false) : plane_lane_table(n, false)) ? p.d_ltw32[axis]
                                                                          : p.d_tw32[axis];
}

template PlaneChoice plane_choice<float>(const Plan& p, const StickTables& st);
template bool launch_plane_stage<float>(const Plan& p, const StickTables& st, float2* work,
                                         int64_t bstride, const float* V, int nb,
                                         hipStream_t stream);
template int launch_plane_group<float>(int count, const Plan* const* plans, float2* const* work,
                                        const int64_t* bstride, const float* const* V,
                                        const int* nb, hipStream_t stream);
template PlaneChoice density_choice<float>(const Plan& p, const StickTables& st);
template bool launch_density_stage<float>(const Plan& p, const StickTables& st, float2* work,
                                           int64_t bstride, const double* weights, int nb,
                                           int most, int* slices, bool accumulate,
                                           double* partial, hipStream_t stream);

}  // namespace qepw

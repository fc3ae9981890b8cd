// The xy-plane stage in complex128 (qepw_plane.h).
#include "qepw_plane.h"

namespace qepw {

template <> const double2* plane_twiddles<double>(const Plan& p, int axis, bool square) {
  const int n = axis == 0 ? p.n1 : p.n2;
  return (square ? plane_square_table(n, true) : plane_lane_table(n, true)) ? p.d_ltw64[axis]
                                                                          : p.d_tw64[axis];
}

template PlaneChoice plane_choice<double>(const Plan& p, const StickTables& st);
template bool launch_plane_stage<double>(const Plan& p, const StickTables& st, double2* work,
                                         int64_t bstride, const double* V, int nb,
                                         hipStream_t stream);
template int launch_plane_group<double>(int count, const Plan* const* plans, double2* const* work,
                                        const int64_t* bstride, const double* const* V,
                                        const int* nb, hipStream_t stream);
template PlaneChoice density_choice<double>(const Plan& p, const StickTables& st);
template bool launch_density_stage<double>(const Plan& p, const StickTables& st, double2* work,
                                           int64_t bstride, const double* weights, int nb,
                                           int most, int* slices, bool accumulate,
                                           double* partial, hipStream_t stream);

}  // namespace qepw

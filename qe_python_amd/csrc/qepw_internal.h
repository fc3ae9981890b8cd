// Internal declarations shared by the HIP translation units.
#pragma once

#include <string>

#include "qepw_common.h"
#include "qepw_plan.h"
#include "../../include/qepw.h"

namespace qepw {

constexpr int kMaxLdsBytes = 160 * 1024;
constexpr int64_t kMaxLaunch = 0xffffffff;  // threads of a launch and dimension

// Raises a kernel's dynamic LDS limit where a launch needs more than the 64 KB
// every kernel may use (the call costs a microsecond of a launch).
inline void allow_lds(const void* kernel, size_t bytes) {
  if (bytes > 64 * 1024)
    (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// Line lengths with a team FFT.
#define QEPW_TEAM_SIZES(X) \
  X(16) X(18) X(20) X(24) X(25) X(27) X(30) X(32) X(36) X(40) X(45) X(48) X(50) X(54) \
  X(60) X(64) X(72) X(75) X(80) X(81) X(90) X(96) X(100) X(108) X(120) X(128) X(135) \
  X(144) X(150) X(160) X(180) X(192)

// Grouped launches (qepw_apply_local_group): up to kMaxFftGroup problems whose
// plane side and z length are among QEPW_GROUP_SIZES.
#define QEPW_GROUP_SIZES(X) X(36) X(48) X(54) X(60) X(64) X(72) X(80) X(96)
constexpr int kMaxFftGroup = 24;

__device__ __forceinline__ int group_of(const int* start, int count, int bx) {
  int p = 0;
  while (p + 1 < count && start[p + 1] <= bx) ++p;
  return p;
}

// qepw_fft.hip
int stick_group_for(int n3, int nst);
size_t apply_local_band_bytes(const Plan& p, int precision);
int apply_local_group(int count, const Plan* const* plans, int precision,
                      const void* const* vectors, const int64_t* ldv, const int* nb,
                      const void* const* potentials, const void* const* kinetics,
                      void* const* results, const int64_t* ldr, void* const* workspaces,
                      const size_t* ws_bytes, hipStream_t stream);
int apply_local(const Plan& p, int precision, const void* vectors, int64_t ldv, int nb,
                const void* potential, const void* kinetic, void* result, int64_t ldr,
                void* workspace, size_t ws_bytes, hipStream_t stream);
size_t density_workspace_bytes(const Plan& p, int precision, int nb);
int accumulate_density(const Plan& p, int precision, const void* vectors, int64_t ldv, int nb,
                       const double* weights, double scale, double* out, void* workspace,
                       size_t ws_bytes, hipStream_t stream);
unsigned team_slot_mask(int n, const std::vector<int>& positions);
size_t inverse_real_bytes(const Plan& p);
int inverse_real(const Plan& p, const void* grid_g, void* out_real, void* workspace,
                 size_t ws_bytes, hipStream_t stream);

// qepw_plane_c128.hip, qepw_plane_c64.hip (the xy-plane stage, qepw_plane.h)
// Whether the lines of length n load their twiddles instead of holding them.
// Held, long FP64 lines spill or halve the waves a CU runs.  Squares, FFT phase of
// 24 planes of 128 bands in FP64, loaded and held, us: 36^2 42.9 and 40, 48^2 62
// and 62, 60^2 88 and 87, 72^2 100 and 96, 80^2 155 and 139, 81^2 178 and 156, but
// 75^2 (fifteen twiddles) 221 and 284, 90^2 186 and 207, 96^2 215 and 231, 108^2 275
// and 334, 128^2 452 and 683; FP32 72^2 75 and 66, 108^2 155 and 145, 128^2 346 and
// 378.
constexpr bool plane_square_table(int n, bool fp64) {
  const int m = team_L(n) > 0 ? n / team_L(n) : 0;
  return fp64 ? m > 10 || n > 81 : m >= 15;
}
// The kernels of any two lengths share their registers among all: FP64 lines hold
// nine twiddles up to 72 and load all others (64 bands, loaded and held as above: 81
// x 64 x 30 99 and 113 us, 50 x 64 x 40 79 and 85, 60 x 80 x 48 154 and 163, 36 x 40
// x 160 120 and 118).
constexpr bool plane_lane_table(int n, bool fp64) {
  const int m = team_L(n) > 0 ? n / team_L(n) : 0;
  return fp64 ? !(m == 9 && n <= 72) : m >= 15;
}
template <typename T> PlaneChoice plane_choice(const Plan& p, const StickTables& st);
template <typename T>
bool launch_plane_stage(const Plan& p, const StickTables& st, cplx<T>* work, int64_t bstride,
                        const T* V, int nb, hipStream_t stream);
template <typename T> PlaneChoice density_choice(const Plan& p, const StickTables& st);
template <typename T>
bool launch_density_stage(const Plan& p, const StickTables& st, cplx<T>* work, int64_t bstride,
                          const double* weights, int nb, int most, int* slices, bool accumulate,
                          double* partial, hipStream_t stream);
// Planes (of all bands and problems) of one grouped launch, and the class of a
// problem: those of one class share a launch (k_plane_group).  Lengths whose kernels
// take up to 156 registers in FP64, or 117 in FP32, share a kernel (0); the others
// have one each, which their registers would otherwise set for all.
inline int64_t plane_group_most(int waves) { return kMaxLaunch / (64 * waves); }
constexpr int plane_group_kind(int n, bool fp64) {
  return (fp64 ? n <= 54 || n == 64 : n <= 72) ? 0 : n;
}
inline int plane_group_class(const Plan& p, const PlaneChoice& c, bool fp64) {
  return (plane_group_kind(p.n1, fp64) * 16 + c.waves) * 2 + (c.prune ? 1 : 0);
}
template <typename T>
int launch_plane_group(int count, const Plan* const* plans, cplx<T>* const* work,
                       const int64_t* bstride, const T* const* V, const int* nb,
                       hipStream_t stream);

// qepw_gemm.hip
size_t gemm_workspace_bytes(int precision, int op_a, int64_t m, int64_t n, int64_t k);
int gemm_set_rule(int precision, int op_a, const int64_t* ranges, int variant, int64_t splits);
void gemm_clear_rules();
int gemm_variant_count();
int gemm_plan(int precision, int op_a, int64_t m, int64_t n, int64_t k, int64_t* out);
int gemm(int precision, int op_a, int64_t m, int64_t n, int64_t k, const double* alpha,
         const void* a, int64_t lda, const void* b, int64_t ldb, const double* beta,
         void* c, int64_t ldc, void* workspace, size_t ws_bytes, hipStream_t stream);
size_t position_gradient_bytes(int precision, int64_t npw, int64_t nproj, int64_t nb);
int position_gradient(int precision, int64_t npw, int64_t nproj, int nb, const void* psi,
                      int64_t ldpsi, const void* coupled, int64_t ldc, const double* f,
                      const void* proj, int64_t ldproj, const double* q, const int* off,
                      int natom, double* out, void* ws, size_t ws_bytes, hipStream_t stream);
int herm_product(int n, const void* x, const void* y, const void* d, void* c, int64_t ld,
                 double alpha, double beta, hipStream_t stream);

// qepw_vec.hip
int column_squared_norms(int precision, const void* v, int64_t ldv, int64_t nrows, int nb,
                         double* out, hipStream_t stream);
int column_inner_products(int precision, const void* l, int64_t ldl, const void* r,
                          int64_t ldr, int64_t nrows, int nb, double* out, hipStream_t stream);
int subtract_band_energies(int precision, void* r, int64_t ldr, const void* x, int64_t ldx,
                           const double* e, int64_t nrows, int nb, hipStream_t stream);
int qe_precondition(int precision, const void* r, int64_t ldr, const int* cols,
                    const double* e, const double* diag, void* out, int64_t ldo,
                    int64_t nrows, int nb, hipStream_t stream);
int normalize_selected_columns(int precision, const void* src, int64_t lds,
                               const double* sq, const int* sel, void* dst, int64_t ldd,
                               int64_t nrows, int nb, hipStream_t stream);
int restart_applied(int precision, const void* x, int64_t ldx, const void* r, int64_t ldr,
                    const double* e, void* hv, int64_t ldh, int64_t nrows, int nb,
                    hipStream_t stream);
int permute_rows(int src_precision, int dst_precision, int direction, const int* perm,
                 const void* src, int64_t lds, void* dst, int64_t ldd, int64_t nrows, int nb,
                 const double* cfac, hipStream_t stream);
int row_real_dot(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t nrows,
                 int ncols, double scale, double* acc, hipStream_t stream);
int copy_columns(int src_precision, int dst_precision, const void* src, int64_t lds,
                 const int* scol, void* dst, int64_t ldd, const int* dcol, const double* scale,
                 int64_t nrows, int ncols, hipStream_t stream);
int set_block(int precision, void* dst, int64_t ldd, int64_t nrows, int ncols, double diag,
              const double* d, hipStream_t stream);
int scale_rows(int precision, const void* src, int64_t lds, const double* s, int64_t sstride,
               const double* cfac, void* dst, int64_t ldd, int64_t nrows, int nb,
               hipStream_t stream);
int build_projectors(int precision, const void* beta, int64_t ldb, int nch, const double* q,
                     const double* tau, int natom, void* out, int64_t ldo, int64_t nrows,
                     hipStream_t stream);
int phase_blocks(int precision, const void* beta, int64_t ldb, int nch, const void* phases,
                 int64_t ldp, int natom, const int* perm, void* out, int64_t ldo, int64_t nrows,
                 hipStream_t stream);
int projector_forces(int precision, const void* dO, int64_t lddo, int64_t dstride,
                     const void* DO, int64_t lddO, const double* f, int nb, const int* off,
                     int natom, double* out, hipStream_t stream);

int column_axpby(int precision, const void* x, int64_t ldx, const double* a, void* y,
                 int64_t ldy, const double* b, int64_t nrows, int ncols, hipStream_t stream);
int column_diagonal_expectations(int precision, const void* v, int64_t ldv, const double* d,
                                 int64_t nrows, int nb, double* out, hipStream_t stream);
int rmm_precondition(int precision, const void* r, int64_t ldr, const int* cols,
                     const double* kinetic, const double* expect, void* out, int64_t ldo,
                     int64_t nrows, int ncols, hipStream_t stream);
int history_combine(int precision, const void* hist, int64_t ldh, int64_t hstride, int count,
                    const int* cols, const double* coef, void* out, int64_t ldo, int64_t nrows,
                    int ncols, hipStream_t stream);

int projector_basis(const double* q, int64_t npw, const double* table, int64_t ldt, int nq,
                    double dq, const int* chan_radial, const int* chan_l, const int* chan_m,
                    int nch, void* beta, int64_t ldb, hipStream_t stream);

// qepw_eig.hip
int hermitian_complete(void* a, int64_t lda, int first, int active, hipStream_t stream);
int shift_scale(const void* a, int64_t lda, int n, double sigma, void* x, int64_t ldx,
                double* bound, hipStream_t stream);
int hermitize(void* x, int64_t ldx, int n, hipStream_t stream);
int sign_check(const void* x, int64_t ldx, const void* x2, int64_t ld2, int n, double* out,
               hipStream_t stream);
int set_diagonal(void* a, int64_t lda, int n, const double* d, hipStream_t stream);
size_t sign_iteration_workspace(int n);
int sign_iteration(void* x, void* x2, void* y, int64_t ld, int n, const double* alphas,
                   int nalpha, int* in_x2, void* ws, size_t ws_bytes, hipStream_t stream);

// qepw_rr.hip
void set_host_lapack(void* zpotrf, void* ztrtri, void* zheevd, void* cheevd);
bool host_lapack_ready();
const std::string& rr_message();
size_t rr_workspace_bytes(int maxsub);
int rr_standardize(void* H, void* S, void* W, void* A, int maxsub, int first, int active,
                   int* not_pd, void* work, size_t work_bytes, hipStream_t stream);
int rr_spectral(const qepw_rr_spectral_args* a, double* values, qepw_rr_spectral_result* out);
int cholesky_qr(int precision, const void* block, int64_t ldb, int64_t npw, int nb,
                double condition, void* out, int64_t ldo, int* ok, void* work,
                size_t work_bytes, hipStream_t stream);

}  // namespace qepw

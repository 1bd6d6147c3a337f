// Launchers of the chi^2 gradient / Gauss-Newton kernels (grad.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "fitdesc.h"

namespace mhre {

// chi2[n] (and grad[n][ldp] when grad != nullptr) of the 9-parameter model
// for the parameter vectors P[n][ldp] against one fit's packed data fd.
// ring != 0: the fit's closures lie inside the ring window (FitDesc::ring_ok),
// so the single-pass ring form is used.  split > 1: a work-group of that many
// waves per point, with split_lds = eht_grad_split_lds bytes of LDS for the fit.
hipError_t launch_eht_grad9(const FitDesc* fd, const float* P, int n, int ldp, double* chi2, float* grad,
                            int ring, int split, size_t split_lds, hipStream_t s);
constexpr int GRAD_SPLIT_MAXW = 16;
constexpr size_t GRAD_SPLIT_STATIC_LDS = 16 << 10;   // bound of its other LDS (tables, sums)
constexpr int GRAD_SPLIT_WAVES_PER_CU = 20;          // its registers allow 5 waves per SIMD
constexpr size_t eht_grad_split_lds(size_t ntile, size_t ncph) {
  return ntile * TILE * sizeof(float2) + ncph * sizeof(float);
}
// chi2[n], J^T r [n][9] and J^T J of the weighted residuals r: its upper
// triangle [n][45] (row-major), or with full the matrices [n][9][9].
hipError_t launch_eht_gn9(const FitDesc* fd, const float* P, int n, int ldp, double* chi2, double* jtr,
                          double* jtj, int full, hipStream_t s);

// Residuals r [rows][neq] and Jacobian J [rows][neq][n] of quadratic systems
// x^T Q_e x + b_e . x - dat_e for parameter rows X [rows][n].
hipError_t launch_quad_jac(const float* Q, const float* b, const float* dat, const int* sys, const float* X,
                           int rows, int neq, int n, float* r, float* J, hipStream_t s);

}  // namespace mhre

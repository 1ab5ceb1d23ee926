// response.h -- parameters and launchers of the dense response contraction (response.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace oqph {

struct ResponseParams {
  const double* T;  // [npair][n][ld]
  const double* M;  // densities [.][n][ld], columns n .. ld zero
  double* F;        // [.][n][n], added into
  const int* col;   // the ncol densities of this product
  int ncol, n, ld, ncu;
  long long npair;
  double scale;
};

void launch_rsp_pack(const double* raw, int n, int ld, int nmat, int nf, double* M, hipStream_t s);
void launch_rsp_unpack(const double* F, int n, int nmat, int nf, double* raw, hipStream_t s);
void launch_response(bool coulomb, const ResponseParams& r, hipStream_t s);

}  // namespace oqph

// Batched production rates and right-hand sides, one state per lane: each
// lane evaluates a whole state with the generated straight-line code of the
// mechanism (lane_rhs_<mech>.h).  Component-major arrays, so lane c's loads and
// stores of component k are coalesced.  Bound by FP64 VALU issue: a state's
// rates are some 20,000 instructions (GRI-3.0), half of them polynomials of
// 2^x.  Against a wavefront per state (prodrates_kernel, rhs_kernel) no lane
// idles in the reductions and no cross-lane traffic is left.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "chem_kernels.h"
#include "lane_rhs_dme39.h"
#include "lane_rhs_ethyred.h"
#include "lane_rhs_gri30.h"
#include "lane_rhs_h2.h"

namespace tgr {

template <int NEQ>
__global__ __launch_bounds__(64) void rhs_lanes_kernel(int64_t n, double p_gp, const double* y, double* f) {
  const int64_t c = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (c >= n) return;
  double s[NEQ], o[NEQ];
#pragma unroll
  for (int k = 0; k < NEQ; ++k) s[k] = y[k * n + c];
  LaneRhs<NEQ>::eval(s, p_gp, o);
#pragma unroll
  for (int k = 0; k < NEQ; ++k) f[k * n + c] = o[k];
}

template <int NEQ>
__global__ __launch_bounds__(64) void prodrates_lanes_kernel(int64_t n, const double* C, const double* T,
                                                             const double* P, double* cdot) {
  constexpr int nsp = NEQ - 1;
  const int64_t c = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (c >= n) return;
  double s[nsp], o[nsp];
#pragma unroll
  for (int k = 0; k < nsp; ++k) s[k] = C[k * n + c];
  LaneRhs<NEQ>::rates(s, T[c], P[c], o);
#pragma unroll
  for (int k = 0; k < nsp; ++k) cdot[k * n + c] = o[k];
}

}  // namespace tgr

using namespace tgr;

extern "C" int tgr_launch_rhs_lanes(int neq, int64_t n, double p_gp, const double* y, double* f, hipStream_t s) {
  if (n <= 0) return 0;
  const dim3 grid((unsigned)((n + 63) / 64));
  switch (neq) {
    case 10: hipLaunchKernelGGL(rhs_lanes_kernel<10>, grid, dim3(64), 0, s, n, p_gp, y, f); break;
    case 37: hipLaunchKernelGGL(rhs_lanes_kernel<37>, grid, dim3(64), 0, s, n, p_gp, y, f); break;
    case 40: hipLaunchKernelGGL(rhs_lanes_kernel<40>, grid, dim3(64), 0, s, n, p_gp, y, f); break;
    case 46: hipLaunchKernelGGL(rhs_lanes_kernel<46>, grid, dim3(64), 0, s, n, p_gp, y, f); break;
    default: return -1;
  }
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

extern "C" int tgr_launch_prodrates_lanes(int neq, int64_t n, const double* C, const double* T, const double* P,
                                          double* cdot, hipStream_t s) {
  if (n <= 0) return 0;
  const dim3 grid((unsigned)((n + 63) / 64));
  switch (neq) {
    case 10: hipLaunchKernelGGL(prodrates_lanes_kernel<10>, grid, dim3(64), 0, s, n, C, T, P, cdot); break;
    case 37: hipLaunchKernelGGL(prodrates_lanes_kernel<37>, grid, dim3(64), 0, s, n, C, T, P, cdot); break;
    case 40: hipLaunchKernelGGL(prodrates_lanes_kernel<40>, grid, dim3(64), 0, s, n, C, T, P, cdot); break;
    case 46: hipLaunchKernelGGL(prodrates_lanes_kernel<46>, grid, dim3(64), 0, s, n, C, T, P, cdot); break;
    default: return -1;
  }
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

// oa_vks_point.h -- what both V_KS engines (oa_vks.hip, oa_vks2.h) compute per
// point, per G and at the end.
#pragma once

#include "oa_common.h"
#include "oa_kernels.h"

namespace oa {

__device__ __forceinline__ int sfreq(int i, int n) { return i <= (n - 1) / 2 ? i : i - n; }

__device__ __forceinline__ double gsq(const double* hi, int a, int b, int c) {
  const double tpi = 6.283185307179586476925;
  const double xk = (a * hi[0] + b * hi[1] + c * hi[2]) * tpi;
  const double yk = (a * hi[3] + b * hi[4] + c * hi[5]) * tpi;
  const double zk = (a * hi[6] + b * hi[7] + c * hi[8]) * tpi;
  return xk * xk + yk * yk + zk * zk;
}

// Perdew-Zunger 1981 LDA per point: exchange factor xf, correlation energy
// factor cf and potential factor mf (cp_pz_lda.C:48-54, 114-138).  One cube
// root serves both powers: rs = (3/(4 pi))^(1/3) / rho^(1/3) and
// xf = -(3/pi)^(1/3) rho^(1/3).
__device__ __forceinline__ void pz_lda(double r, double& xf, double& cf, double& mf) {
  const double gamma = -0.14230, beta1 = 1.05290, beta2 = 0.33340;
  const double au = 0.03110, bu = -0.0480, cu = 0.00200, du = -0.01160;
  const double power = 1.0 / 3.0;
  const double rat1 = (7.0 / 6.0) * beta1, rat2 = (4.0 / 3.0) * beta2;
  const double c_rs = 0.62035049089940001667;  // (3/(4 pi))^(1/3)
  const double c_x = 0.98474502184269654118;   // (3/pi)^(1/3)
  const double cr = cbrt(r);
  const double rs = c_rs / cr;
  const double sq = sqrt(rs);
  xf = -c_x * cr;
  if (rs >= 1.0) {
    const double c1 = 1.0 + beta1 * sq + beta2 * rs;
    const double c2 = 1.0 + rat1 * sq + rat2 * rs;
    cf = gamma / c1;
    mf = cf * (c2 / c1);
  } else {
    const double l = log(rs);
    cf = au * l + bu + cu * rs * l + du * rs;
    mf = au * l + (bu - power * au) + 2.0 * power * cu * rs * l + power * (2.0 * du - cu) * rs;
  }
}

// sum of NV values over the workgroup (fixed order); result valid on thread 0
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* sh) {
#pragma unroll
  for (int k = 0; k < NV; k++)
    for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < NV; k++) sh[w * NV + k] = v[k];
  __syncthreads();
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < NV; k++) {
      double acc = 0.0;
      for (int i = 0; i < (int)blockDim.x / 64; i++) acc += sh[i * NV + k];
      v[k] = acc;
    }
}

// fixed-order sums of the partials: E_xc = (3/4 ex + ec) Omega/N,
// muxc = sum V_xc rho Omega/N (cp_pz_lda.C:158-167), E_H = half the sum,
// E_ext (cp_hart_ext.C:385-387)
// sh: five doubles per wave
__device__ __forceinline__ void vks_sum(const double* __restrict__ px, int nbx,
                                        const double* __restrict__ pl, int nbl, double sc,
                                        StepDev* res, double* sh) {
  double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  // eight loads in flight; past the end a clamped index, not added
  auto sum = [](const double* p, int n, int nv, double* to) {
    for (int i0 = threadIdx.x; i0 < n; i0 += 8 * blockDim.x)
      for (int k = 0; k < nv; k++) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const int i = i0 + u * (int)blockDim.x;
          v[u] = p[nv * min(i, n - 1) + k];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) to[k] += i0 + u * (int)blockDim.x < n ? v[u] : 0.0;
      }
  };
  double ex[3] = {0.0, 0.0, 0.0}, eh[2] = {0.0, 0.0};
  sum(px, nbx, 3, ex);
  sum(pl, nbl, 2, eh);
  for (int k = 0; k < 3; k++) acc[k] = ex[k];
  for (int k = 0; k < 2; k++) acc[3 + k] = eh[k];
  block_sum<5>(acc, sh);
  if (threadIdx.x == 0) {
    res->exc = (0.75 * acc[0] + acc[1]) * sc;
    res->muxc = acc[2] * sc;
    res->ehart = 0.5 * acc[3];
    res->eloc = acc[4];
  }
}

}  // namespace oa

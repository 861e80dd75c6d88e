// oa_pointwise.hip -- G-space pointwise kernels and small reductions of the
// CP electronic step.
//   k_sd       : psi += dt/m F  (CP_integrate_min_STD, cp_min_std.C:56-86)
//   cg_gamma, k_cg_update : conjugate-gradient direction and update
//                (CP_integrate_min_CG, cp_min_CG.C:55-105; reset rule
//                 CP_State_GSpacePlane.C:2646-2671)
//   k_red_sync : redundant kx=0 points <- conj(partner)
//                (CP_State_GSpacePlane.C:2862-3061)
//   k_vperm    : V(r) into the lane order of the row-class R->G pass
//   k_reduce_to, k_dot, k_resid, k_fill_zero, k_zero_rows: deterministic
//   reductions and graph-safe zero fills.
#include <algorithm>

#include "oa_common.h"
#include "oa_kernels.h"

namespace oa {

__device__ __forceinline__ double block_sum(double v) {
  __shared__ double red[16];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += red[w];
  return t;
}

__global__ void k_sd(double2* __restrict__ psi, const double2* __restrict__ f,
                     const double* __restrict__ dtm, const int* __restrict__ twin, int nst,
                     int npts, int ld, double* __restrict__ fpart) {
  const size_t tot = (size_t)nst * npts;
  double fn = 0.0;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const int s = (int)(e / npts), p = (int)(e - (size_t)s * npts);
    const size_t o = (size_t)s * ld + p;
    const double2 fv = f[o];
    const double m = dtm[p];
    const int tw = twin ? twin[p] : -1;
    double2 c = psi[o];
    c.x += fv.x * m;
    c.y += fv.y * m;
    if (tw != -2) psi[o] = c;  // a redundant point is written by its partner
    if (tw >= 0) psi[(size_t)s * ld + tw] = make_double2(c.x, -c.y);
    fn += fv.x * fv.x + fv.y * fv.y;
  }
  const double t = block_sum(fn);
  if (threadIdx.x == 0) fpart[blockIdx.x] = t;
}

hipError_t sd_update(double2* psi, const double2* f, const double* dtm, const int* twin, int nst,
                     int npts, int ld, double* fpart, int nfpart, hipStream_t st) {
  hipLaunchKernelGGL(k_sd, dim3(nfpart), dim3(256), 0, st, psi, f, dtm, twin, nst, npts, ld,
                     fpart);
  return hipGetLastError();
}

// acceptCgOverlap (CP_State_GSpacePlane.C:131-135) and the reset rule
// (:2651-2671): gamma = 0 on the first iteration, or when |F| grew by more
// than 5% after at least five steps without a reset, or more than doubled;
// else fovlap / fovlap_old.
__device__ __forceinline__ void cg_gamma(double fnorm2, CgDev* __restrict__ cg) {
  CgDev s = *cg;
  s.fovlap_old = s.fovlap;
  s.fmag_old = s.fmag;
  s.fovlap = fnorm2;
  s.fmag = sqrt(s.fovlap);
  s.iter++;
  int reset = 0;
  if (s.iter == 1) {
    reset = 1;
    s.num_reset = 0;
  } else if ((s.fmag > 1.05 * s.fmag_old && s.num_reset >= 5) || s.fmag > 2.0 * s.fmag_old) {
    reset = 1;
    s.num_reset = 0;
  }
  s.num_reset++;
  s.gamma = reset ? 0.0 : s.fovlap / s.fovlap_old;
  *cg = s;
}

// cg = gamma cg + F where g2 <= ecut; psi += dt/m cg (cp_min_CG.C:55-105), and
// the redundant kx=0 points from their partners (twin: -1, -2 for a redundant
// point, or the index of the redundant twin, as in k_sd).  Block (b, s): 1024
// points of state s, four per thread with every load issued before the first
// use: five streams of 16 bytes per point at the rate of a copy (256 states x
// 65,912 points 264 -> 132 us; one point per iteration and a division for its
// state left too few bytes in flight).
constexpr int kCgPer = 4;
__global__ __launch_bounds__(256) void k_cg_update(
    double2* __restrict__ psi, double2* __restrict__ cgd, const double2* __restrict__ f,
    const double* __restrict__ dtm, const double* __restrict__ g2, const int* __restrict__ twin,
    double ecut, int npts, int ld, const CgDev* __restrict__ cg) {
  const double gamma = cg->gamma;
  const size_t row = (size_t)blockIdx.y * ld;
  const int p0 = blockIdx.x * (256 * kCgPer) + threadIdx.x;
  double2 d[kCgPer], fv[kCgPer], c[kCgPer];
  double m[kCgPer], gg[kCgPer];
  int tw[kCgPer];
#pragma unroll
  for (int u = 0; u < kCgPer; u++) {
    const int p = min(p0 + 256 * u, npts - 1);
    d[u] = cgd[row + p];
    fv[u] = f[row + p];
    c[u] = psi[row + p];
    m[u] = dtm[p];
    gg[u] = g2[p];
    tw[u] = twin[p];
  }
#pragma unroll
  for (int u = 0; u < kCgPer; u++) {
    const int p = p0 + 256 * u;
    if (p >= npts) continue;
    if (gg[u] <= ecut) {
      d[u].x = d[u].x * gamma + fv[u].x;
      d[u].y = d[u].y * gamma + fv[u].y;
      cgd[row + p] = d[u];
    }
    c[u].x += d[u].x * m[u];
    c[u].y += d[u].y * m[u];
    if (tw[u] != -2) psi[row + p] = c[u];
    if (tw[u] >= 0) psi[row + tw[u]] = make_double2(c[u].x, -c[u].y);
  }
}

hipError_t cg_update(double2* psi, double2* cgdir, const double2* f, const double* dtm,
                     const double* g2, const int* twin, double ecut, int nst, int npts, int ld,
                     const CgDev* cg, hipStream_t st) {
  hipLaunchKernelGGL(k_cg_update, dim3((npts + 256 * kCgPer - 1) / (256 * kCgPer), nst),
                     dim3(256), 0, st, psi, cgdir, f, dtm, g2, twin, ecut, npts, ld, cg);
  return hipGetLastError();
}

__global__ void k_red_sync(double2* __restrict__ psi, const int* __restrict__ red,
                           const int* __restrict__ partner, int nred, int nst, int ld) {
  const size_t tot = (size_t)nst * nred;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const int s = (int)(e / nred), r = (int)(e - (size_t)s * nred);
    const double2 v = psi[(size_t)s * ld + partner[r]];
    psi[(size_t)s * ld + red[r]] = make_double2(v.x, -v.y);
  }
}

hipError_t red_sync(double2* psi, const int* red, const int* partner, int nred, int nst, int ld,
                    hipStream_t st) {
  if (nred == 0) return hipSuccess;
  const size_t tot = (size_t)nst * nred;
  int blocks = (int)((tot + 255) / 256);
  if (blocks > 2048) blocks = 2048;
  hipLaunchKernelGGL(k_red_sync, dim3(blocks), dim3(256), 0, st, psi, red, partner, nred, nst,
                     ld);
  return hipGetLastError();
}

// One workgroup per sum; each thread's loads are issued eight at a time
// (branch-free: index clamped, value masked) rather than one per iteration.  cg:
// the first sum is |F|^2 of a new conjugate-gradient direction.  The sums of a step
// (EKE, E_loc, |F|^2 and the direction's gamma) were four launches of 3 us, with as
// much again between them.
constexpr int kRedThreads = 1024;
__global__ __launch_bounds__(kRedThreads) void k_reduce_to(RedJob j0, RedJob j1, RedJob j2,
                                                           CgDev* cg) {
  const RedJob j = blockIdx.x == 0 ? j0 : blockIdx.x == 1 ? j1 : j2;
  const double* __restrict__ part = j.part;
  const int n = j.n;
  double v = 0.0;
  for (int i0 = 0; i0 < n; i0 += 8 * kRedThreads) {
    double a[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int i = i0 + (int)threadIdx.x + u * kRedThreads;
      const double w = part[min(i, n - 1)];
      a[u] = i < n ? w : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 8; u++) v += a[u];
  }
  const double t = block_sum(v);
  if (threadIdx.x == 0) {
    *j.out = t * j.scale;
    if (cg && blockIdx.x == 0) cg_gamma(t * j.scale, cg);
  }
}

hipError_t reduce_to(const RedJob* jobs, int njobs, CgDev* cg, hipStream_t st) {
  if (njobs < 1 || njobs > 3) return hipErrorInvalidValue;
  for (int i = 0; i < njobs; i++)
    if (jobs[i].n < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_reduce_to, dim3(njobs), dim3(kRedThreads), 0, st, jobs[0],
                     jobs[std::min(1, njobs - 1)], jobs[njobs - 1], cg);
  return hipGetLastError();
}

__global__ void k_dot(const double* __restrict__ a, const double* __restrict__ b, size_t n,
                      double* __restrict__ part) {
  double v = 0.0;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n;
       e += (size_t)gridDim.x * blockDim.x)
    v += a[e] * b[e];
  const double t = block_sum(v);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

hipError_t dot_parts(const double* a, const double* b, size_t n, double* part, int nparts,
                     hipStream_t st) {
  hipLaunchKernelGGL(k_dot, dim3(nparts), dim3(256), 0, st, a, b, n, part);
  return hipGetLastError();
}

__global__ void k_resid(const double* __restrict__ S, int n, StepDev* res) {
  __shared__ double rmax[16];
  double mx = 0.0, ss = 0.0;
  const size_t nn = (size_t)n * n;
  for (size_t e = threadIdx.x; e < nn; e += blockDim.x) {
    const size_t i = e / n, j = e - i * n;
    const double d = 0.5 * S[e] - (i == j ? 1.0 : 0.0);
    mx = fmax(mx, fabs(d));
    ss += d * d;
  }
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_down(mx, o, 64));
  if ((threadIdx.x & 63) == 0) rmax[threadIdx.x >> 6] = mx;
  const double tot = block_sum(ss);
  if (threadIdx.x == 0) {
    double m = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) m = fmax(m, rmax[w]);
    res->resid_max = m;
    res->resid_rms = sqrt(tot / (double)nn);
  }
}

hipError_t resid_stats(const double* S, int n, StepDev* res, hipStream_t st) {
  hipLaunchKernelGGL(k_resid, dim3(1), dim3(1024), 0, st, S, n, res);
  return hipGetLastError();
}

__global__ void k_vperm(VPerm vp, const double* __restrict__ v, int nz) {
  const size_t tot = (size_t)nz * vp.n * vp.n;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const size_t r = e / vp.n;
    const int x = (int)(e - r * vp.n), z = (int)(r / vp.n), y = (int)(r - (size_t)z * vp.n);
    vp.put(z, y, x, v[e]);
  }
}

hipError_t vperm_set(const VPerm& vp, const double* v, int nz, hipStream_t st) {
  if (!vp.p) return hipSuccess;
  hipLaunchKernelGGL(k_vperm, dim3(1024), dim3(256), 0, st, vp, v, nz);
  return hipGetLastError();
}

template <typename T>
__global__ void k_zero_rows(cpx<T>* __restrict__ z, size_t ncol, int ny) {
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < ncol;
       e += (size_t)gridDim.x * blockDim.x)
    z[e * ny + ny / 2] = {(T)0, (T)0};
}

hipError_t zero_rows(void* zbuf, size_t ncol, int ny, bool fp32, hipStream_t st) {
  if (fp32)
    hipLaunchKernelGGL(k_zero_rows<float>, dim3(1024), dim3(256), 0, st, (cpx<float>*)zbuf, ncol,
                       ny);
  else
    hipLaunchKernelGGL(k_zero_rows<double>, dim3(1024), dim3(256), 0, st, (cpx<double>*)zbuf,
                       ncol, ny);
  return hipGetLastError();
}

__global__ void k_fill_zero(uint32_t* __restrict__ p, size_t n) {
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n;
       e += (size_t)gridDim.x * blockDim.x)
    p[e] = 0u;
}

hipError_t fill_zero(void* p, size_t bytes, hipStream_t st) {
  const size_t n = bytes / 4;
  if (n == 0) return hipSuccess;
  int blocks = (int)((n + 255) / 256);
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_fill_zero, dim3(blocks), dim3(256), 0, st, (uint32_t*)p, n);
  return hipGetLastError();
}

}  // namespace oa

// oa_vks2.h -- V_KS(r) from rho(r) on the two-factor register engine, for grids
// whose three lengths are compiled (the passes and conventions of oa_vks.hip):
//
//   (k_rho_xc, oa_vks.hip: sum of the rho partials, PZ-LDA   parts -> rho, v)
//   k_vx2  : x r2c                                        rho -> hx
//   k_vy2  : y FFT of the kx columns, either way          hx <-> hl (ky box)
//   k_vl2  : z FFT, Hartree + V_loc, z FFT back           hl -> hl
//   k_vxb2 : x c2r, added to V_xc                         hx -> v
//
// hx is [z][y][kx] and hl [z][ky][kx], so the lanes of every pass run along kx or
// x; the energy sums are the work of one more workgroup of the y pass back.  One
// grid per step, FP64: bound by the latency of six dependent launches with two memory
// round trips each and, at 100^3, by the 80 MB that they move.  rho and V_KS from the
// partial sums: 45^3 51 -> 30 us, 100^3 97 -> 60, 160^3 259 -> 167; in LDS Stockham
// passes with a rho and an energy sum in launches of their own before.
#pragma once

#include <algorithm>

#include "oa_fft2_kernels.h"
#include "oa_vks_point.h"

namespace oa2 {

using oa::VksArgs;

enum VKind { VX = 0, VYF, VL, VYB, VXB };  // in order of use

typedef cpx<double> cd;

// byte offset of element i, out of a buffer's range where !ok
__device__ __forceinline__ unsigned boff(bool ok, unsigned i, int size) {
  return ok ? i * (unsigned)size : 0x7fffffffu;
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ double ld8(__amdgpu_buffer_rsrc_t r, unsigned o) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0));
}
__device__ __forceinline__ cd ld16(__amdgpu_buffer_rsrc_t r, unsigned o) {
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(cd, (u4)__builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0));
}

// the twiddles of lane j's second pass, read ahead of the exchange
template <int S, int R2>
__device__ __forceinline__ void load_w(cd (&w)[R2], const double2* tw, int j) {
#pragma unroll
  for (int t = 1; t < R2; t++) w[t] = twiddle<double, S>(tw, t * j);
}

// This lane's pair of rows of all planes' (XRows: a wave takes TPW of them, a
// workgroup a.pr)
template <int R1, int R2>
struct VRow {
  int j, z, y1;
  bool active, two;
  cd* ex;
  __device__ __forceinline__ VRow(const VksArgs& a, cd* smem) {
    using X = XRows<double, R1, R2>;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, npairs = (a.ny + 1) / 2;
    const int tr = lane / X::G, p = blockIdx.x * a.pr + wave * X::TPW + tr;
    j = lane - tr * X::G;
    active = tr < X::TPW && p < npairs * a.nz;
    z = p / npairs;
    y1 = 2 * (p - z * npairs);
    two = y1 + 1 < a.ny;
    ex = smem + (wave * X::TPW + min(tr, X::TPW - 1)) * X::SZ;
  }
};

template <int R1, int R2>
__global__ __launch_bounds__(kThreads) void k_vx2(VksArgs a) {
  using X = XRows<double, R1, R2>;
  constexpr int N = X::N, G = X::G, P1 = X::P1;
  extern __shared__ __align__(16) cd smem[];
  const VRow<R1, R2> m(a, smem);
  const int j = m.j;
  const bool in = m.active && j < R2;
  const auto pr = rsrc(a.rho, (size_t)N * a.ny * a.nz * 8);
  const unsigned at = (m.z * a.ny + m.y1) * N + j;
  double r[2][R1];
#pragma unroll
  for (int t = 0; t < R1; t++)
#pragma unroll
    for (int h = 0; h < 2; h++)
      r[h][t] = ld8(pr, boff(in && (h == 0 || m.two), at + h * N + t * R2, 8));
  cd w[R2];
  load_w<-1>(w, a.twx, min(j, R1 - 1));
  const double sc = a.vol / ((double)a.nx * a.ny * a.nz);
  cd v[R1];
#pragma unroll
  for (int t = 0; t < R1; t++) v[t] = {r[0][t] * sc, r[1][t] * sc};
  Dft<double, R1, -1>::run(v);
  if (in) {
#pragma unroll
    for (int t = 0; t < R1; t++) m.ex[j * P1 + t] = v[t];
  }
  wave_lds();
  if (m.active && j < R1) {
    cd u[R2];
#pragma unroll
    for (int t = 0; t < R2; t++) u[t] = m.ex[j + t * P1];
#pragma unroll
    for (int t = 1; t < R2; t++) u[t] = cm(u[t], w[t]);
    Dft<double, R2, -1>::run(u);
    wave_lds();
#pragma unroll
    for (int t = 0; t < R2; t++) m.ex[j + t * R1] = u[t];
  }
  wave_lds();
  // Z = X_a + i X_b: X_a(k) = (Z_k + conj Z_-k)/2, X_b(k) = (Z_k - conj Z_-k)/(2i)
  if (m.active) {
    double2* o = a.hx + (size_t)(m.z * a.ny + m.y1) * a.nkx;
    for (int k = j; k < a.nkx; k += G) {
      const cd zk = m.ex[k], zm = m.ex[k == 0 ? 0 : N - k];
      o[k] = make_double2(0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y));
      if (m.two) o[a.nkx + k] = make_double2(0.5 * (zk.y + zm.y), -0.5 * (zk.x - zm.x));
    }
  }
}

template <int R1, int R2>
__global__ __launch_bounds__(kThreads) void k_vxb2(VksArgs a) {
  using X = XRows<double, R1, R2>;
  constexpr int N = X::N, P1 = X::P1;
  extern __shared__ __align__(16) cd smem[];
  const VRow<R1, R2> m(a, smem);
  const int j = m.j;
  const bool out = m.active && j < R1;
  double vx[2][R2];  // V_xc at x = j + t R1
  const auto pv = rsrc(a.v, (size_t)N * a.ny * a.nz * 8);
  const unsigned at = (m.z * a.ny + m.y1) * N + j;
#pragma unroll
  for (int t = 0; t < R2; t++)
#pragma unroll
    for (int h = 0; h < 2; h++) vx[h][t] = ld8(pv, boff(out && (h == 0 || m.two), at + h * N + t * R1, 8));
  // Z_k = X_a(k) + i X_b(k), Z_-k = conj X_a(k) + i conj X_b(k), Im of kx = 0 dropped
  const auto ph = rsrc(a.hx, (size_t)a.nkx * a.ny * a.nz * 16);
  cd v[R1];
#pragma unroll
  for (int t = 0; t < R1; t++) {
    const int k = j + t * R2, kk = k < a.nkx ? k : N - k;
    const bool ok = m.active && j < R2 && kk < a.nkx;
    const unsigned e = (m.z * a.ny + m.y1) * a.nkx + kk;
    const cd xa = ld16(ph, boff(ok, e, 16)), xb = ld16(ph, boff(ok && m.two, e + a.nkx, 16));
    const double sg = k == 0 ? 0.0 : k < a.nkx ? 1.0 : -1.0;
    v[t] = {xa.x - sg * xb.y, xb.x + sg * xa.y};
  }
  cd w[R2];
  load_w<1>(w, a.twx, min(j, R1 - 1));
  Dft<double, R1, 1>::run(v);
  if (m.active && j < R2) {
#pragma unroll
    for (int t = 0; t < R1; t++) m.ex[j * P1 + t] = v[t];
  }
  wave_lds();
  if (out) {
    cd u[R2];
#pragma unroll
    for (int t = 0; t < R2; t++) u[t] = m.ex[j + t * P1];
#pragma unroll
    for (int t = 1; t < R2; t++) u[t] = cm(u[t], w[t]);
    Dft<double, R2, 1>::run(u);
#pragma unroll
    for (int t = 0; t < R2; t++) {
      vx[0][t] += u[t].x;
      vx[1][t] += u[t].y;
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
      if (h == 1 && !m.two) break;
#pragma unroll
      for (int t = 0; t < R2; t++) a.v[at + h * N + t * R1] = vx[h][t];
      if (a.vp.p) {
        const oa::VPermRow row(a.vp, m.z, m.y1 + h);
#pragma unroll
        for (int t = 0; t < R2; t++) row.put(j + t * R1, vx[h][t]);
      }
    }
  }
}

// Columns of the y and z passes (a.cb, a.lb of them in a workgroup): lane = column,
// thread group j of a transform; element e of column col at e * ntr + col of LDS
template <int R1, int R2, int S>
__device__ __forceinline__ void col_fft(cd (&v)[R1], cd (&u)[R2], const cd (&w)[R2], cd* ex,
                                        bool active, int ntr, int col, int j) {
  if (active && j < R2) {
    Dft<double, R1, S>::run(v);
#pragma unroll
    for (int t = 0; t < R1; t++) ex[(j * R1 + t) * ntr + col] = v[t];
  }
  __syncthreads();
  if (active && j < R1) {
#pragma unroll
    for (int t = 0; t < R2; t++) u[t] = ex[(j + t * R1) * ntr + col];
#pragma unroll
    for (int t = 1; t < R2; t++) u[t] = cm(u[t], w[t]);
    Dft<double, R2, S>::run(u);
  }
}

// S = -1: hx -> hl, S = +1: hl (zero outside the ky box) -> hx, and the last
// workgroup of the grid sums the energy partials
template <int R1, int R2, int S>
__global__ __launch_bounds__(kThreads) void k_vy2(VksArgs a) {
  constexpr int N = R1 * R2, G = R1 > R2 ? R1 : R2;
  extern __shared__ __align__(16) cd ex[];
  const int ntr = a.cb, j = threadIdx.x / ntr, col = threadIdx.x - j * ntr;
  const int c = blockIdx.x * ntr + col;
  const int ncol = a.nz * a.nkx;
  if (S > 0 && (int)blockIdx.x == (ncol + ntr - 1) / ntr) {
    oa::vks_sum(a.part_x, a.nbx, a.part_l, a.nbl, a.vol / ((double)a.nx * a.ny * a.nz), a.res,
                reinterpret_cast<double*>(ex));
    return;
  }
  const bool active = c < ncol && j < G;
  const int z = c / a.nkx, kx = c - z * a.nkx;
  const auto src = S < 0 ? rsrc(a.hx, (size_t)ncol * N * 16) : rsrc(a.hl, (size_t)ncol * a.nky * 16);
  cd v[R1], u[R2], w[R2];
#pragma unroll
  for (int t = 0; t < R1; t++) {
    const int y = j + t * R2, ky = oa::sfreq(y, N) + a.kyr;
    const bool ok = active && j < R2 && (S < 0 || (ky >= 0 && ky < a.nky));
    v[t] = ld16(src, boff(ok, (z * (S < 0 ? N : a.nky) + (S < 0 ? y : ky)) * a.nkx + kx, 16));
  }
  load_w<S>(w, a.twy, min(j, R1 - 1));
  col_fft<R1, R2, S>(v, u, w, ex, active, ntr, col, j);
  if (active && j < R1) {
#pragma unroll
    for (int t = 0; t < R2; t++) {
      const int y = j + t * R1, ky = oa::sfreq(y, N) + a.kyr;
      const double2 o = make_double2(u[t].x, u[t].y);
      if (S > 0)
        a.hx[((size_t)z * N + y) * a.nkx + kx] = o;
      else if (ky >= 0 && ky < a.nky)
        a.hl[((size_t)z * a.nky + ky) * a.nkx + kx] = o;
    }
  }
}

// One column = one (kx, ky) line.  Back from kz = j + t R1, the factors in the
// other order.
template <int R1, int R2>
__global__ __launch_bounds__(kThreads) void k_vl2(VksArgs a) {
  constexpr int N = R1 * R2, G = R1 > R2 ? R1 : R2;
  extern __shared__ __align__(16) cd ex[];
  __shared__ double red[kThreads / 64 * 2];
  const int ntr = a.lb, j = threadIdx.x / ntr, col = threadIdx.x - j * ntr;
  const int l = blockIdx.x * ntr + col;
  const int nl = a.nky * a.nkx;
  const bool active = l < nl && j < G;
  const int kx = l % a.nkx, ky = l / a.nkx - a.kyr;
  const auto src = rsrc(a.hl, (size_t)nl * N * 16), pv = rsrc(a.vloc, (size_t)nl * N * 16);
  cd v[R1], u[R2], vl[R2], w[R2];
#pragma unroll
  for (int t = 0; t < R1; t++) v[t] = ld16(src, boff(active && j < R2, (j + t * R2) * nl + l, 16));
#pragma unroll
  for (int t = 0; t < R2; t++) vl[t] = ld16(pv, boff(active && j < R1, (j + t * R1) * nl + l, 16));
  load_w<-1>(w, a.twz, min(j, R1 - 1));
  col_fft<R1, R2, -1>(v, u, w, ex, active, ntr, col, j);
  const double fpi = 4.0 * 3.14159265358979323846;
  const double wt = kx == 0 ? 1.0 : 2.0;
  double acc[2] = {0.0, 0.0};
  __syncthreads();
  if (active && j < R1) {
#pragma unroll
    for (int t = 0; t < R2; t++) {
      const double g2 = oa::gsq(a.hmati, kx, ky, oa::sfreq(j + t * R1, N));
      const cd r = u[t];
      cd out = {0.0, 0.0};
      if (g2 == 0.0) {
        out = {vl[t].x, 0.0};
        acc[1] += vl[t].x * r.x;
      } else if (g2 <= a.ecut4) {
        const double hf = fpi / (g2 * a.vol);
        acc[0] += hf * (r.x * r.x + r.y * r.y) * wt;
        acc[1] += (r.x * vl[t].x + r.y * vl[t].y) * wt;  // Re(rho conj V_loc)
        out = {r.x * hf + vl[t].x, r.y * hf + vl[t].y};
      }
      u[t] = out;
    }
    Dft<double, R2, 1>::run(u);
#pragma unroll
    for (int t = 1; t < R2; t++) u[t] = cm(u[t], cd{w[t].x, -w[t].y});
#pragma unroll
    for (int t = 0; t < R2; t++) ex[(j * R2 + t) * ntr + col] = u[t];
  }
  __syncthreads();
  if (active && j < R2) {
#pragma unroll
    for (int t = 0; t < R1; t++) v[t] = ex[(j + t * R2) * ntr + col];
    Dft<double, R1, 1>::run(v);
#pragma unroll
    for (int t = 0; t < R1; t++)
      a.hl[(size_t)(j + t * R2) * nl + l] = make_double2(v[t].x, v[t].y);
  }
  oa::block_sum<2>(acc, red);
  if (threadIdx.x == 0)
    for (int i = 0; i < 2; i++) a.part_l[(size_t)blockIdx.x * 2 + i] = acc[i];
}

template <int R1, int R2>
hipError_t launch_vks(int kind, const VksArgs& a, hipStream_t st) {
  using X = XRows<double, R1, R2>;
  constexpr int N = X::N, G = X::G;
  const int rows = (a.nz * ((a.ny + 1) / 2) + a.pr - 1) / a.pr;
  const int cols = (a.nz * a.nkx + a.cb - 1) / a.cb, lines = (a.nky * a.nkx + a.lb - 1) / a.lb;
  const dim3 tx(a.pr / X::TPW * 64), ty((a.cb * G + 63) / 64 * 64), tz((a.lb * G + 63) / 64 * 64);
  const size_t sx = (size_t)a.pr * X::SZ * sizeof(cd);
  const size_t sy = std::max<size_t>(512, (size_t)a.cb * N * sizeof(cd));
  const size_t sz = (size_t)a.lb * N * sizeof(cd);
  switch (kind) {
    case VX: hipLaunchKernelGGL((k_vx2<R1, R2>), dim3(rows), tx, sx, st, a); break;
    case VYF: hipLaunchKernelGGL((k_vy2<R1, R2, -1>), dim3(cols), ty, sy, st, a); break;
    case VL: hipLaunchKernelGGL((k_vl2<R1, R2>), dim3(lines), tz, sz, st, a); break;
    case VYB: hipLaunchKernelGGL((k_vy2<R1, R2, 1>), dim3(cols + 1), ty, sy, st, a); break;
    case VXB: hipLaunchKernelGGL((k_vxb2<R1, R2>), dim3(rows), tx, sx, st, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace oa2

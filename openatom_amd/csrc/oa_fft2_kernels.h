// oa_fft2_kernels.h -- the six passes of the state FFT chain on the
// register-resident two-factor engine (oa_fft2.h).  Each kernel is a
// template on the transform length N = R1*R2 of its axis; oa_fft2_inst.hip
// instantiates one length per translation unit.
//
//   k2_zfwd : sphere gather + z-FFT (FFTW_FORWARD)  psi(G) -> zbuf[s][z][kx][ky]
//   k2_yfwd : y-FFT (FFTW_FORWARD), transposing     zbuf   -> xbuf[s][z][y][kx]
//   k2_xc2r : pair-row Hermitian x-FFT, rho         xbuf   -> rho partials
//   k2_xr2c : the same again, V psi occ, x-FFT      xbuf,V -> xout (conjugated)
//   k2_ybwd : y-FFT (FFTW_BACKWARD)                 xout   -> zbuf
//   k2_zbwd : z-FFT, pack, -2/N, kinetic force, EKE zbuf   -> F(G)
// Conventions are those of fftCache.C:460-553, 1099-1319 and
// CP_State_GSpacePlane.C:1582-1778 (see oa_fft.hip for the restatement).
#pragma once

#include "oa_fft2.h"
#include "oa_kernels.h"

namespace oa2 {

using oa::FftCtx;

constexpr int kThreads = 256;

template <int R1, int R2>
struct Shape {
  static constexpr int N = R1 * R2;
  static constexpr int G = R1 > R2 ? R1 : R2;  // threads per transform
  static constexpr int NTR = kThreads / G;     // transforms per workgroup
};

__device__ __forceinline__ int signed_k(int i, int n) { return (i <= (n - 1) / 2) ? i : i - n; }

// XCD-aware block order of a 2D grid.  The chip hands workgroups to its 8
// XCDs (each with its own L2) round-robin by linear block id, so blocks x
// and x+1 would run on different XCDs.  This map gives each XCD a
// contiguous range of logical blocks (x fastest): neighbouring line blocks,
// which share the 128-byte lines at their edges, then meet in one L2.
constexpr int kXcds = 8;
__device__ __forceinline__ void xcd_block(int& bx, int& by) {
  const int nx = gridDim.x, total = nx * gridDim.y;
  const int lin = blockIdx.x + blockIdx.y * nx;
  const int xcd = lin % kXcds, k = lin / kXcds;
  const int q = total / kXcds, r = total % kXcds;
  const int logical = xcd < r ? xcd * (q + 1) + k : r * (q + 1) + (xcd - r) * q + k;
  bx = logical % nx;
  by = logical / nx;
}

// ------------------------------------------------------------------ z passes

// PR: every stored |kz| <= (N - 1) / 4 (pruned pass 1, Sph in oa_fft2.h)
// FP32: 512 threads, so that a workgroup's stores to one z are as long as the FP64
// ones; LD: the lanes across lines meet every bank with an odd stride, one with 128 or
// 160.  Bound by the scattered runs of zbuf: 512 states of 160^3, 2.7 GB, 970 -> 864 us
// (940 with the stride alone); 100^3 and 108^3 as before.
template <typename T>
constexpr int kZThreads = sizeof(T) == 4 ? 512 : 256;
template <typename T, int R1, int R2, bool PR>
__global__ __launch_bounds__(kZThreads<T>) void k2_zfwd(FftCtx c) {
  using Sh = Shape<R1, R2>;
  constexpr int N = Sh::N, G = Sh::G, NTR = kZThreads<T> / G, LD = N | 1;
  __shared__ cpx<T> ex[NTR * LD];
  int bx, s;
  xcd_block(bx, s);
  const int l0 = bx * NTR;
  const int nl = min(NTR, c.g.nlines - l0);
  const int tid = threadIdx.x;
  // pass 2's zbuf column, loaded up front (behind pass 1)
  const int tr2 = tid % NTR, j2 = tid / NTR;
  const int w2 = c.lines[l0 + min(tr2, nl - 1)].w;
  {  // pass 1: lanes along z (contiguous sphere points)
    const int tr = tid / G, j = tid - tr * G;
    if (tr < nl && j < R2) {
      const int4 L = c.lines[l0 + tr];
      const double2* ps = c.psi + (size_t)s * c.g.ld + L.x;
      // branch-free: every load issued before any is waited for (a load in
      // a divergent branch is waited for on its own); lines hold >= 1 point
      cpx<T> v[R1];
#pragma unroll
      for (int t = 0; t < R1; t++) {
        if (Sph<N, R2>::cut(PR, t)) {
          v[t] = {(T)0, (T)0};
          continue;
        }
        const int d = signed_k(j + t * R2, N) - L.z;
        const double2 a = ps[min(max(d, 0), L.y - 1)];
        const bool in = d >= 0 && d < L.y;
        v[t] = {in ? (T)a.x : (T)0, in ? (T)a.y : (T)0};
      }
      Dft<T, R1, -1>::run(v);
#pragma unroll
      for (int t = 0; t < R1; t++) ex[tr * LD + j * R1 + t] = v[t];
    }
  }
  __syncthreads();
  {  // pass 2: lanes along lines (adjacent (kx,ky) columns of zbuf)
    const int tr = tr2, j = j2;
    if (tr < nl && j < R1) {
      cpx<T> u[R2];
#pragma unroll
      for (int t = 0; t < R2; t++) u[t] = ex[tr * LD + j + t * R1];
#pragma unroll
      for (int t = 1; t < R2; t++) u[t] = cm(u[t], twiddle<T, -1>(c.twz, t * j));
      Dft<T, R2, -1>::run(u);
      const size_t plane = (size_t)c.g.nplane_x * c.g.ny;
      cpx<T>* zs = (cpx<T>*)c.zbuf + (size_t)s * c.g.nz * plane + w2;
#pragma unroll
      for (int t = 0; t < R2; t++) zs[(size_t)(j + t * R1) * plane] = u[t];
    }
  }
}

// PR: every stored |kz| <= (N - 1) / 4 (pass-2 outputs outside it dropped)
template <typename T, int R1, int R2, bool PR>
__global__ __launch_bounds__(kThreads) void k2_zbwd(FftCtx c) {
  using Sh = Shape<R1, R2>;
  constexpr int N = Sh::N, G = Sh::G, NTR = Sh::NTR;
  constexpr int kPre = 4;  // passes over the points whose operands are loaded up front
  __shared__ cpx<T> ex[NTR * N];
  __shared__ unsigned char wt_l[NTR * N];  // per point: 1 on kx = 0 lines, 2 elsewhere
  __shared__ double red[kThreads / 64];
  int bx, s;
  xcd_block(bx, s);
  const int l0 = bx * NTR;
  const int nl = min(NTR, c.g.nlines - l0);
  const int tid = threadIdx.x;
  const size_t plane = (size_t)c.g.nplane_x * c.g.ny;
  // The workgroup's lines are one contiguous run of stored points [p0, p1):
  // the pack stage reads psi and |G|^2 and writes F along it, lanes on
  // consecutive points.  Lanes along the z of each line would store runs
  // of R1 points at arbitrary alignment, partial sectors of HBM that cost
  // more traffic than the data.
  const int p0 = c.lines[l0].x;
  const int4 Llast = c.lines[l0 + nl - 1];
  const int np = Llast.x + Llast.y - p0;  // <= nl * N
  const double2* ps = c.psi + (size_t)s * c.g.ld + p0;
  double2* fs = c.force + (size_t)s * c.g.ld + p0;
  const double* g2 = c.g2 + p0;
  // pass 2's twiddles and line, and the first pack operands, loaded up
  // front (branch-free, clamped) so that their latency hides behind pass 1
  const int tr2 = tid / G, j2 = tid - tr2 * G;
  cpx<T> tw2[R2];
#pragma unroll
  for (int t = 1; t < R2; t++) tw2[t] = twiddle<T, +1>(c.twz, t * min(j2, R1 - 1));
  const int4 L = c.lines[l0 + min(tr2, nl - 1)];
  const int w1 = c.lines[l0 + min(tid % NTR, nl - 1)].w;
  const double oc = c.occ[s];
  double gq[kPre];
  double2 cq[kPre];
#pragma unroll
  for (int i = 0; i < kPre; i++) {
    const int o = min(tid + i * kThreads, np - 1);
    gq[i] = g2[o];
    cq[i] = ps[o];
  }
  {  // pass 1: lanes along lines
    const int tr = tid % NTR, j = tid / NTR;
    if (tr < nl && j < R2) {
      const cpx<T>* zs = (const cpx<T>*)c.zbuf + (size_t)s * c.g.nz * plane + w1;
      cpx<T> v[R1];
#pragma unroll
      for (int t = 0; t < R1; t++) v[t] = zs[(size_t)(j + t * R2) * plane];
      Dft<T, R1, +1>::run(v);
#pragma unroll
      for (int t = 0; t < R1; t++) ex[tr * N + j * R1 + t] = v[t];
    }
  }
  __syncthreads();
  {  // pass 2: lanes along z; the results go back to LDS in stored-point order
    const int tr = tr2, j = j2;
    const bool act = tr < nl && j < R1;
    cpx<T> u[R2];
    if (act) {
#pragma unroll
      for (int t = 0; t < R2; t++) u[t] = ex[tr * N + j + t * R1];
#pragma unroll
      for (int t = 1; t < R2; t++) u[t] = cm(u[t], tw2[t]);
      Dft<T, R2, +1>::run(u);
    }
    __syncthreads();  // ex is rewritten below
    if (act) {
      const int ob = L.x - p0;
      const unsigned char w = (L.w < c.g.ny) ? 1 : 2;  // kx = 0 lines have dst < ny
#pragma unroll
      for (int t = 0; t < R2; t++) {
        const int d = signed_k(j + t * R1, N) - L.z;
        if (!Sph<N, R1>::cut(PR, t) && d >= 0 && d < L.y) {
          ex[ob + d] = u[t];
          wt_l[ob + d] = w;
        }
      }
    }
  }
  __syncthreads();
  // pack: -2/N scale (w doubles the kx > 0 half), kinetic force, EKE
  double eke = 0.0;
  auto pack = [&](int o, double gg, double2 cc) __attribute__((always_inline)) {
    const cpx<T> u = ex[o];
    const double w = (double)wt_l[o];
    double2 f;
    if (gg <= c.ecut_ry) {
      const double wt = oc * w * gg;
      f.x = w * (c.scale * (double)u.x) - wt * cc.x;
      f.y = w * (c.scale * (double)u.y) - wt * cc.y;
      eke += wt * (cc.x * cc.x + cc.y * cc.y);
    } else {
      f.x = 0.0;
      f.y = 0.0;
    }
    fs[o] = f;
  };
#pragma unroll
  for (int i = 0; i < kPre; i++) {
    const int o = tid + i * kThreads;
    if (o < np) pack(o, gq[i], cq[i]);
  }
  for (int o = tid + kPre * kThreads; o < np; o += kThreads) pack(o, g2[o], ps[o]);
  for (int o = 32; o > 0; o >>= 1) eke += __shfl_down(eke, o, 64);
  if ((tid & 63) == 0) red[tid >> 6] = eke;
  __syncthreads();
  if (tid == 0) {
    double tsum = 0.0;
    for (int w = 0; w < kThreads / 64; w++) tsum += red[w];
    c.eke_part[(size_t)s * gridDim.x + bx] = 0.5 * tsum;
  }
}

// ------------------------------------------------------------------ y passes

template <typename T, int R1, int R2>
__global__ __launch_bounds__(kThreads) void k2_yfwd(FftCtx c) {
  using Sh = Shape<R1, R2>;
  constexpr int N = Sh::N, G = Sh::G, NTR = Sh::NTR;
  __shared__ cpx<T> ex[NTR * N];
  const int kx0 = blockIdx.x * NTR, z = blockIdx.y, s = blockIdx.z;
  const int npx = c.g.nplane_x;
  const int nk = min(NTR, npx - kx0);
  const int tid = threadIdx.x;
  const size_t off = ((size_t)s * c.g.nz + z) * (size_t)npx * N;
  {  // pass 1: lanes along y of one column (contiguous in zbuf)
    const int tr = tid / G, j = tid - tr * G;
    if (tr < nk && j < R2) {
      const int kx = kx0 + tr;
      const int lo = c.kylo[kx], hi = c.kyhi[kx];
      const cpx<T>* src = (const cpx<T>*)c.zbuf + off + (size_t)kx * N;
      cpx<T> v[R1];
#pragma unroll
      for (int t = 0; t < R1; t++) {
        const int y = j + t * R2;
        const int kyv = signed_k(y, N);
        v[t] = (kyv >= lo && kyv <= hi) ? src[y] : cpx<T>{(T)0, (T)0};
      }
      Dft<T, R1, -1>::run(v);
#pragma unroll
      for (int t = 0; t < R1; t++) ex[tr * N + j * R1 + t] = v[t];
    }
  }
  __syncthreads();
  {  // pass 2: lanes along kx (contiguous in xbuf)
    const int tr = tid % NTR, j = tid / NTR;
    if (tr < nk && j < R1) {
      cpx<T> u[R2];
#pragma unroll
      for (int t = 0; t < R2; t++) u[t] = ex[tr * N + j + t * R1];
#pragma unroll
      for (int t = 1; t < R2; t++) u[t] = cm(u[t], twiddle<T, -1>(c.twy, t * j));
      Dft<T, R2, -1>::run(u);
      cpx<T>* dst = (cpx<T>*)c.xbuf + off + kx0 + tr;
#pragma unroll
      for (int t = 0; t < R2; t++) dst[(size_t)(j + t * R1) * npx] = u[t];
    }
  }
}

template <typename T, int R1, int R2>
__global__ __launch_bounds__(kThreads) void k2_ybwd(FftCtx c) {
  using Sh = Shape<R1, R2>;
  constexpr int N = Sh::N, G = Sh::G, NTR = Sh::NTR;
  __shared__ cpx<T> ex[NTR * N];
  const int kx0 = blockIdx.x * NTR, z = blockIdx.y, s = blockIdx.z;
  const int npx = c.g.nplane_x;
  const int nk = min(NTR, npx - kx0);
  const int tid = threadIdx.x;
  const size_t off = ((size_t)s * c.g.nz + z) * (size_t)npx * N;
  {  // pass 1: lanes along kx (contiguous in xbuf)
    const int tr = tid % NTR, j = tid / NTR;
    if (tr < nk && j < R2) {
      const cpx<T>* src = (const cpx<T>*)c.xout + off + kx0 + tr;
      cpx<T> v[R1];
#pragma unroll
      for (int t = 0; t < R1; t++) v[t] = src[(size_t)(j + t * R2) * npx];
      Dft<T, R1, +1>::run(v);
#pragma unroll
      for (int t = 0; t < R1; t++) ex[tr * N + j * R1 + t] = v[t];
    }
  }
  __syncthreads();
  {  // pass 2: lanes along y of one column
    const int tr = tid / G, j = tid - tr * G;
    if (tr < nk && j < R1) {
      cpx<T> u[R2];
#pragma unroll
      for (int t = 0; t < R2; t++) u[t] = ex[tr * N + j + t * R1];
#pragma unroll
      for (int t = 1; t < R2; t++) u[t] = cm(u[t], twiddle<T, +1>(c.twy, t * j));
      Dft<T, R2, +1>::run(u);
      const int kx = kx0 + tr;
      const int lo = c.kylo[kx], hi = c.kyhi[kx];
      cpx<T>* dst = (cpx<T>*)c.zbuf + off + (size_t)kx * N;
#pragma unroll
      for (int t = 0; t < R2; t++) {
        const int y = j + t * R1;
        const int kyv = signed_k(y, N);
        if (kyv >= lo && kyv <= hi) dst[y] = u[t];
      }
    }
  }
}

// ------------------------------------------------------------------ x passes
// Workgroup = (block of NTR pair-rows, z, chunk of states); loops over the
// chunk's states.  Lanes run along x in both passes (rows are contiguous).
// Bound by latency and then memory: the next state's coefficients are loaded while
// this one's are transformed.  96 states of 72 x 80 x 90 in FP32: G->R 150 -> 51 us,
// R->G 160 -> 83 us (105 and 210 MB), before with barriers for the whole workgroup
// between passes and psi(r) written and read.
// A wave transforms TPW pairs of rows by itself: what one lane leaves in LDS another
// lane of the same wave reads, in program order, so no barrier stands between the
// passes of a state or between states, and a wave that waits for memory holds up no
// other.
template <typename T, int R1, int R2>
struct XRows {
  static constexpr int N = R1 * R2, G = R1 > R2 ? R1 : R2;
  static constexpr int TPW = 64 / G, NTR = kThreads / 64 * TPW;
  static constexpr int P1 = R1 | 1;     // odd LDS stride of an R1-long run
  static constexpr int SZ = R2 * P1;    // >= N
};
__device__ __forceinline__ void wave_lds() {  // LDS order within a wave, for the compiler
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The two rows' coefficients of this lane (k = j + t R2): off = byte offset of
// X1[|k|] in the plane's rows or out of range (buffer loads give zero there), sg
// the sign that makes X1 +- i X2 or its mirror image of them.
template <typename T, int R1, int R2>
struct XIn {
  unsigned off[R1];
  T sg[R1];
  bool two;  // the pair has a second row
  cpx<T> a[R1], b[R1];
  __device__ __forceinline__ void init(bool active, int y1, int ny, int npx, int j) {
    constexpr int N = R1 * R2;
    two = y1 + 1 < ny;
#pragma unroll
    for (int t = 0; t < R1; t++) {
      const int k = j + t * R2, kk = k < npx ? k : N - k;
      const bool in = active && j < R2 && kk < npx;
      off[t] = in ? (unsigned)((y1 * npx + kk) * sizeof(cpx<T>)) : 0x7fffffffu;
      sg[t] = k == 0 ? (T)0 : k < npx ? (T)1 : (T)-1;
    }
  }
  __device__ __forceinline__ cpx<T> ld(__amdgpu_buffer_rsrc_t r, unsigned o, int so) {
    if constexpr (sizeof(T) == 4) {
      typedef unsigned u2 __attribute__((ext_vector_type(2)));
      return __builtin_bit_cast(cpx<T>, (u2)__builtin_amdgcn_raw_buffer_load_b64(r, o, so, 0));
    } else {
      typedef unsigned u4 __attribute__((ext_vector_type(4)));
      return __builtin_bit_cast(cpx<T>, (u4)__builtin_amdgcn_raw_buffer_load_b128(r, o, so, 0));
    }
  }
  // rows: of one state and z, bytes long
  __device__ __forceinline__ void load(const cpx<T>* rows, int bytes, int npx) {
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<cpx<T>*>(rows), (short)0, bytes, 0x00020000);
#pragma unroll
    for (int t = 0; t < R1; t++) a[t] = ld(r, off[t], 0);
#pragma unroll
    for (int t = 0; t < R1; t++)
      b[t] = ld(r, two ? off[t] + (unsigned)(npx * sizeof(cpx<T>)) : 0x7fffffffu, 0);
  }
  __device__ __forceinline__ void pairs(cpx<T> (&v)[R1]) const {
#pragma unroll
    for (int t = 0; t < R1; t++)
      v[t] = {a[t].x - sg[t] * b[t].y, b[t].x + sg[t] * a[t].y};
  }
};

// Second half of the x-FFT to real space: u[t] = the two rows at x = j + t R1
// (of the lanes j < R1), their coefficients' first pass being in v of the lanes
// j < R2
template <typename T, int R1, int R2>
__device__ __forceinline__ void x_to_real(cpx<T> (&v)[R1], cpx<T> (&u)[R2], cpx<T>* ex,
                                          const cpx<T> (&w)[R2], bool active, int j) {
  constexpr int P1 = XRows<T, R1, R2>::P1;
  Dft<T, R1, -1>::run(v);
  if (active && j < R2) {
#pragma unroll
    for (int t = 0; t < R1; t++) ex[j * P1 + t] = v[t];
  }
  wave_lds();
  if (active && j < R1) {
#pragma unroll
    for (int t = 0; t < R2; t++) u[t] = ex[j + t * P1];
  }
  wave_lds();
#pragma unroll
  for (int t = 1; t < R2; t++) u[t] = cm(u[t], w[t]);
  Dft<T, R2, -1>::run(u);
}

// PSIR: psi(r) of state c.psir_state into c.psir instead of rho partials
template <typename T, int R1, int R2, bool PSIR>
__global__ __launch_bounds__(kThreads) void k2_xc2r(FftCtx c) {
  using X = XRows<T, R1, R2>;
  constexpr int N = X::N, G = X::G, TPW = X::TPW;
  __shared__ cpx<T> smem[X::NTR * X::SZ];
  const int ny = c.g.ny, npx = c.g.nplane_x;
  const int npairs = (ny + 1) / 2;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int tr = lane / G, j = lane - tr * G;
  const int q = (blockIdx.x * (kThreads / 64) + wave) * TPW + tr;
  const int z = blockIdx.y, chunk = blockIdx.z;
  const bool active = tr < TPW && q < npairs;
  cpx<T>* ex = smem + (wave * TPW + min(tr, TPW - 1)) * X::SZ;
  const int st0 = PSIR ? c.psir_state : chunk * c.cs;
  const int st1 = PSIR ? st0 + 1 : min(c.g.nst, st0 + c.cs);
  const int y1 = 2 * q, y2 = y1 + 1;
  const size_t NP = (size_t)N * ny, plane = (size_t)ny * npx;
  const int bytes = (int)(plane * sizeof(cpx<T>));
  const cpx<T>* xb = (const cpx<T>*)c.xbuf + z * plane;
  cpx<T> w[R2];
#pragma unroll
  for (int t = 1; t < R2; t++) w[t] = twiddle<T, -1>(c.twx, t * min(j, R1 - 1));
  double acc[2 * R2];
#pragma unroll
  for (int i = 0; i < 2 * R2; i++) acc[i] = 0.0;
  XIn<T, R1, R2> in;
  in.init(active, y1, ny, npx, j);
  if (st0 < st1) in.load(xb + st0 * plane * c.g.nz, bytes, npx);
  for (int s = st0; s < st1; s++) {
    cpx<T> v[R1], u[R2];
    in.pairs(v);
    if (s + 1 < st1) in.load(xb + (s + 1) * plane * c.g.nz, bytes, npx);
    x_to_real<T, R1, R2>(v, u, ex, w, active, j);
    if constexpr (PSIR) {
      if (active && j < R1) {
        T* pr = (T*)c.psir + (size_t)z * NP;
#pragma unroll
        for (int t = 0; t < R2; t++) {
          const int x = j + t * R1;
          pr[(size_t)y1 * N + x] = u[t].x;
          if (y2 < ny) pr[(size_t)y2 * N + x] = u[t].y;
        }
      }
    } else {
      const double oc = c.occ[s];
#pragma unroll
      for (int t = 0; t < R2; t++) {
        acc[2 * t] += oc * (double)u[t].x * (double)u[t].x;
        acc[2 * t + 1] += oc * (double)u[t].y * (double)u[t].y;
      }
    }
  }
  if (!PSIR && active && j < R1) {
    double* rp = c.rho_part + (size_t)chunk * NP * c.g.nz + (size_t)z * NP;
#pragma unroll
    for (int t = 0; t < R2; t++) {
      const int x = j + t * R1;
      rp[(size_t)y1 * N + x] = acc[2 * t];
      if (y2 < ny) rp[(size_t)y2 * N + x] = acc[2 * t + 1];
    }
  }
}

// psi(r) again from xbuf, V psi, and the x-FFT back of both rows to c.xout, which
// leaves xbuf to oa_psir_get: reading nplane_x coefficients a row twice moves half
// the bytes of writing psi(r) and reading it.  The lanes hold x = j + t R1, so the
// way back takes the factors in the other order.
template <typename T, int R1, int R2>
__global__ __launch_bounds__(kThreads) void k2_xr2c(FftCtx c) {
  using X = XRows<T, R1, R2>;
  constexpr int N = X::N, G = X::G, TPW = X::TPW, P1 = X::P1;
  __shared__ cpx<T> smem[X::NTR * X::SZ];
  const int ny = c.g.ny, npx = c.g.nplane_x;
  const int npairs = (ny + 1) / 2;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int tr = lane / G, j = lane - tr * G;
  const int q = (blockIdx.x * (kThreads / 64) + wave) * TPW + tr;
  const int z = blockIdx.y, chunk = blockIdx.z;
  const bool active = tr < TPW && q < npairs;
  cpx<T>* ex = smem + (wave * TPW + min(tr, TPW - 1)) * X::SZ;
  const int st0 = chunk * c.cs_r, st1 = min(c.g.nst, st0 + c.cs_r);
  const int y1 = 2 * q, y2 = y1 + 1;
  const size_t NP = (size_t)N * ny, plane = (size_t)ny * npx;
  const int bytes = (int)(plane * sizeof(cpx<T>));
  const cpx<T>* xb = (const cpx<T>*)c.xbuf + z * plane;
  cpx<T>* xo = (cpx<T>*)c.xout + z * plane;
  cpx<T> w[R2];
#pragma unroll
  for (int t = 1; t < R2; t++) w[t] = twiddle<T, -1>(c.twx, t * min(j, R1 - 1));
  T v1[R2], v2[R2];  // V at x = j + t R1 of both rows
#pragma unroll
  for (int t = 0; t < R2; t++) {
    const double* vz = c.vks + (size_t)z * NP;
    const int x = j + t * R1;
    v1[t] = active && j < R1 ? (T)vz[(size_t)y1 * N + x] : (T)0;
    v2[t] = active && j < R1 && y2 < ny ? (T)vz[(size_t)y2 * N + x] : (T)0;
  }
  XIn<T, R1, R2> in;
  in.init(active, y1, ny, npx, j);
  if (st0 < st1) in.load(xb + st0 * plane * c.g.nz, bytes, npx);
  for (int s = st0; s < st1; s++) {
    cpx<T> v[R1], u[R2];
    in.pairs(v);
    if (s + 1 < st1) in.load(xb + (s + 1) * plane * c.g.nz, bytes, npx);
    x_to_real<T, R1, R2>(v, u, ex, w, active, j);
    const T oc = (T)c.occ[s];
#pragma unroll
    for (int t = 0; t < R2; t++) u[t] = {u[t].x * (v1[t] * oc), u[t].y * (v2[t] * oc)};
    Dft<T, R2, -1>::run(u);
#pragma unroll
    for (int t = 1; t < R2; t++) u[t] = cm(u[t], w[t]);
    if (active && j < R1) {
#pragma unroll
      for (int t = 0; t < R2; t++) ex[t * P1 + j] = u[t];
    }
    wave_lds();
    if (active && j < R2) {
#pragma unroll
      for (int t = 0; t < R1; t++) v[t] = ex[j * P1 + t];
    }
    wave_lds();
    Dft<T, R1, -1>::run(v);
    if (active && j < R2) {
#pragma unroll
      for (int t = 0; t < R1; t++) ex[j + t * R2] = v[t];
    }
    wave_lds();
    // split the two real rows and keep kx < nplane_x, conjugated
    cpx<T>* xs = xo + s * plane * c.g.nz + (size_t)y1 * npx;
    if (active) {
      for (int k = j; k < npx; k += G) {
        const cpx<T> Zk = ex[k], Zm = ex[k == 0 ? 0 : N - k];
        xs[k] = {(T)0.5 * (Zk.x + Zm.x), -(T)0.5 * (Zk.y - Zm.y)};
        if (y2 < ny) xs[npx + k] = {(T)0.5 * (Zk.y + Zm.y), (T)0.5 * (Zk.x - Zm.x)};
      }
    }
    wave_lds();
  }
}

// ------------------------------------------------------------------ launch

enum Kind { ZFWD = 0, YFWD, XC2R, XR2C, YBWD, ZBWD, XPSIR };

template <typename T, int R1, int R2>
hipError_t launch(int kind, const FftCtx& c, hipStream_t st) {
  constexpr int NZ = kZThreads<T> / Shape<R1, R2>::G;
  constexpr int NTR = Shape<R1, R2>::NTR, NX = XRows<T, R1, R2>::NTR;
  const Geom& g = c.g;
  switch (kind) {
    case ZFWD:
      if (c.prune_z)
        hipLaunchKernelGGL((k2_zfwd<T, R1, R2, true>), dim3((g.nlines + NZ - 1) / NZ, g.nst),
                           dim3(kZThreads<T>), 0, st, c);
      else
        hipLaunchKernelGGL((k2_zfwd<T, R1, R2, false>), dim3((g.nlines + NZ - 1) / NZ, g.nst),
                           dim3(kZThreads<T>), 0, st, c);
      break;
    case ZBWD:
      if (c.prune_z)
        hipLaunchKernelGGL((k2_zbwd<T, R1, R2, true>), dim3((g.nlines + NTR - 1) / NTR, g.nst),
                           dim3(kThreads), 0, st, c);
      else
        hipLaunchKernelGGL((k2_zbwd<T, R1, R2, false>), dim3((g.nlines + NTR - 1) / NTR, g.nst),
                           dim3(kThreads), 0, st, c);
      break;
    case YFWD:
      hipLaunchKernelGGL((k2_yfwd<T, R1, R2>), dim3((g.nplane_x + NTR - 1) / NTR, g.nz, g.nst),
                         dim3(kThreads), 0, st, c);
      break;
    case YBWD:
      hipLaunchKernelGGL((k2_ybwd<T, R1, R2>), dim3((g.nplane_x + NTR - 1) / NTR, g.nz, g.nst),
                         dim3(kThreads), 0, st, c);
      break;
    case XC2R:
      hipLaunchKernelGGL((k2_xc2r<T, R1, R2, false>),
                         dim3(((g.ny + 1) / 2 + NX - 1) / NX, g.nz, c.nchunk), dim3(kThreads),
                         0, st, c);
      break;
    case XR2C:
      hipLaunchKernelGGL((k2_xr2c<T, R1, R2>),
                         dim3(((g.ny + 1) / 2 + NX - 1) / NX, g.nz, c.nchunk_r), dim3(kThreads),
                         0, st, c);
      break;
    case XPSIR:
      hipLaunchKernelGGL((k2_xc2r<T, R1, R2, true>),
                         dim3(((g.ny + 1) / 2 + NX - 1) / NX, g.nz), dim3(kThreads), 0, st, c);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace oa2

// oa_plane4.h -- fused y+x plane passes by row class, for square planes whose
// populated |kx|, |ky| are <= (N - 1) / 4 (pruned grids) and N a multiple of 4.
//
// The sphere fills at most half of a plane's frequencies, so the rows
// y = M r + c of one class c (r < L = N / M) are a length-L transform of the
// folded, phase-shifted columns: an N-point y-FFT splits into M independent
// L-point ones at no extra arithmetic (M = 2), and only one class of rows has
// to be on chip at a time.  One workgroup runs, per state and class:
//
//   y forward of the columns (L = A x B, in registers with one LDS exchange),
//   whose last pass writes the pair rows Z_q[k] = X_q[k] + i X_q+L/2[k] that the
//   Hermitian x transform reads (rows q and q + L/2 of the class share one
//   complex transform);
//   x c2r (N = X1 x X2) in place in the pair-row buffer E, psi(r) in registers;
//   k4_g2r: rho accumulated in registers, one class per workgroup;
//   k4_r2g: V psi, x r2c in place, y backward whose first pass reads the pair
//   rows and separates them on the way; the classes' contributions to the
//   kept ky are summed in registers and stored once per state.
//
// What bounds it: VALU issue and the LDS pipe.  Against one pass over the
// whole plane (oa_plane3.h) a class needs half the LDS (E only: L/2 rows of N),
// which doubles the resident workgroups; every row of a class is in flight at
// once (no rounds); the x passes run in place, so an exchange costs one barrier
// and no second buffer; the x twiddles stay in registers (c2r and r2c use the
// same X2 - 1 of them: the r2c applies them on its first pass); and the pair
// rows are formed and separated by the y passes, which removes a read per
// element from the c2r and the whole separation loop after the r2c.
//
// LDS banks: lanes of the x passes are different pair rows at the same
// position and differ by the odd row stride RE = N + 1; lanes of the y passes
// that touch E are consecutive columns (stride 1).  The y exchange buffer has
// an odd column stride.  All conflict-free for 8- and 16-byte elements.
#pragma once

#include <type_traits>

#include "oa_fft2.h"
#include "oa_kernels.h"

namespace oa4 {

using oa::FftCtx;
using oa2::cm;
using oa2::Dft;

// odd column stride >= n of the y exchange buffer, a run of b lanes per
// column apart modulo 16 elements
constexpr int exch_stride(int n, int b) {
  for (int s = n | 1;; s += 2)
    if (((s - b) % 16 + 16) % 16 == 1 || ((s - b) % 16 + 16) % 16 == 15 || b % 2) return s;
}

// N = X1 x X2 along x (X2 outputs of the c2r per thread); M row classes of
// L = N / M rows; y transforms L = A x B, B even.  SEP: the y exchange buffer
// lies beside E (fewer barriers) instead of inside it (less LDS).
template <int X1_, int X2_, int M_, int A_, int B_, bool SEP_, bool TXL_ = false>
struct P4 {
  static constexpr int X1 = X1_, X2 = X2_, M = M_, A = A_, B = B_;
  static constexpr bool SEP = SEP_, TXL = TXL_;
  static constexpr int N = X1 * X2, L = N / M, NQ = L / 2;
  static constexpr int KM = (N - 1) / 4, NPX = KM + 1;
  static constexpr int NA = M / 2;  // frequencies folded onto one class input
  static constexpr int NT = (NQ * (X1 > X2 ? X1 : X2) + 63) / 64 * 64;
  static constexpr int RE = N + 1;
  static constexpr int CY = exch_stride(L, B);
  static constexpr int KSLOT = NQ * X1;
  static constexpr int KPER = M * X2 * KSLOT;
  static constexpr int ESZ = NQ * RE, XSZ = NPX * CY;
  // y passes with A threads per column: the second of the two such passes of a
  // class (y_bwd1) goes to the last waves, so that the waves share this work
  static constexpr int W2 = (NPX * A + 63) / 64 * 64;
  static constexpr int SH2 = W2 < NT ? NT - W2 : 0;
  static constexpr int ELEMS =
      (SEP ? ESZ + XSZ : (ESZ > XSZ ? ESZ : XSZ)) + N + (TXL ? N : 0);
  static_assert(N % 4 == 0 && (M == 2 || M == 4) && M * A * B == N && B % 2 == 0 && L % 2 == 0,
                "row classes need N = M A B with B even");
  static_assert(NPX * A <= NT && NPX * B <= NT, "one y item per thread");
};

template <typename T, class S>
constexpr size_t smem4() {
  return sizeof(cpx<T>) * (size_t)S::ELEMS + sizeof(int2) * S::NPX;
}

// a times exp(sign 2 pi i MM / NN), the trivial roots without a multiply
template <typename T, int SIGN, int MM, int NN>
__device__ __forceinline__ cpx<T> rot(cpx<T> a) {
  constexpr int m = ((MM % NN) + NN) % NN;
  if constexpr (m == 0) return a;
  else if constexpr (2 * m == NN) return {-a.x, -a.y};
  else if constexpr (4 * m == NN) return {-(T)SIGN * a.y, (T)SIGN * a.x};
  else if constexpr (4 * m == 3 * NN) return {(T)SIGN * a.y, -(T)SIGN * a.x};
  else {
    constexpr oa2::TwTab<NN> tw = oa2::make_tw<NN>();
    const cpx<T> w = {(T)tw.c[m], (T)(SIGN * tw.s[m])};
    return cm(a, w);
  }
}

template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// x items: thread j of pair row q (rows fastest over the lanes); the pass with
// X2 threads per row uses j < X2, the one with X1 threads j < X1
template <class S>
struct XItem {
  int q, j;
  __device__ __forceinline__ XItem() {
    const int t = (int)threadIdx.x;
    j = t / S::NQ;
    q = t - j * S::NQ;
  }
};

// Per-thread geometry and tables of one kernel.
template <typename T, class S>
struct Lane {
  unsigned off[S::NA][S::A];  // byte offset in a zbuf plane of each folded column input
  bool in[S::NA][S::A];       // populated (else off is a zero element of the plane)
  cpx<T> tx[S::TXL ? 1 : S::X2 - 1];  // W_N^{t j2}, t = 1 .. X2 - 1
  const cpx<T>* txl;                  // ... or their LDS table
};

template <typename T, class S>
__device__ __forceinline__ void lane_init(Lane<T, S>& l, const FftCtx& c, const int2* KY,
                                          const cpx<T>* TX, int npx) {
  const int tid = threadIdx.x, jx = min(tid / S::NQ, S::X1 - 1);
  const int col = tid / S::B, j = tid - col * S::B;
  const int cc = min(col, npx - 1);
  const int lo = KY[cc].x, hi = KY[cc].y;
#pragma unroll
  for (int t = 0; t < S::A; t++) {
    const int n = j + t * S::B;
#pragma unroll
    for (int a = 0; a < S::NA; a++) {
      const bool neg = S::NA == 1 ? n >= S::L / 2 : a == 1;
      const int ky = neg ? n - S::L : n, y = neg ? n + S::N - S::L : n;
      l.in[a][t] = col < npx && ky >= lo && ky <= hi;
      l.off[a][t] = (unsigned)((cc * S::N + (l.in[a][t] ? y : S::N / 2)) * sizeof(cpx<T>));
    }
  }
  l.txl = TX;
  if (!S::TXL) {
#pragma unroll
    for (int t = 1; t < S::X2; t++) {
      const double2 w = c.twx[t * jx];
      l.tx[S::TXL ? 0 : t - 1] = {(T)w.x, (T)w.y};
    }
  }
}

template <typename T, class S>
__device__ __forceinline__ cpx<T> tx_at(const Lane<T, S>& l, int j, int t) {
  return S::TXL ? l.txl[j * S::X2 + t] : l.tx[S::TXL ? 0 : t - 1];
}

// tables: TY[C][j B + t] = W_N^{t (M j + C)} and the columns' ky ranges
template <typename T, class S>
__device__ __forceinline__ void load_tables(cpx<T>* TY, int2* KY, const FftCtx& c, int npx) {
  for (int i = threadIdx.x; i < S::N; i += S::NT) {
    const int cl = i / S::L, r = i - cl * S::L, j = r / S::B, t = r - j * S::B;
    const double2 w = c.twx[t * (S::M * j + cl)];
    TY[i] = {(T)w.x, (T)w.y};
    if (S::TXL) {  // TX[j X2 + t] = W_N^{t j}
      const int jx = i / S::X2, tt = i - jx * S::X2;
      const double2 v = c.twx[tt * jx];
      TY[S::N + i] = {(T)v.x, (T)v.y};
    }
  }
  for (int i = threadIdx.x; i < S::NPX; i += S::NT)
    KY[i] = i < npx ? make_int2(c.kylo[i], c.kyhi[i]) : make_int2(1, 0);
}

// p at a byte offset.  p is uniform and the offset a 32-bit register, opaque
// here so that it is widened in this block, where the compiler can fold it
// into the access (scalar base + vector offset) instead of adding 64 bits.
template <typename P>
__device__ __forceinline__ P* at_byte(P* p, unsigned o) {
  asm volatile("" : "+v"(o));
  using B = std::conditional_t<std::is_const_v<P>, const char, char>;
  return reinterpret_cast<P*>(reinterpret_cast<B*>(p) + o);
}

template <typename T, class S>
using Raw = cpx<T>[S::NA][S::A];

// the folded column inputs of one state: unconditional loads, those outside a
// column's populated range from its row N/2, which no stored |ky| reaches and
// the context keeps zero, so nothing is masked
template <typename T, class S>
__device__ __forceinline__ void load_raw(const cpx<T>* __restrict__ zs, const Lane<T, S>& l,
                                         Raw<T, S>& raw) {
#pragma unroll
  for (int a = 0; a < S::NA; a++)
#pragma unroll
    for (int t = 0; t < S::A; t++) raw[a][t] = *at_byte(zs, l.off[a][t]);
}

// y forward, first pass, class C: DFT-A of the folded inputs n = j + t B
template <typename T, class S, int C>
__device__ __forceinline__ void y_fwd1(const Lane<T, S>& l, const Raw<T, S>& raw, cpx<T>* X) {
  const int i = (int)threadIdx.x, col = i / S::B, j = i - col * S::B;
  cpx<T>* x = X + min(col, S::NPX - 1) * S::CY + j;
  cpx<T> v[S::A];
  static_for<0, S::A>([&](auto tc) __attribute__((always_inline)) {
    constexpr int t = decltype(tc)::value;
    cpx<T> f = raw[0][t];
    if constexpr (S::NA == 2) {
      cpx<T> y = raw[S::NA - 1][t];
      y = rot<T, +1, C, S::M>(y);
      f = {f.x + y.x, f.y + y.y};
    } else if constexpr (C == 1) {
      // n >= L/2 stands for n - L, whose phase has the opposite sign
      constexpr int lo = t * S::B, hi = lo + S::B - 1;
      if constexpr (lo >= S::L / 2) {
        f = {-f.x, -f.y};
      } else if constexpr (hi >= S::L / 2) {
        const bool neg = j >= S::L / 2 - lo;
        f = {neg ? -f.x : f.x, neg ? -f.y : f.y};
      }
    }
    v[t] = rot<T, -1, t * C, S::M * S::A>(f);
  });
  Dft<T, S::A, -1>::run(v);
  if (S::NT == S::NPX * S::B || i < S::NPX * S::B)
#pragma unroll
    for (int t = 0; t < S::A; t++) x[t * S::B] = v[t];
}

// y forward, second pass: DFT-B, then the pair rows (q, q + L/2) into E
template <typename T, class S>
__device__ __forceinline__ void y_fwd2(const cpx<T>* X, cpx<T>* E, const cpx<T>* TYC) {
  cpx<T> u[S::B];
  const int jy = (int)threadIdx.x / S::NPX, col = (int)threadIdx.x - jy * S::NPX;
  if (jy < S::A) {
    const cpx<T>* x = X + col * S::CY + jy * S::B;
    cpx<T> w[S::B];
#pragma unroll
    for (int t = 0; t < S::B; t++) u[t] = x[t];
#pragma unroll
    for (int t = 1; t < S::B; t++) w[t] = TYC[jy * S::B + t];
    Dft<T, S::B, -1>::template run_tw<true>(u, w);
  }
  if (!S::SEP) __syncthreads();
  if (jy < S::A) {
    // kx = 0: Im dropped (c2r); both writes then hit position 0
    cpx<T>* ek = E + jy * S::RE + col;
    cpx<T>* em = E + jy * S::RE + (col == 0 ? 0 : S::N - col);
    const T im = col == 0 ? (T)0 : (T)1;
#pragma unroll
    for (int t = 0; t < S::B / 2; t++) {
      const cpx<T> a = u[t], b = u[t + S::B / 2];
      ek[t * S::A * S::RE] = {oa2::fm(-im, b.y, a.x), oa2::fm(im, a.y, b.x)};
      em[t * S::A * S::RE] = {oa2::fm(im, b.y, a.x), oa2::fm(-im, a.y, b.x)};
    }
  }
}

// x c2r, first pass, in place: thread j of a row owns the positions j + t X2
template <typename T, class S>
__device__ __forceinline__ void c2r1(cpx<T>* E) {
  const XItem<S> m;
  if (m.j < S::X2) {
    cpx<T>* e = E + m.q * S::RE + m.j;
    cpx<T> v[S::X1];
    static_for<0, S::X1>([&](auto tc) __attribute__((always_inline)) {
      constexpr int t = decltype(tc)::value;
      constexpr int lo = t * S::X2, hi = lo + S::X2 - 1;
      if constexpr (lo > S::KM && hi < S::N - S::KM) {
        v[t] = {(T)0, (T)0};
      } else {
        v[t] = e[lo];
        if constexpr (!(hi <= S::KM || lo >= S::N - S::KM)) {
          const int k = m.j + lo;
          if (k > S::KM && k < S::N - S::KM) v[t] = {(T)0, (T)0};
        }
      }
    });
    Dft<T, S::X1, -1>::run(v);
#pragma unroll
    for (int t = 0; t < S::X1; t++) e[t * S::X2] = v[t];
  }
}

// x c2r, second pass: psi(r) at x = j2 + t X1 of the rows q (real part) and
// q + L/2 (imaginary part)
template <typename T, class S>
__device__ __forceinline__ void c2r2(const Lane<T, S>& l, const cpx<T>* E, cpx<T> (&u)[S::X2]) {
  const XItem<S> m;
  const cpx<T>* f = E + m.q * S::RE + m.j * S::X2;
#pragma unroll
  for (int t = 0; t < S::X2; t++) u[t] = f[t];
  cpx<T> w[S::X2];
#pragma unroll
  for (int t = 1; t < S::X2; t++) w[t] = tx_at<T, S>(l, m.j, t);
  Dft<T, S::X2, -1>::template run_tw<true>(u, w);
}

// x r2c: first pass in the same lanes and slots, then the second pass
template <typename T, class S>
__device__ __forceinline__ void r2c1(const Lane<T, S>& l, cpx<T>* E, cpx<T> (&w)[S::X2]) {
  Dft<T, S::X2, -1>::run(w);
  const XItem<S> m;
  cpx<T>* f = E + m.q * S::RE + m.j * S::X2;
  f[0] = w[0];
#pragma unroll
  for (int t = 1; t < S::X2; t++) f[t] = cm(w[t], tx_at<T, S>(l, m.j, t));
}

template <typename T, class S>
__device__ __forceinline__ void r2c2(cpx<T>* E) {
  const XItem<S> m;
  if (m.j < S::X2) {
    cpx<T>* e = E + m.q * S::RE + m.j;
    cpx<T> v[S::X1];
#pragma unroll
    for (int t = 0; t < S::X1; t++) v[t] = e[t * S::X2];
    Dft<T, S::X1, -1>::run(v);
    static_for<0, S::X1>([&](auto tc) __attribute__((always_inline)) {
      constexpr int t = decltype(tc)::value;
      constexpr int lo = t * S::X2, hi = lo + S::X2 - 1;
      if constexpr (!(lo > S::KM && hi < S::N - S::KM)) e[lo] = v[t];
    });
  }
}

// y backward, first pass: separate the pair rows (twice their values: the
// caller scales by one half), DFT-B over the rows j + t A
template <typename T, class S>
__device__ __forceinline__ void y_bwd1(const cpx<T>* E, cpx<T>* X) {
  cpx<T> v[S::B];
  const int i = (int)threadIdx.x - S::SH2;
  const int jy = i < 0 ? S::A : i / S::NPX, col = i - jy * S::NPX;
  if (jy < S::A) {
    const cpx<T>* ek = E + jy * S::RE + col;
    const cpx<T>* em = E + jy * S::RE + (col == 0 ? 0 : S::N - col);
#pragma unroll
    for (int t = 0; t < S::B / 2; t++) {
      const cpx<T> zk = ek[t * S::A * S::RE], zm = em[t * S::A * S::RE];
      v[t] = {zk.x + zm.x, zm.y - zk.y};
      v[t + S::B / 2] = {zk.y + zm.y, zk.x - zm.x};
    }
    Dft<T, S::B, +1>::run(v);
  }
  if (!S::SEP) __syncthreads();
  if (jy < S::A) {
    cpx<T>* x = X + col * S::CY + jy * S::B;
#pragma unroll
    for (int t = 0; t < S::B; t++) x[t] = v[t];
  }
}

// y backward, second pass, class C: DFT-A, the class's phases, added to the
// kept frequencies
template <typename T, class S, int C>
__device__ __forceinline__ void y_bwd2(const cpx<T>* X, const cpx<T>* TY, Raw<T, S>& D) {
  const int i = (int)threadIdx.x, col = i / S::B, k0 = i - col * S::B;
  const cpx<T>* x = X + min(col, S::NPX - 1) * S::CY + k0;
  cpx<T> u[S::A], w[S::A];
#pragma unroll
  for (int j = 0; j < S::A; j++) {
    u[j] = x[j * S::B];
    if (C > 0 || j > 0) {
      w[j] = TY[C * S::L + j * S::B + k0];
      w[j].y = -w[j].y;
    }
  }
  Dft<T, S::A, +1>::template run_tw<C == 0>(u, w);
  static_for<0, S::A>([&](auto kc) __attribute__((always_inline)) {
    constexpr int k1 = decltype(kc)::value;
    cpx<T> f = rot<T, +1, k1 * C, S::M * S::A>(u[k1]);
    if constexpr (S::NA == 2) {
      const cpx<T> y = rot<T, -1, C, S::M>(f);
      cpx<T>& d1 = D[S::NA - 1][k1];
      if constexpr (C == 0) d1 = y;
      else d1 = {d1.x + y.x, d1.y + y.y};
    } else if constexpr (C == 1) {
      constexpr int lo = k1 * S::B, hi = lo + S::B - 1;
      if constexpr (lo >= S::L / 2) {
        f = {-f.x, -f.y};
      } else if constexpr (hi >= S::L / 2) {
        const bool neg = k0 >= S::L / 2 - lo;
        f = {neg ? -f.x : f.x, neg ? -f.y : f.y};
      }
    }
    cpx<T>& d0 = D[0][k1];
    if constexpr (C == 0) d0 = f;
    else d0 = {d0.x + f.x, d0.y + f.y};
  });
}

// the row of pair q of class c that the real part carries; the imaginary part
// carries the row N / 2 further
template <class S>
__device__ __forceinline__ int row1(int q, int c) {
  return S::M * q + c;
}

// G->R plane pass.  One workgroup per (z-plane, state chunk, class); blocks go
// to the 8 XCDs round-robin, and the M classes of a (plane, chunk), which read
// the same columns, sit 8 blocks apart: on one XCD, at the same time.  PSIR:
// write psi(r) of state c.psir_state into c.psir instead of rho partials.
// KEEP: also write psi(r) to c.psk.
template <typename T, class S, bool PSIR, bool KEEP, int MINW>
__global__ __launch_bounds__(S::NT, MINW) void k4_g2r(FftCtx c) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int N = S::N;
  const int npx = c.g.nplane_x;
  cpx<T>* E = reinterpret_cast<cpx<T>*>(smem_raw);
  cpx<T>* X = S::SEP ? E + S::ESZ : E;
  cpx<T>* TY = E + (S::ELEMS - N - (S::TXL ? N : 0));
  int2* KY = reinterpret_cast<int2*>(E + S::ELEMS);
  const int grp = blockIdx.x / (8 * S::M), r8 = blockIdx.x - grp * (8 * S::M);
  const int cls = r8 >> 3, unit = grp * 8 + (r8 & 7), nchunk = PSIR ? 1 : c.nchunk;
  if (unit >= c.g.nz * nchunk) return;
  const int chunk = unit / c.g.nz, z = unit - chunk * c.g.nz;
  const int st0 = PSIR ? c.psir_state : chunk * c.cs;
  const int st1 = PSIR ? st0 + 1 : min(c.g.nst, st0 + c.cs);
  const size_t plane = (size_t)npx * N, zst = plane * c.g.nz;
  load_tables<T, S>(TY, KY, c, npx);
  __syncthreads();
  Lane<T, S> l;
  lane_init<T, S>(l, c, KY, TY + N, npx);
  const cpx<T>* zs = (const cpx<T>*)c.zbuf + (size_t)st0 * zst + (size_t)z * plane;
  double acc[2 * S::X2];
#pragma unroll
  for (int b = 0; b < 2 * S::X2; b++) acc[b] = 0.0;
  Raw<T, S> raw;
  load_raw<T, S>(zs, l, raw);
  for (int s = st0; s < st1; s++) {
    const double oc = c.occ[s];
    if (!S::SEP) __syncthreads();  // E is read by the previous state's last pass
    static_for<0, S::M>([&](auto cc) __attribute__((always_inline)) {
      constexpr int C = decltype(cc)::value;
      if (cls == C) y_fwd1<T, S, C>(l, raw, X);
    });
    zs += s + 1 < st1 ? zst : 0;
    load_raw<T, S>(zs, l, raw);  // the next state's columns
    __syncthreads();
    y_fwd2<T, S>(X, E, TY + cls * S::L);
    __syncthreads();
    c2r1<T, S>(E);
    __syncthreads();
    if ((int)threadIdx.x < S::KSLOT) {
      cpx<T> u[S::X2];
      c2r2<T, S>(l, E, u);
      if (KEEP) {
        cpx<T>* kp = (cpx<T>*)c.psk +
                     (((size_t)s * c.g.nz + z) * S::M + cls) * (S::X2 * S::KSLOT) + threadIdx.x;
#pragma unroll
        for (int t = 0; t < S::X2; t++) kp[t * S::KSLOT] = u[t];
      }
      if (PSIR) {
        const XItem<S> m;
        T* pr = (T*)c.psir + ((size_t)z * N + row1<S>(m.q, cls)) * N + m.j;
#pragma unroll
        for (int t = 0; t < S::X2; t++) {
          pr[t * S::X1] = u[t].x;
          pr[(size_t)N * (N / 2) + t * S::X1] = u[t].y;
        }
      } else {
#pragma unroll
        for (int t = 0; t < S::X2; t++) {
          acc[2 * t] += oc * (double)u[t].x * (double)u[t].x;
          acc[2 * t + 1] += oc * (double)u[t].y * (double)u[t].y;
        }
      }
    }
  }
  if (PSIR || (int)threadIdx.x >= S::KSLOT) return;
  const XItem<S> m;
  double* rp = c.rho_part + (((size_t)chunk * c.g.nz + z) * N + row1<S>(m.q, cls)) * N + m.j;
#pragma unroll
  for (int t = 0; t < S::X2; t++) {
    rp[t * S::X1] = acc[2 * t];
    rp[(size_t)N * (N / 2) + t * S::X1] = acc[2 * t + 1];
  }
}

// R->G plane pass.  Grid (nz, state chunks), all classes per workgroup.  V comes
// from c.vperm ([nz][M][X2][KSLOT] pairs of rows in this pass's lane order);
// VREG holds it in registers over the chunk.  RHO: also rho partials of the
// chunk.  KEEP: psi(r) is read back from c.psk instead of recomputed.
template <typename T, class S, bool VREG, bool RHO, bool KEEP, int MINW>
__global__ __launch_bounds__(S::NT, MINW) void k4_r2g(FftCtx c) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int N = S::N;
  const int npx = c.g.nplane_x;
  cpx<T>* E = reinterpret_cast<cpx<T>*>(smem_raw);
  cpx<T>* X = S::SEP ? E + S::ESZ : E;
  cpx<T>* TY = E + (S::ELEMS - N - (S::TXL ? N : 0));
  int2* KY = reinterpret_cast<int2*>(E + S::ELEMS);
  const int z = blockIdx.x, chunk = blockIdx.y;
  const int st0 = chunk * c.cs_r, st1 = min(c.g.nst, st0 + c.cs_r);
  if (st0 >= st1) return;
  const size_t plane = (size_t)npx * N, zst = plane * c.g.nz;
  load_tables<T, S>(TY, KY, c, npx);
  __syncthreads();
  Lane<T, S> l;
  lane_init<T, S>(l, c, KY, TY + N, npx);
  const int slot = min((int)threadIdx.x, S::KSLOT - 1);
  const cpx<T>* vp = (const cpx<T>*)c.vperm + (size_t)z * S::KPER + slot;
  cpx<T> vr[VREG ? S::M : 1][VREG ? S::X2 : 1];
  if (VREG) {
#pragma unroll
    for (int cl = 0; cl < S::M; cl++)
#pragma unroll
      for (int t = 0; t < S::X2; t++)
        vr[VREG ? cl : 0][VREG ? t : 0] = vp[(cl * S::X2 + t) * S::KSLOT];
  }
  double acc[RHO ? S::M : 1][RHO ? 2 * S::X2 : 1];
  if (RHO) {
#pragma unroll
    for (int cl = 0; cl < S::M; cl++)
#pragma unroll
      for (int b = 0; b < 2 * S::X2; b++) acc[RHO ? cl : 0][RHO ? b : 0] = 0.0;
  }
  size_t zo = (size_t)st0 * zst + (size_t)z * plane;
  const cpx<T>* zb = (const cpx<T>*)c.zbuf;
  Raw<T, S> raw;
  if (!KEEP) load_raw<T, S>(zb + zo, l, raw);
  for (int s = st0; s < st1; s++) {
    Raw<T, S> D;
    static_for<0, S::M>([&](auto cc) __attribute__((always_inline)) {
      constexpr int C = decltype(cc)::value;
      cpx<T> u[S::X2];
      __syncthreads();  // the exchange buffer is read by the previous class's last pass
      if (KEEP) {
        const cpx<T>* kp = (const cpx<T>*)c.psk +
                           (((size_t)s * c.g.nz + z) * S::M + C) * (S::X2 * S::KSLOT) + slot;
#pragma unroll
        for (int t = 0; t < S::X2; t++) u[t] = kp[t * S::KSLOT];
      } else {
        y_fwd1<T, S, C>(l, raw, X);
        __syncthreads();
        y_fwd2<T, S>(X, E, TY + C * S::L);
        __syncthreads();
        c2r1<T, S>(E);
      }
      cpx<T> vv[VREG ? 1 : S::X2];
      if (!VREG) {  // this class's V, behind the barrier and the transform
#pragma unroll
        for (int t = 0; t < S::X2; t++) vv[VREG ? 0 : t] = vp[(C * S::X2 + t) * S::KSLOT];
      }
      if (!KEEP) __syncthreads();
      if ((int)threadIdx.x < S::KSLOT) {
        if (!KEEP) c2r2<T, S>(l, E, u);
        if (RHO) {
          const double od = c.occ[s];
#pragma unroll
          for (int t = 0; t < S::X2; t++) {
            double& a0 = acc[RHO ? C : 0][RHO ? 2 * t : 0];
            double& a1 = acc[RHO ? C : 0][RHO ? 2 * t + 1 : 0];
            a0 += od * (double)u[t].x * (double)u[t].x;
            a1 += od * (double)u[t].y * (double)u[t].y;
          }
        }
#pragma unroll
        for (int t = 0; t < S::X2; t++) {
          const cpx<T> v = VREG ? vr[VREG ? C : 0][VREG ? t : 0] : vv[VREG ? 0 : t];
          u[t] = {u[t].x * v.x, u[t].y * v.y};
        }
        r2c1<T, S>(l, E, u);
      }
      __syncthreads();
      r2c2<T, S>(E);
      // the columns of the next class or state, loaded here so that they are
      // not live in the x passes
      if (!KEEP) load_raw<T, S>(zb + zo + (C == S::M - 1 && s + 1 < st1 ? zst : 0), l, raw);
      __syncthreads();
      y_bwd1<T, S>(E, X);
      __syncthreads();
      y_bwd2<T, S, C>(X, TY, D);
    });
    const T sc = (T)(0.5 * c.occ[s]);  // one half from the pair rows
    cpx<T>* out = (cpx<T>*)c.zout + zo;
#pragma unroll
    for (int a = 0; a < S::NA; a++)
#pragma unroll
      for (int t = 0; t < S::A; t++)
        if (l.in[a][t]) *at_byte(out, l.off[a][t]) = {D[a][t].x * sc, D[a][t].y * sc};
    zo += zst;
  }
  if (!RHO || (int)threadIdx.x >= S::KSLOT) return;
  const XItem<S> m;
  double* rp = c.rho_part + (((size_t)chunk * c.g.nz + z) * N + row1<S>(m.q, 0)) * N + m.j;
#pragma unroll
  for (int cl = 0; cl < S::M; cl++)
#pragma unroll
    for (int t = 0; t < S::X2; t++) {
      rp[(size_t)cl * N + t * S::X1] = acc[RHO ? cl : 0][RHO ? 2 * t : 0];
      rp[(size_t)(cl + N / 2) * N + t * S::X1] = acc[RHO ? cl : 0][RHO ? 2 * t + 1 : 0];
    }
}

// ------------------------------------------------------------------ launch

// Row classes of a compiled length N = R1 x R2 (R1 <= R2; x as R2 x R1) and the
// y factors A x B of a class; lengths that are no multiple of 4 have none.
// FP64 planes of 160 points run four classes: two need 640 threads, whose
// 168 registers the FP64 passes exceed.
template <int N, bool FP64>
struct Cls {
  static constexpr int M = 0, A = 1, B = 1;
};
#define OA_CLS(n, m, a, b, f)                       \
  template <>                                       \
  struct Cls<n, f> {                                \
    static constexpr int M = m, A = a, B = b;       \
  };
#define OA_CLS2(n, a, b) OA_CLS(n, 2, a, b, false) OA_CLS(n, 2, a, b, true)
OA_CLS2(24, 3, 4)
OA_CLS2(32, 4, 4)
OA_CLS2(36, 3, 6)
OA_CLS2(40, 5, 4)
OA_CLS2(48, 4, 6)
OA_CLS2(60, 5, 6)
OA_CLS2(64, 4, 8)
OA_CLS2(72, 6, 6)
OA_CLS2(80, 5, 8)
OA_CLS2(96, 6, 8)
OA_CLS2(100, 5, 10)
OA_CLS2(108, 9, 6)
OA_CLS2(120, 6, 10)
OA_CLS2(128, 8, 8)
OA_CLS2(144, 9, 8)
OA_CLS(160, 2, 8, 10, false)
OA_CLS(160, 4, 5, 8, true)
#undef OA_CLS2
#undef OA_CLS

// Shapes of the two passes, each the fastest of the variants measured (us, 128
// states at 100^3, 64 states otherwise; exchange buffer inside E / beside E,
// x twiddles in registers / in LDS):
//   FP32: beside E, registers.  G->R 92 / 93 at 100, 91 / 85 at 108; R->G
//     153 / 153 at 100.  Above 108 points the R->G pass's x twiddles go to LDS
//     (160: 409 us in registers, 404 in LDS; without the classes 737).
//   FP64: inside E (half the LDS).  G->R: x twiddles in LDS where a third
//     workgroup then fits the registers (up to 256 threads: 152 / 142 at 100;
//     195 / 199 at 128).  R->G: in registers (273 / 293 at 100, 308 / 307 at
//     128).  Without the classes: G->R 186 and 378, R->G 372 and 745.
template <typename T, int X1, int X2>
struct Shapes {
  static constexpr int N = X1 * X2;
  static constexpr bool D = sizeof(T) == 8;
  using C = Cls<N, D>;
  using P0 = P4<X1, X2, C::M, C::A, C::B, false>;
  using G = P4<X1, X2, C::M, C::A, C::B, !D, D && P0::NT <= 256>;
  using R = P4<X1, X2, C::M, C::A, C::B, !D, !D && (N > 108)>;
  // waves per SIMD the registers are limited for
  static constexpr int WG = D ? (P0::NT <= 256 ? 3 : 2) : 4;
  static constexpr int WR = D ? 2 : 3;
  static constexpr bool VREG = !D;
};

// rho accumulation beside the R->G pass: at most 40 FP64 accumulators
template <typename T, int X1, int X2>
constexpr bool rho_ok4() {
  using H = Shapes<T, X1, X2>;
  return H::R::M * X2 <= 20 && H::R::NT <= 256;
}

enum PlaneKind { G2R = 0, R2G = 1, G2R_PSIR = 2, R2G_RHO = 3 };

template <typename T, int X1, int X2>
hipError_t launch_plane4(int kind, const FftCtx& c, hipStream_t st) {
  using H = Shapes<T, X1, X2>;
  using G = typename H::G;
  using R = typename H::R;
  constexpr int N = H::N;
  if (c.g.nx != N || c.g.ny != N || c.g.nplane_x > G::NPX) return hipErrorInvalidValue;
  constexpr size_t sg = smem4<T, G>(), sr = smem4<T, R>();
  void (*fn)(FftCtx) = nullptr;
  const bool g2r = kind == G2R || kind == G2R_PSIR;
  switch (kind) {
    case G2R:  // c.psk set: the KEEP variant also writes psi(r) for the R->G pass
      fn = c.psk ? k4_g2r<T, G, false, true, H::WG> : k4_g2r<T, G, false, false, H::WG>;
      break;
    case G2R_PSIR:
      fn = k4_g2r<T, G, true, false, H::WG>;
      break;
    case R2G:  // c.psk set: psi(r) read back from the G->R pass's KEEP output
      if (!c.vperm) return hipErrorInvalidValue;
      fn = c.psk ? k4_r2g<T, R, H::VREG, false, true, H::WR>
                 : k4_r2g<T, R, H::VREG, false, false, H::WR>;
      break;
    case R2G_RHO:
      if (!c.vperm) return hipErrorInvalidValue;
      if constexpr (rho_ok4<T, X1, X2>()) fn = k4_r2g<T, R, H::VREG, true, false, 1>;
      break;
    default:
      break;
  }
  if (!fn) return hipErrorInvalidValue;
  const size_t sm = g2r ? sg : sr;
  if (const hipError_t e = oa::grant_lds((const void*)fn, sm); e != hipSuccess) return e;
  if (g2r) {
    const int units = c.g.nz * (kind == G2R_PSIR ? 1 : c.nchunk);
    hipLaunchKernelGGL(fn, dim3((units + 7) / 8 * 8 * G::M), dim3(G::NT), sm, st, c);
  } else {
    hipLaunchKernelGGL(fn, dim3(c.g.nz, c.nchunk_r), dim3(R::NT), sm, st, c);
  }
  return hipGetLastError();
}

// workgroups per plane of the G->R grid and resident workgroups per CU
template <typename T, int X1, int X2>
hipError_t plane4_info(int* rowparts, int* occ_g2r, int* occ_r2g, int* rho_ok) {
  using H = Shapes<T, X1, X2>;
  using G = typename H::G;
  using R = typename H::R;
  constexpr size_t sg = smem4<T, G>(), sr = smem4<T, R>();
  *rowparts = G::M;
  const bool want = *rho_ok != 0;
  *rho_ok = 0;
  const void* g = (const void*)k4_g2r<T, G, false, false, H::WG>;
  const void* r = (const void*)k4_r2g<T, R, H::VREG, false, false, H::WR>;
  hipError_t e;
  if ((e = oa::grant_lds(g, sg)) != hipSuccess || (e = oa::grant_lds(r, sr)) != hipSuccess)
    return e;
  if constexpr (rho_ok4<T, X1, X2>()) {
    if (want) {
      const void* h = (const void*)k4_r2g<T, R, H::VREG, true, false, 1>;
      if ((e = oa::grant_lds(h, sr)) != hipSuccess ||
          (e = hipOccupancyMaxActiveBlocksPerMultiprocessor(rho_ok, h, R::NT, sr)) != hipSuccess)
        return e;
      *rho_ok = *rho_ok > 1 ? *rho_ok : 1;
    }
  }
  if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(occ_g2r, g, G::NT, sg)) != hipSuccess)
    return e;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ_r2g, r, R::NT, sr);
}

}  // namespace oa4

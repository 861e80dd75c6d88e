// oa_fft2.h -- register-resident two-factor FFT engine for the state FFTs.
//
// A length N = R1*R2 transform is done by a group of max(R1, R2) threads:
//   pass 1: thread j (< R2) holds x[j + t*R2] (t < R1) in registers and runs
//           a radix-R1 DFT; its outputs land at j*R1 + t of an LDS buffer;
//   pass 2: thread j' (< R1) reads buf[j' + t*R1] (t < R2), multiplies by
//           W_N^{t j'} and runs a radix-R2 DFT; X[j' + t*R1] is the result
//           in natural order (the two Stockham passes with Ns = 1, R1).
// One LDS exchange per transform.  The thread -> (transform, j) map of each
// pass is chosen per kernel so that the global loads and stores of that pass
// are contiguous across lanes.  Radix-R DFTs up to 16 are unrolled in
// registers: 2, 3, 4, 5 directly, composites of coprime factors by the
// prime-factor map (no twiddles), the others as P x Q Cooley-Tukey with
// compile-time twiddles.
#pragma once

#include "oa_common.h"

namespace oa2 {

using ::cpx;

// ---------------------------------------------------------------- constants
constexpr double kTwoPi = 6.283185307179586476925286766559;

constexpr double ct_sin_small(double x) {  // |x| <= pi/4
  double x2 = x * x, term = x, sum = x;
  for (int k = 1; k < 14; ++k) {
    term *= -x2 / ((2.0 * k) * (2.0 * k + 1.0));
    sum += term;
  }
  return sum;
}

constexpr double ct_cos_small(double x) {
  double x2 = x * x, term = 1.0, sum = 1.0;
  for (int k = 1; k < 14; ++k) {
    term *= -x2 / ((2.0 * k - 1.0) * (2.0 * k));
    sum += term;
  }
  return sum;
}

// cos and sin of 2 pi m / n, reduced exactly to |delta| <= pi/4
constexpr void ct_cs(int m, int n, double& c, double& s) {
  m %= n;
  if (m < 0) m += n;
  // nearest quarter turn q: 4m/n rounded
  int q = (8 * m + n) / (2 * n);
  const double delta = kTwoPi * (double)(4 * m - q * n) / (4.0 * n);
  const double cd = ct_cos_small(delta), sd = ct_sin_small(delta);
  switch (q & 3) {
    case 0: c = cd; s = sd; break;
    case 1: c = -sd; s = cd; break;
    case 2: c = -cd; s = -sd; break;
    default: c = sd; s = -cd; break;
  }
}

template <int R>
struct TwTab {
  double c[R];
  double s[R];
};

template <int R>
constexpr TwTab<R> make_tw() {
  TwTab<R> t{};
  for (int m = 0; m < R; ++m) ct_cs(m, R, t.c[m], t.s[m]);
  return t;
}

// The same for FP32, of the entries W^(n2 k1) that a P x Q split multiplies by.
// Rounded to nearest, sqrt(1/2), cos(pi/8), sin(pi/8) and sin(pi/3) all come out
// 1.6 to 3.1e-8 too small, and the results of every pass with them.  Here each entry
// takes, of the floats on both sides of its parts, the pair that keeps the sum of
// the moduli's errors so far nearest to zero.  psi(r) of random coefficients against
// FP64, cubes of 27 to 160: mean error -6.5 to +5.5e-8 -> -2.8 to +1.2e-8, rms (the mean in
// it) 1.34 to 1.60e-7 -> 1.31 to 1.59e-7 (less at seven of nine lengths; 1.49 -> 1.55 at 90,
// 1.50 -> 1.54 at 160), with the radix kernels as they are.
struct Near {
  double v[2];
};
constexpr Near ct_floats(double x) {  // the float nearest to x, the one on its other side
  const float f = (float)x;
  if ((double)f == x || f == 0.0f) return {{x, x}};
  double ulp = 1.0 / (1 << 24);
  for (double a = f < 0 ? -(double)f : (double)f; a < 0.5; a *= 2) ulp *= 0.5;
  return {{(double)f, (double)f < x ? (double)f + ulp : (double)f - ulp}};
}
template <int P, int Q>
constexpr TwTab<P * Q> make_tw32() {
  constexpr int R = P * Q;
  TwTab<R> t = make_tw<R>();
  double sum = 0.0;
  for (int m = 1; m < R; ++m) {
    int uses = 0;
    for (int n2 = 1; n2 < Q; ++n2)
      for (int k1 = 1; k1 < P; ++k1) uses += (n2 * k1) % R == m;
    const double c = t.c[m], s = t.s[m];
    const Near nc = ct_floats(c), ns = ct_floats(s);
    double best = 1.0, err = 0.0;
    for (int i = 0; i < 4; ++i) {
      const double a = nc.v[i & 1], b = ns.v[i >> 1];
      const double e = c * (a - c) + s * (b - s), z = sum + uses * e;
      if ((z < 0 ? -z : z) < best) {
        best = z < 0 ? -z : z;
        err = e;
        t.c[m] = a;
        t.s[m] = b;
      }
    }
    sum += uses * err;
  }
  return t;
}
template <typename T, int P, int Q>
constexpr TwTab<P * Q> make_tw_for() {
  if constexpr (sizeof(T) == 4)
    return make_tw32<P, Q>();
  else
    return make_tw<P * Q>();
}

// ---------------------------------------------------------------- radix DFTs
template <typename T>
__device__ __forceinline__ cpx<T> cm(cpx<T> a, cpx<T> b) {
  return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}

__device__ __forceinline__ float fm(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fm(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}

// Every small DFT starts with sums and differences of pairs.  Inputs that
// carry a twiddle each take part in them as they are: (a wa) +- (b wb) is one
// complex product, four fused multiply-adds for the sum and two for the
// difference 2 a wa - sum: 10 operations instead of the 12 of two products
// and two additions.  w == nullptr: plain inputs; ONE: w[0] is 1 (not read).
template <bool ONE, typename T>
__device__ __forceinline__ void pair_tw(const cpx<T>* v, const cpx<T>* w, int i, int j,
                                        cpx<T>& s, cpx<T>& d) {
  const cpx<T> a = v[i], b = v[j];
  if (w == nullptr) {
    s = {a.x + b.x, a.y + b.y};
    d = {a.x - b.x, a.y - b.y};
  } else {
    const cpx<T> p = ONE && i == 0 ? a : cm(a, w[i]), wb = w[j];
    s = {fm(b.x, wb.x, fm(-b.y, wb.y, p.x)), fm(b.x, wb.y, fm(b.y, wb.x, p.y))};
    d = {fm((T)2, p.x, -s.x), fm((T)2, p.y, -s.y)};
  }
}

// run(v): DFT of v in place; run_tw<ONE>(v, w): DFT of v[i] w[i]
template <typename T, int R, int S>
struct Dft;

template <typename T, int S>
struct Dft<T, 1, S> {
  static __device__ __forceinline__ void run(cpx<T>*) {}
  template <bool ONE>
  static __device__ __forceinline__ void run_tw(cpx<T>* v, const cpx<T>* w) {
    if (!ONE) v[0] = cm(v[0], w[0]);
  }
};

template <typename T, int S>
struct Dft<T, 2, S> {
  template <bool ONE>
  static __device__ __forceinline__ void run_tw(cpx<T>* v, const cpx<T>* w) {
    cpx<T> s, d;
    pair_tw<ONE>(v, w, 0, 1, s, d);
    v[0] = s;
    v[1] = d;
  }
  static __device__ __forceinline__ void run(cpx<T>* v) { run_tw<false>(v, nullptr); }
};

template <typename T, int S>
struct Dft<T, 3, S> {
  template <bool ONE>
  static __device__ __forceinline__ void run_tw(cpx<T>* v, const cpx<T>* w) {
    // FP32: 0.866025388 three times and the next float once (see make_tw32).  Outputs
    // 1 and 2 of a real input are each other's conjugates but for this ulp, 6e-8 d.x, as
    // much as one rounding of the sum.
    const T h = (T)S * (T)0.86602540378443864676;
    const T h1 = sizeof(T) == 4 ? (T)S * (T)0.866025447845458984 : h;
    cpx<T> t1, d;
    pair_tw<ONE>(v, w, 1, 2, t1, d);
    const cpx<T> a0 = ONE || w == nullptr ? v[0] : cm(v[0], w[0]);
    const cpx<T> t2 = {fm((T)-0.5, t1.x, a0.x), fm((T)-0.5, t1.y, a0.y)};
    v[0] = {a0.x + t1.x, a0.y + t1.y};
    v[1] = {fm(-h, d.y, t2.x), fm(h, d.x, t2.y)};
    v[2] = {fm(h, d.y, t2.x), fm(-h1, d.x, t2.y)};
  }
  static __device__ __forceinline__ void run(cpx<T>* v) { run_tw<false>(v, nullptr); }
};

template <typename T, int S>
struct Dft<T, 4, S> {
  template <bool ONE>
  static __device__ __forceinline__ void run_tw(cpx<T>* v, const cpx<T>* w) {
    cpx<T> t0, t1, t2, t3;
    pair_tw<ONE>(v, w, 0, 2, t0, t1);
    pair_tw<ONE>(v, w, 1, 3, t2, t3);
    const cpx<T> r = {-(T)S * t3.y, (T)S * t3.x};
    v[0] = {t0.x + t2.x, t0.y + t2.y};
    v[2] = {t0.x - t2.x, t0.y - t2.y};
    v[1] = {t1.x + r.x, t1.y + r.y};
    v[3] = {t1.x - r.x, t1.y - r.y};
  }
  static __device__ __forceinline__ void run(cpx<T>* v) { run_tw<false>(v, nullptr); }
};

// 32 operations: the sine parts are factored as s2 (phi d1 + d2) and
// s2 (d1 - phi d2), phi = sin(2 pi/5) / sin(4 pi/5), so that s2 goes into the
// outputs' multiply-adds, and the cosine parts as v0 - (b1 + b2)/4 +-
// (sqrt(5)/4) (b1 - b2).  In FP32 the rounding errors of these constants
// (-1.4e-8, 1.0e-8, 1.5e-8 relative) nearly cancel over the outputs; factoring
// out s1 instead scales them all by 2e-8, which adds up over the passes.
template <typename T, int S>
struct Dft<T, 5, S> {
  template <bool ONE>
  static __device__ __forceinline__ void run_tw(cpx<T>* v, const cpx<T>* w) {
    const T k5 = (T)0.55901699437494742410;               // sqrt(5) / 4
    const T s2 = (T)S * (T)0.58778525229247312917;        // sin(4 pi / 5)
    const T phi = (T)1.61803398874989484820;              // sin(2 pi / 5) / sin(4 pi / 5)
    cpx<T> b1, b2, d1, d2;
    pair_tw<ONE>(v, w, 1, 4, b1, d1);
    pair_tw<ONE>(v, w, 2, 3, b2, d2);
    const cpx<T> a0 = ONE || w == nullptr ? v[0] : cm(v[0], w[0]);
    const cpx<T> t = {b1.x + b2.x, b1.y + b2.y}, e = {b1.x - b2.x, b1.y - b2.y};
    const cpx<T> m = {fm((T)-0.25, t.x, a0.x), fm((T)-0.25, t.y, a0.y)};
    const cpx<T> p1 = {fm(k5, e.x, m.x), fm(k5, e.y, m.y)};
    const cpx<T> p2 = {fm(-k5, e.x, m.x), fm(-k5, e.y, m.y)};
    const cpx<T> r1 = {fm(phi, d1.x, d2.x), fm(phi, d1.y, d2.y)};
    const cpx<T> r2 = {fm(-phi, d2.x, d1.x), fm(-phi, d2.y, d1.y)};
    v[0] = {a0.x + t.x, a0.y + t.y};
    v[1] = {fm(-s2, r1.y, p1.x), fm(s2, r1.x, p1.y)};
    v[4] = {fm(s2, r1.y, p1.x), fm(-s2, r1.x, p1.y)};
    v[2] = {fm(-s2, r2.y, p2.x), fm(s2, r2.x, p2.y)};
    v[3] = {fm(s2, r2.y, p2.x), fm(-s2, r2.x, p2.y)};
  }
  static __device__ __forceinline__ void run(cpx<T>* v) { run_tw<false>(v, nullptr); }
};

// R = P*Q: n = Q n1 + n2, k = k1 + P k2;
// X[k1 + P k2] = sum_n2 W_Q^{n2 k2} W_R^{n2 k1} sum_n1 x[Q n1 + n2] W_P^{n1 k1}
template <typename T, int P, int Q, int S>
struct DftPQ {
  static __device__ __forceinline__ void run(cpx<T>* v) { run_tw<false>(v, nullptr); }
  template <bool ONE>
  static __device__ __forceinline__ void run_tw(cpx<T>* v, const cpx<T>* w) {
    constexpr int R = P * Q;
    constexpr TwTab<R> tw = make_tw_for<T, P, Q>();
    cpx<T> y[Q][P];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) {
      cpx<T> a[P];
#pragma unroll
      for (int n1 = 0; n1 < P; ++n1) a[n1] = v[Q * n1 + n2];
      if (w == nullptr) {
        Dft<T, P, S>::run(a);
      } else {
        cpx<T> wa[P];
#pragma unroll
        for (int n1 = 0; n1 < P; ++n1) wa[n1] = w[Q * n1 + n2];
        if (n2 == 0) Dft<T, P, S>::template run_tw<ONE>(a, wa);
        else Dft<T, P, S>::template run_tw<false>(a, wa);
      }
#pragma unroll
      for (int k1 = 0; k1 < P; ++k1) {
        const int m = (n2 * k1) % R;
        if (m == 0) {
          y[n2][k1] = a[k1];
        } else {
          const cpx<T> wm = {(T)tw.c[m], (T)(S * tw.s[m])};
          y[n2][k1] = cm(a[k1], wm);
        }
      }
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
      cpx<T> b[Q];
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) b[n2] = y[n2][k1];
      Dft<T, Q, S>::run(b);
#pragma unroll
      for (int k2 = 0; k2 < Q; ++k2) v[k1 + P * k2] = b[k2];
    }
  }
};

// R = P*Q with gcd(P, Q) = 1 (Good-Thomas prime-factor map, no twiddles):
// n = (Q n1 + P n2) mod R, k = (Q a k1 + P b k2) mod R with a = Q^-1 mod P,
// b = P^-1 mod Q, so that W_R^{nk} = W_P^{n1 k1} W_Q^{n2 k2}.
constexpr int ct_inv_mod(int x, int m) {
  for (int i = 1; i < m; ++i)
    if ((x * i) % m == 1) return i;
  return 1;
}

template <typename T, int P, int Q, int S>
struct DftPFA {
  static __device__ __forceinline__ void run(cpx<T>* v) { run_tw<false>(v, nullptr); }
  template <bool ONE>
  static __device__ __forceinline__ void run_tw(cpx<T>* v, const cpx<T>* w) {
    constexpr int R = P * Q;
    constexpr int A = ct_inv_mod(Q % P, P), B = ct_inv_mod(P % Q, Q);
    cpx<T> y[Q][P];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) {
      cpx<T> a[P];
#pragma unroll
      for (int n1 = 0; n1 < P; ++n1) a[n1] = v[(Q * n1 + P * n2) % R];
      if (w == nullptr) {
        Dft<T, P, S>::run(a);
      } else {
        cpx<T> wa[P];
#pragma unroll
        for (int n1 = 0; n1 < P; ++n1) wa[n1] = w[(Q * n1 + P * n2) % R];
        if (n2 == 0) Dft<T, P, S>::template run_tw<ONE>(a, wa);
        else Dft<T, P, S>::template run_tw<false>(a, wa);
      }
#pragma unroll
      for (int k1 = 0; k1 < P; ++k1) y[n2][k1] = a[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
      cpx<T> b[Q];
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) b[n2] = y[n2][k1];
      Dft<T, Q, S>::run(b);
#pragma unroll
      for (int k2 = 0; k2 < Q; ++k2) v[(Q * A * k1 + P * B * k2) % R] = b[k2];
    }
  }
};

template <typename T, int S> struct Dft<T, 6, S> : DftPFA<T, 2, 3, S> {};
template <typename T, int S> struct Dft<T, 8, S> : DftPQ<T, 2, 4, S> {};
template <typename T, int S> struct Dft<T, 9, S> : DftPQ<T, 3, 3, S> {};
template <typename T, int S> struct Dft<T, 10, S> : DftPFA<T, 2, 5, S> {};
template <typename T, int S> struct Dft<T, 12, S> : DftPFA<T, 4, 3, S> {};
template <typename T, int S> struct Dft<T, 15, S> : DftPFA<T, 3, 5, S> {};
template <typename T, int S> struct Dft<T, 16, S> : DftPQ<T, 4, 4, S> {};

// pass-2 twiddle W_N^{m} from the table exp(-2 pi i j / N), conjugated for S = +1
template <typename T, int S>
__device__ __forceinline__ cpx<T> twiddle(const double2* __restrict__ tw, int m) {
  const double2 w = tw[m];
  return {(T)w.x, (T)(S < 0 ? w.y : -w.y)};
}

// Pruning to the sphere.  A grid that holds the density sphere |G|^2 <= 4
// Ecut has N >= 2 kr + 1 with kr >= 2 kmax, so the wavefunction components
// satisfy |k| <= KM = (N - 1) / 4 along every axis.  A radix pass reading
// (or writing) index i = j + t*STRIDE, j < STRIDE, touches only zeros (or
// unneeded outputs) for every j when KM < t*STRIDE and t*STRIDE + STRIDE - 1
// < N - KM, i.e. for t in [T0, T1].  Pruned kernels set those inputs to zero
// at compile time and do not store those outputs, so the compiler drops
// their arithmetic (the engine's translation units are built with
// -fno-signed-zeros, which lets x + 0 fold to x; only the sign of zero
// results can differ).
template <int N, int STRIDE>
struct Sph {
  static constexpr int KM = (N - 1) / 4;
  static constexpr int T0 = KM / STRIDE + 1;
  static constexpr int T1 = (N - KM - STRIDE) / STRIDE;
  static __device__ __forceinline__ constexpr bool cut(bool on, int t) {
    return on && t >= T0 && t <= T1;
  }
};

}  // namespace oa2

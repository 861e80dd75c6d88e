// oa_gemm.hip -- dense FP64 contractions of the CP electronic step on
// CDNA4 matrix cores (v_mfma_f64_16x16x4f64).
//
//   gram    : S = 2 Re Psi^H Psi over stored points with kx=0 halved
//             (PairCalculator::multiplyForward, ckPairCalculator.C:682-802)
//             and Lambda = Re Psi^H F (asymmetric PairCalculator, alpha = 1).
//             One workgroup owns a 64 x 64 (48 x 48) output block and one
//             slice of the long point axis; the slices' partial blocks are
//             summed in a fixed order.
//   rotate  : Psi' = Psi T and F -= w Psi Lambda
//             (bwMultiplyHelper, ckPairCalculator.C:1189-1425;
//              unpackLambda, CP_State_GSpacePlane.C:2045-2225), optionally
//             followed in the same pass by the steepest-descent update
//             psi += dt/m F (CP_integrate_min_STD, cp_min_std.C:56-86).
//   ns      : Newton-Schulz iteration for (S/2)^{-1/2}
//             (Ortho::do_iteration/step_2/step_3/tolerance_check,
//              ortho.C:862-985; serial twin cp_lowdin.C:180-265): plain
//             launches with a device-side early exit (one workgroup up to 64
//             states, small tiles above); on request one cooperative launch
//             that loops on the device with grid barriers.
//
// MFMA operand layout (measured on gfx950): lane l supplies A[l%16][l/16]
// and B[l/16][l%16] and receives D[l/16 + 4v][l%16] in element v.  Within
// one MFMA the assignment of the four k values to the four lane groups is
// free as long as A and B agree: in the gram, lane group g takes the
// contiguous run k0+4g..k0+4g+3 over four consecutive MFMAs, so every lane
// issues one 32-byte load per operand row and 16 k values.
#include <hip/hip_cooperative_groups.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "oa_common.h"
#include "oa_gemm_common.h"
#include "oa_kernels.h"

namespace oa {

typedef double v4d __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4d mfma16(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ v4d vzero() { return (v4d){0.0, 0.0, 0.0, 0.0}; }

// ================================================================== gram

__host__ __device__ constexpr int up_i(int idx, int m) {
  int i = 0;
  while (idx >= m - i) {
    idx -= m - i;
    i++;
  }
  return i;
}
__host__ __device__ constexpr int up_j(int idx, int m) {
  int i = 0;
  while (idx >= m - i) {
    idx -= m - i;
    i++;
  }
  return i + idx;
}
// f[e] = X[row][kk + e]: one 32-byte load, kk a multiple of 4 inside the
// row's allocation (chunks start on multiples of 16 below K <= lda, lda a
// multiple of 16).  Unconditional: rows past the matrix are clamped by the
// caller (their outputs are never stored) and elements outside the slice's
// region are zeroed where they are consumed (gmask), so no load sits in a
// branch and the ring's loads stay in flight.
__device__ __forceinline__ void gfrag(const double* __restrict__ X, int lda, int row, int kk,
                                      double (&f)[4]) {
  const double4 v = *reinterpret_cast<const double4*>(X + (size_t)row * lda + kk);
  f[0] = v.x;
  f[1] = v.y;
  f[2] = v.z;
  f[3] = v.w;
}

// zero f[e] for kk + e outside [rs, re)
__device__ __forceinline__ void gmask(int kk, int rs, int re, double (&f)[4]) {
#pragma unroll
  for (int e = 0; e < 4; e++) f[e] = (kk + e >= rs && kk + e < re) ? f[e] : 0.0;
}

template <int NF>
struct Frag {
  double f[NF][4];
};
constexpr int kGramRing = 3;

// Output block of MT x NT tiles from tile (ti0, tj0) (DIAG: the upper ones of a
// diagonal block of a symmetric product): each wave holds all of it for every fourth
// chunk of the slice, and the four waves' sums meet in LDS (4 x SM doubles).
template <int MT, int NT, bool DIAG, int SM>
__device__ __forceinline__ void gram_block(const GramArgs& a, const double* __restrict__ B,
                                           const GSlice& s, int sp, int ti0, int tj0,
                                           double (*sm)[SM]) {
  constexpr int NF = DIAG ? NT : MT + NT, NTW = DIAG ? NT * (NT + 1) / 2 : MT * NT;
  static_assert(NTW * 256 <= SM && (!DIAG || MT == NT), "");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  int row[NF];
#pragma unroll
  for (int f = 0; f < NF; f++) {
    const int r = 16 * (f < MT ? ti0 + f : tj0 + f - MT) + l16;
    row[f] = r < (f < MT ? a.n : a.nb) ? r : 0;  // rows past n: outputs not stored
  }
  v4d acc[NTW];
#pragma unroll
  for (int t = 0; t < NTW; t++) acc[t] = vzero();
  auto mfmas = [&](const double (&f)[NF][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; e++)
      static_for<0, NTW>([&](auto tc) __attribute__((always_inline)) {
        constexpr int t = decltype(tc)::value;
        constexpr int ia = DIAG ? up_i(t, NT) : t / NT, ib = DIAG ? up_j(t, NT) : MT + t % NT;
        acc[t] = mfma16(f[ia][e], f[ib][e], acc[t]);
      });
  };
  Frag<NF> ring[kGramRing];
  chunk_ring(
      0, (s.c1 - s.c0 - wave + 3) >> 2, ring,
      [&](int c, Frag<NF>& d) __attribute__((always_inline)) {
        const int kk = s.base + 16 * (s.c0 + wave + 4 * c) + 4 * g;
#pragma unroll
        for (int f = 0; f < NF; f++) gfrag(f < MT ? a.A : B, a.lda, row[f], kk, d.f[f]);
      },
      [&](int c, const Frag<NF>& d) __attribute__((always_inline)) {
        const int k0 = s.base + 16 * (s.c0 + wave + 4 * c);
        if (k0 >= s.rs && k0 + 16 <= s.re) {
          mfmas(d.f);
        } else {  // a chunk at the region's edge (padding past K may hold anything)
          Frag<NF> m = d;
#pragma unroll
          for (int f = 0; f < NF; f++) gmask(k0 + 4 * g, s.rs, s.re, m.f[f]);
          mfmas(m.f);
        }
      });
  // Tile t is summed and stored by wave t & 3, in the order (0 + 2) + (1 + 3) whichever
  // wave it is: one barrier.  By halves to wave 0, which then stored everything, were
  // three more: S of 33, 64, 128, 256 states x 10,324 reals 16.2, 21.2, 23.6, 43.7 us
  // then, 15.1, 19.7, 21.9, 41.2 now; 256 x 62,106 138 and 136
  static_for<0, NTW>([&](auto tc) __attribute__((always_inline)) {
    constexpr int t = decltype(tc)::value;
    if (wave != (t & 3)) {
#pragma unroll
      for (int v = 0; v < 4; v++) sm[wave][(4 * t + v) * 64 + lane] = acc[t][v];
    }
  });
  __syncthreads();
  double* part = a.part + (size_t)sp * a.n * a.nb;
  static_for<0, NTW>([&](auto tc) __attribute__((always_inline)) {
    constexpr int t = decltype(tc)::value, o = t & 3;
    constexpr int ti = DIAG ? up_i(t, NT) : t / NT, tj = DIAG ? up_j(t, NT) : t % NT;
    if (wave != o) return;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int e = (4 * t + v) * 64 + lane;
      const double d = (acc[t][v] + sm[o ^ 2][e]) + (sm[o ^ 1][e] + sm[o ^ 3][e]);
      const int r = 16 * (ti0 + ti) + g + 4 * v, col = 16 * (tj0 + tj) + l16;
      if (r < a.n && col < a.nb) part[(size_t)r * a.nb + col] = s.w * d;
    }
  });
}

// One-dimensional grid of (K slice, output block), blocks fastest, a contiguous
// range of it for each XCD: the blocks of a slice read the same rows at about the
// same time through one L2.  With the sums of the slices, in us (before: 128 x 128
// blocks of four different waves, idle where n is not a multiple of 128): S of 84 states
// x 30,024 reals 23 (26), 128 x 58,400 37 (38), 132 46 (103), 180 x 73,412 82 (130),
// 256 x 121,214 194 (220), 512 x 236,230 1071 (1277); full products 25 (32), 45 (51), 57
// (140), 98 (174), 254 (287), 1839 (2012).  Bound by the matrix pipe, 61 to 66 TFLOP/s
// from 256 states up, and by the start and end of a slice below.
template <int NT>
__global__ __launch_bounds__(256) void k_gram(GramArgs a, int nbe, int nbe_b, int nblk, int nlo) {
  __shared__ double sm[4][NT * NT * 256];
  const int total = gridDim.x, xcd = blockIdx.x & 7, k = blockIdx.x >> 3;
  const int q = total >> 3, r = total & 7;
  const int logical = xcd * q + min(xcd, r) + k;
  const int sp = logical / nblk;
  int b = logical - sp * nblk, bi, bj;
  const GSlice s = gram_slice(a, sp, nlo);
  if (a.sym && NT == 4 && nblk == 4) {  // GramShape: two diagonal blocks, two halves
    if (b < 2)
      gram_block<NT, NT, true>(a, a.A, s, sp, NT * b, NT * b, sm);
    else
      gram_block<(NT + 1) / 2, NT, false>(a, a.A, s, sp, NT / 2 * (b - 2), NT, sm);
    return;
  }
  if (a.sym) {
    bi = 0;
    while (b >= nbe - bi) {
      b -= nbe - bi;
      bi++;
    }
    bj = bi + b;
    if (bi == bj) {
      gram_block<NT, NT, true>(a, a.A, s, sp, NT * bi, NT * bi, sm);
      return;
    }
  } else {
    bi = b / nbe_b;
    bj = b - bi * nbe_b;
  }
  gram_block<NT, NT, false>(a, a.sym ? a.A : a.B, s, sp, NT * bi, NT * bj, sm);
}

// nb <= 32 < n (the non-local projections of few atoms): blocks of 64 rows and all
// columns, the rest as in k_gram.  128 states x 32 atoms x 65,922 reals 61 -> 22 us;
// before, a wave of a 128-row block had 32 rows for all of K, and too little in flight.
// From 33 rows: whole blocks of 64 x 64 are 16 tiles for 4 or 8 (64 x 8 atoms x 62,106
// reals, one call, 66 -> 60 us).
template <int NT>
__global__ __launch_bounds__(256) void k_gram_nb(GramArgs a, int nblk, int nlo) {
  __shared__ double sm[4][4 * NT * 256];
  const int sp = blockIdx.x / nblk, b = blockIdx.x - sp * nblk;
  gram_block<4, NT, false>(a, a.B, gram_slice(a, sp, nlo), sp, 4 * b, 0, sm);
}

// Tiles per block edge and blocks of the output: a single block up to 64 rows and
// columns, else blocks of 3 or 4 tiles, whichever computes fewer tiles (9 tiles an
// edge: 45 instead of 78 for the symmetric product), 4 where they are equal (more
// products per loaded row).  With two blocks an edge of 4 tiles the one off the
// diagonal of a symmetric product is cut in two, so that no workgroup has more than 10
// tiles (no other symmetric product has 4 blocks): 128 states 43 -> 37 us.
struct GramShape {
  int nt, nbe, nbe_b, blocks;
};
static GramShape gram_shape(int n, int nb, int sym) {
  auto shape = [&](int nt) {
    const int w = 16 * nt, e = (n + w - 1) / w, f = (nb + w - 1) / w;
    return GramShape{nt, e, f, sym ? e * (e + 1) / 2 : e * f};
  };
  auto tiles = [&](const GramShape& s) {
    const int full = s.nt * s.nt, diag = s.nt * (s.nt + 1) / 2;
    return sym ? s.nbe * diag + (s.blocks - s.nbe) * full : s.blocks * full;
  };
  const int edge = std::max(n, nb);
  if (edge <= kGramSmall) return shape((edge + 15) / 16);
  const GramShape s3 = shape(3);
  GramShape s4 = shape(4);
  if (tiles(s3) < tiles(s4)) return s3;
  if (sym && s4.nbe == 2) s4.blocks = 4;
  return s4;
}

static bool gram_skinny(int n, int nb, int sym) { return !sym && nb <= 32 && n > 32; }

int gram_slices(int n, int nb, int K, int sym, int ncu) {
  const int blocks = gram_skinny(n, nb, sym) ? (n + 63) / 64 : gram_shape(n, nb, sym).blocks;
  // whole rounds of a workgroup per CU, the more the longer (about 200 chunks a wave):
  // then the lighter blocks on the diagonal even out (512 states: 7 slices 1.15 ms, 14
  // 1.07; but 128 states: 64 slices 37 us, 128 47)
  const double rounds = (double)(K / 64) / 200.0 * blocks / ncu;
  const int ns = std::max(1, (int)std::ceil(rounds - 0.25)) * ncu / blocks;
  return std::min(std::max(2, ns), std::max(2, K / 64));  // four chunks or more each
}

hipError_t gram_f64(const GramArgs& a, hipStream_t st) {
  if (a.nslice < 1 || (a.k_lo > 0 && a.k_lo < a.K && a.nslice < 2) || (a.lda & 3) ||
      a.n < 1 || a.nb < 1 || (a.sym && a.nb != a.n))
    return hipErrorInvalidValue;
  const int nlo = gram_nlo(a);
  if (gram_skinny(a.n, a.nb, a.sym)) {
    const int nblk = (a.n + 63) / 64;
    hipLaunchKernelGGL(a.nb <= 16 ? k_gram_nb<1> : k_gram_nb<2>, dim3(nblk * a.nslice), dim3(256),
                       0, st, a, nblk, nlo);
    return hipGetLastError();
  }
  const GramShape s = gram_shape(a.n, a.nb, a.sym);
  void (*const fn)(GramArgs, int, int, int, int) = s.nt == 1   ? k_gram<1>
                                                   : s.nt == 2 ? k_gram<2>
                                                   : s.nt == 3 ? k_gram<3>
                                                               : k_gram<4>;
  hipLaunchKernelGGL(fn, dim3(s.blocks * a.nslice), dim3(256), 0, st, a, s.nbe, s.nbe_b, s.blocks,
                     nlo);
  return hipGetLastError();
}

// C[e] = alpha * sum_sp part[sp][e'] with e' = e or its mirror; 64 outputs
// per workgroup, 16 groups of slices summed through LDS in a fixed order
template <typename P>
__global__ __launch_bounds__(1024) void k_gram_reduce(const P* __restrict__ part, int nslice,
                                                      int n, int nb, int sym, double alpha,
                                                      double* __restrict__ C) {
  __shared__ double red[16][64];
  const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
  const size_t nn = (size_t)n * nb;
  const size_t e = (size_t)blockIdx.x * 64 + x;
  double s0 = 0.0, s1 = 0.0;
  if (e < nn) {
    int i = (int)(e / nb), j = (int)(e - (size_t)i * nb);
    if (sym && (i >> 4) > (j >> 4)) {  // sym: nb == n
      const int t = i;
      i = j;
      j = t;
    }
    const P* p = part + (size_t)i * nb + j;
    // thread y sums slices y, y+16, y+32, ...: 16 loads in flight,
    // branch-free (slice index clamped, value masked)
    for (int base = 0; base < nslice; base += 256) {
      double v[16];
#pragma unroll
      for (int u = 0; u < 16; u++) {
        const int sp = base + y + 16 * u;
        const double w = (double)p[(size_t)min(sp, nslice - 1) * nn];
        v[u] = sp < nslice ? w : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 16; u += 2) {
        s0 += v[u];
        s1 += v[u + 1];
      }
    }
  }
  red[y][x] = s0 + s1;
  __syncthreads();
  if (y == 0 && e < nn) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < 16; w++) t += red[w][x];
    C[e] = alpha * t;
  }
}

// Symmetric product: four workgroups per upper 16 x 16 tile (the tiles the
// gram wrote), each a quarter of the tile's rows; written to C and, off the
// diagonal, to its mirror.  Thread (y, x): element x of the 4 x 16 quarter,
// slices y, y + 16, ...; loads branch-free (slice index clamped, value
// masked), 16 in flight; the 16 slice groups are summed through LDS in a
// fixed order.
template <typename P>
__global__ __launch_bounds__(1024) void k_gram_reduce_sym(const P* __restrict__ part,
                                                          int nslice, int n, double alpha,
                                                          double* __restrict__ C) {
  __shared__ double red[16][64];
  const int nt = (n + 15) >> 4;
  int b = blockIdx.x >> 2, ti = 0;
  while (b >= nt - ti) {
    b -= nt - ti;
    ti++;
  }
  const int tj = ti + b;
  const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
  const int i = ti * 16 + (blockIdx.x & 3) * 4 + (x >> 4), j = tj * 16 + (x & 15);
  const size_t nn = (size_t)n * n;
  // a diagonal tile takes both halves from the upper triangle's partials, so
  // C is symmetric bit for bit also where the partials of (i, j) and (j, i)
  // were summed in different orders (split-BF16 term products)
  const int ir = ti == tj ? min(i, j) : i, jr = ti == tj ? max(i, j) : j;
  const P* p = part + (size_t)min(ir, n - 1) * n + min(jr, n - 1);
  double s0 = 0.0, s1 = 0.0;
  for (int base = 0; base < nslice; base += 256) {
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int sp = base + y + 16 * u;
      const double w = (double)p[(size_t)min(sp, nslice - 1) * nn];
      v[u] = sp < nslice ? w : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 16; u += 2) {
      s0 += v[u];
      s1 += v[u + 1];
    }
  }
  red[y][x] = s0 + s1;
  __syncthreads();
  if (y == 0 && i < n && j < n) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < 16; w++) t += red[w][x];
    const double v = alpha * t;
    C[(size_t)i * n + j] = v;
    if (ti < tj) C[(size_t)j * n + i] = v;  // a diagonal tile holds both halves
  }
}

template <typename P>
static hipError_t gram_reduce_t(const P* part, int nslice, int n, int nb, int sym, double alpha,
                                double* C, hipStream_t st) {
  if (sym && nb != n) return hipErrorInvalidValue;
  // up to 64 states the product wrote whole tiles in FP64, so the plain sum can read the
  // mirrored elements again: 4.1 us for 16 states, 7.4 by tiles.  Beyond 32 its strided
  // reads of them cost more than the tiles' turn through LDS: S at 10,324 reals takes
  // 18.7 us plain and 14.7 by tiles for 40 states, 27.7 and 19.8 for 64 (62,106 reals:
  // 36.1 and 23.4)
  if (sym && !(sizeof(P) == 8 && n <= 32)) {
    const int nt = (n + 15) >> 4;
    hipLaunchKernelGGL(k_gram_reduce_sym<P>, dim3(4 * (nt * (nt + 1) / 2)), dim3(1024), 0, st,
                       part, nslice, n, alpha, C);
    return hipGetLastError();
  }
  const size_t nn = (size_t)n * nb;
  hipLaunchKernelGGL(k_gram_reduce<P>, dim3((unsigned)((nn + 63) / 64)), dim3(1024), 0, st,
                     part, nslice, n, nb, sym, alpha, C);
  return hipGetLastError();
}

hipError_t gram_reduce(const double* part, int nslice, int n, int nb, int sym, double alpha,
                       double* C, hipStream_t st) {
  return gram_reduce_t(part, nslice, n, nb, sym, alpha, C, st);
}

// FP32 partials (split-BF16 gram), summed in FP64
hipError_t gram_reduce_f32(const float* part, int nslice, int n, int nb, int sym, double alpha,
                           double* C, hipStream_t st) {
  return gram_reduce_t(part, nslice, n, nb, sym, alpha, C, st);
}

// ================================================================== rotate
// Y[j][k] = beta Y[j][k] + s(k) sum_{i < ni} M[i][j] X[i][k] as D = M^T X: the
// output tile rows are j and its columns k, so the stores run along k.
constexpr int kRK = 64;

// n or ni > 128.  Workgroup: 64 columns k, W waves of JT 16-row tiles j each;
// wave: 16 JT x 64 outputs, so a step of four i costs JT + 2 loads per lane for
// 4 JT MFMAs.  A lane's B values are four consecutive k (two 16-byte loads; the
// output column l16 of tile y is k = kb + 4 l16 + y, any assignment works as long
// as the stores follow it), so a row of Y is read and written 32 bytes per lane.
// The loads of a step are issued kRwRing steps ahead into a register ring (two
// ahead: 20 % slower, four: the same), two waves per SIMD (one: 10 % slower).
// Bound by the matrix pipe, and below 400 states by the start and end of a
// block.  Y = M^T X (and Y += ...): 512 states x 260,992 reals 68 (62) TFLOP/s,
// 256 x 131,824 50 (47), 180 x 73,600 45 (46); 50 (50), 45 (40), 32 (32) before,
// with 32 x 64 outputs per wave, 1.5 times the loads per MFMA and Y accessed in
// 8-byte pieces.  A library product of the first two shapes reaches 71 and 49.  With the
// tiles of rw_shape, Y = M^T X as a step's stage: 512 x 241,238 67, 256 x 134,952 57,
// 180 x 75,332 50.
constexpr int kRwRing = 3;

template <int JT>
struct RwStep {
  double a[JT];
  double4 b;
};

template <int JT, bool USE_Y>
__global__ __launch_bounds__(256, 2) void k_rotate_w(RotArgs a) {
  __shared__ double red[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int kb = blockIdx.x * kRK;
  const int jb = (blockIdx.y * nw + wave) * 16 * JT;
  double fn = 0.0;
  if (jb < a.n) {
    v4d acc[JT][4];
#pragma unroll
    for (int x = 0; x < JT; x++)
#pragma unroll
      for (int y = 0; y < 4; y++) acc[x][y] = vzero();
    // byte offsets of the lane inside a step's four rows; rows j past n are
    // computed from duplicated data and never stored
    unsigned mo[JT];
#pragma unroll
    for (int x = 0; x < JT; x++)
      mo[x] = (unsigned)((g * a.n + min(jb + 16 * x + l16, a.n - 1)) * sizeof(double));
    const unsigned xo = (unsigned)((g * a.ldx + kb + 4 * l16) * sizeof(double));
    const int nfull = a.ni >> 2;
    auto load = [&](int st, RwStep<JT>& d) __attribute__((always_inline)) {
      const char* mp = (const char*)(a.M + (size_t)st * 4 * a.n);
      const char* xp = (const char*)(a.X + (size_t)st * 4 * a.ldx);
#pragma unroll
      for (int x = 0; x < JT; x++) d.a[x] = *(const double*)(mp + mo[x]);
      d.b = *(const double4*)(xp + xo);
    };
    auto mma = [&](const RwStep<JT>& d) __attribute__((always_inline)) {
      const double bv[4] = {d.b.x, d.b.y, d.b.z, d.b.w};
#pragma unroll
      for (int x = 0; x < JT; x++)
#pragma unroll
        for (int y = 0; y < 4; y++) acc[x][y] = mfma16(d.a[x], bv[y], acc[x][y]);
    };
    if (nfull > 0) {
      RwStep<JT> ring[kRwRing];
      static_for<0, kRwRing>([&](auto dc) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value;
        load(min(d, nfull - 1), ring[d]);
      });
      // every load is issued on every path (past the end: the last step again)
      for (int st = 0; st < nfull; st += kRwRing) {
        static_for<0, kRwRing>([&](auto dc) __attribute__((always_inline)) {
          constexpr int d = decltype(dc)::value;
          if (st + d < nfull) mma(ring[d]);
          load(min(st + d + kRwRing, nfull - 1), ring[d]);
        });
      }
    }
    if (a.ni & 3) {  // the last, partial step: rows past ni clamped, their M zeroed
      RwStep<JT> d;
      const int i = 4 * nfull + g, ic = min(i, a.ni - 1);
#pragma unroll
      for (int x = 0; x < JT; x++) {
        const double m = a.M[(size_t)ic * a.n + min(jb + 16 * x + l16, a.n - 1)];
        d.a[x] = i < a.ni ? m : 0.0;
      }
      d.b = *(const double4*)(a.X + (size_t)ic * a.ldx + kb + 4 * l16);
      mma(d);
    }
    const int k0 = kb + 4 * l16;
    double s[4];
#pragma unroll
    for (int y = 0; y < 4; y++) s[y] = k0 + y < a.k_lo ? a.s_lo : a.s_hi;
#pragma unroll
    for (int x = 0; x < JT; x++) {
      double4 yo[4];
      if (USE_Y) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int j = min(jb + 16 * x + g + 4 * v, a.n - 1);
          yo[v] = *(const double4*)(a.Y + (size_t)j * a.ldx + k0);
        }
      }
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int j = jb + 16 * x + g + 4 * v;
        double o[4];
#pragma unroll
        for (int y = 0; y < 4; y++) o[y] = s[y] * acc[x][y][v];
        if (USE_Y) {
          o[0] = a.beta * yo[v].x + o[0];
          o[1] = a.beta * yo[v].y + o[1];
          o[2] = a.beta * yo[v].z + o[2];
          o[3] = a.beta * yo[v].w + o[3];
        }
        if (j < a.n) {
          double* yp = a.Y + (size_t)j * a.ldx + k0;
          if (k0 + 3 < a.K) {
            *(double4*)yp = make_double4(o[0], o[1], o[2], o[3]);
            fn += (o[0] * o[0] + o[1] * o[1]) + (o[2] * o[2] + o[3] * o[3]);
          } else {
#pragma unroll
            for (int y = 0; y < 4; y++)
              if (k0 + y < a.K) {
                yp[y] = o[y];
                fn += o[y] * o[y];
              }
          }
        }
      }
    }
  }
  if (a.fpart) {
    for (int o = 32; o > 0; o >>= 1) fn += __shfl_down(fn, o, 64);
    if (lane == 0) red[wave] = fn;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int w = 0; w < nw; w++) t += red[w];
      a.fpart[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = t;
    }
  }
}

// Waves per workgroup and 16-row tiles per wave for n output rows and K columns: the
// pair with the shortest chain of tiles on one SIMD.  ceil(workgroups / CUs) of a CU
// spread their waves over its four SIMDs; a wave costs its jt tiles and a little for the
// loads that it does not share (0.1), and the first and the last one of a SIMD run
// without a neighbour (jt / 2).  Few columns then take small tiles, which leave no CU
// without a workgroup, and many columns the tiles that compute the fewest rows past n.
// Over 17 state counts from 129 to 512 and 10 column counts from 1,142 to 252,902 the
// rule is within 1 % of the fastest pair on average (the fewest rows past n alone: 15 %).
// Y = M^T X, us, 4 x 4, 4 x 3, 3 x 3, 4 x 2: 256 x 1,142 51, 51, 40, 32; 512 x 17,874
// 203, 199, 226, 170; 384 x 62,106 380, 308, 357, 303; 144 x 252,902 306, 233, 228, 263;
// 512 x 252,902 1,964, 2,116, 2,235, 2,064.
struct RwShape {
  int waves, jt, blocks;
};
static RwShape rw_shape(int n, int K) {
  const int nt = (n + 15) / 16, ncu = cu_count();
  RwShape best{};
  long long low = -1;
  const int cand[4][2] = {{4, 4}, {4, 3}, {3, 3}, {4, 2}};
  for (const auto& c : cand) {
    const int per = c[0] * c[1], blocks = (nt + per - 1) / per;
    const long long wgs = (long long)((K + kRK - 1) / kRK) * blocks;
    const long long waves = ((wgs + ncu - 1) / ncu * c[0] + 3) / 4;  // of one SIMD
    const long long cost = waves * (10 * c[1] + 1) + 5 * c[1];
    if (low < 0 || cost < low) {
      low = cost;
      best = {c[0], c[1], blocks};
    }
  }
  return best;
}

// n, ni <= 128: persistent workgroups of 8 waves (two per SIMD).  M is staged
// once per workgroup in LDS (16 NCH x 128, zero beyond ni x n, row stride 129);
// workgroup b walks the 64-column k-blocks b, b + gridDim.x, ...  Wave w
// owns the output rows j in [32 (w & 3), +32) and the k tiles 2 (w >> 2),
// 2 (w >> 2) + 1 of a block.  The work items are (k-block, chunk of 16 i);
// a ring of R X buffers (R = 4, or 3 when the epilogue needs both Y and the
// SD operands) keeps the loads of item q+R in flight while the MFMAs of
// items q+1..q+R-1 issue, across k-block boundaries.  The
// epilogue's operands (Y when beta != 0, psi and dt/m for the SD update)
// are loaded a few items before the block ends, behind its MFMAs.
constexpr int rot_ring(bool use_y, bool use_sd) { return use_y && use_sd ? 3 : 4; }
constexpr int gcd_c(int a, int b) { return b == 0 ? a : gcd_c(b, a % b); }
constexpr int kRotLd = 129;                    // LDS row stride of M
constexpr int kRotThreads = 512;
constexpr size_t rot_smem(int nch) { return (size_t)16 * nch * kRotLd * sizeof(double); }

struct XFrag {
  double v[4][2];  // [i step][k tile]
};

// NCH: i chunks of 16 per k-block (1, 2, 4 or 8; M is zero beyond ni).  The
// item loop is unrolled over G = lcm(NCH, R) items so that ring
// slots and block epilogues sit at fixed places of the loop body.  USE_Y
// (beta != 0) and USE_SD (sd_psi set) are compile-time so that the
// epilogue operands only take registers when used: the ring's loads must
// fit beside them to stay in flight.
template <int NCH, bool USE_Y, bool USE_SD>
__global__ __launch_bounds__(kRotThreads) void k_rotate_p(RotArgs a) {
  extern __shared__ __align__(16) double msm[];
  __shared__ double red[kRotThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int jb = (wave & 3) * 32, kt0 = 2 * (wave >> 2);
  const bool wact = jb < a.n;
  // Workgroup b owns the 16-column tiles [t0, t1), an even split of all
  // tiles (so at most one tile more than any other workgroup), taken in
  // blocks of four; tiles past t1 in a last partial block cost their waves
  // no MFMAs and are not stored.
  const int ntile = (a.K + 15) >> 4;
  const int t0 = (int)(((long long)blockIdx.x * ntile) / gridDim.x);
  const int t1 = (int)(((long long)(blockIdx.x + 1) * ntile) / gridDim.x);
  const int nmine = (t1 - t0 + 3) >> 2;
  constexpr int RING = rot_ring(USE_Y, USE_SD);
  constexpr int G = NCH / gcd_c(NCH, RING) * RING;
  const int nitems = nmine * NCH;
  auto kcol = [&](int q) { return (t0 + 4 * (q / NCH)) * 16; };  // first column of q's block
  // Branch-free loads (clamped to valid rows and columns) so that the
  // ring's loads stay in flight: rows i >= ni meet zero rows of the staged
  // M, columns k >= K produce outputs that are not stored.
  auto load = [&](int q, XFrag& d) __attribute__((always_inline)) {
    const int kb = kcol(q), ic = q % NCH;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int i = min(ic * 16 + 4 * s + g, a.ni - 1);
#pragma unroll
      for (int y = 0; y < 2; y++) {
        const int k = min(kb + 16 * (kt0 + y) + l16, a.K - 1);
        d.v[s][y] = a.X[(size_t)i * a.ldx + k];
      }
    }
  };
  v4d acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 2; y++) acc[x][y] = vzero();
  double yold[USE_Y ? 2 : 1][2][4], pold[USE_SD ? 2 : 1][2][4], dm[2];
  auto preload = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
    for (int y = 0; y < 2; y++) {
      const int k = min(kb + 16 * (kt0 + y) + l16, a.K - 1);
      if (USE_SD) dm[y] = a.dtm[k >> 1];
#pragma unroll
      for (int x = 0; x < 2; x++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int j = min(jb + 16 * x + g + 4 * v, a.n - 1);
          if (USE_Y) yold[x][y][v] = a.Y[(size_t)j * a.ldx + k];
          if (USE_SD) pold[x][y][v] = a.sd_psi[(size_t)j * a.ldx + k];
        }
    }
  };
  double fn = 0.0;
  // output of one k-block: Y = beta Y + s(k) acc, optionally the SD update
  auto epilogue = [&](int kb) __attribute__((always_inline)) {
    if (USE_SD) __syncthreads();  // all waves are done reading these X columns
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int y = 0; y < 2; y++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int j = jb + 16 * x + g + 4 * v;
          const int k = kb + 16 * (kt0 + y) + l16;
          const double s = (k < a.k_lo) ? a.s_lo : a.s_hi;
          double val = s * acc[x][y][v];
          if (USE_Y) val = a.beta * yold[USE_Y ? x : 0][y][v] + val;
          if (j < a.n && k < a.K && (kb >> 4) + kt0 + y < t1) {
            a.Y[(size_t)j * a.ldx + k] = val;
            if (USE_SD)
              a.sd_psi[(size_t)j * a.ldx + k] = pold[USE_SD ? x : 0][y][v] + dm[y] * val;
            if (a.fpart) fn += val * val;
          }
          acc[x][y][v] = 0.0;
        }
  };
  // Every load below is issued on every path (items and blocks past the
  // workgroup's share load clamped addresses and are never stored): a
  // load that only some paths issue makes the compiler wait for all.
  XFrag ring[RING];
  static_for<0, RING>([&](auto dc) __attribute__((always_inline)) {
    constexpr int d = decltype(dc)::value;
    load(d, ring[d]);
  });
  {  // stage M: every load of a thread is issued before its LDS stores
    constexpr int PER = 16 * NCH * 128 / kRotThreads;
    double mv[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const int e = tid + kRotThreads * u, i = e >> 7, j = e & 127;
      const double m = a.M[(size_t)min(i, a.ni - 1) * a.n + min(j, a.n - 1)];
      mv[u] = (i < a.ni && j < a.n) ? m : 0.0;
    }
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const int e = tid + kRotThreads * u, i = e >> 7, j = e & 127;
      msm[i * kRotLd + j] = mv[u];
    }
  }
  __syncthreads();
  if (nitems > 0) {
    // the epilogue's operands are loaded PRE items before the block ends
    // (short register lifetime, still behind MFMAs)
    constexpr int PRE = NCH >= 3 ? NCH - 3 : 0;
    for (int q0 = 0; q0 < nitems; q0 += G) {
      static_for<0, G>([&](auto dc) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value;
        constexpr int sl = d % RING, ic = d % NCH;  // q0 is a multiple of G
        const int q = q0 + d;
        const int tb = t0 + 4 * (q / NCH) + kt0;  // this wave's first tile of the block
        const bool v0 = wact && tb < t1, v1 = wact && tb + 1 < t1;
        if (v0) {
#pragma unroll
          for (int s = 0; s < 4; s++) {
            const double* mrow = msm + (ic * 16 + 4 * s + g) * kRotLd + jb + l16;
            const double am0 = mrow[0], am1 = mrow[16];
            acc[0][0] = mfma16(am0, ring[sl].v[s][0], acc[0][0]);
            acc[1][0] = mfma16(am1, ring[sl].v[s][0], acc[1][0]);
            if (v1) {
              acc[0][1] = mfma16(am0, ring[sl].v[s][1], acc[0][1]);
              acc[1][1] = mfma16(am1, ring[sl].v[s][1], acc[1][1]);
            }
          }
        }
        if (ic == PRE) preload(kcol(q));
        load(q + RING, ring[sl]);
        if (ic == NCH - 1 && q < nitems) epilogue(kcol(q));
      });
    }
  }
  if (a.fpart) {
    for (int o = 32; o > 0; o >>= 1) fn += __shfl_down(fn, o, 64);
    if (lane == 0) red[wave] = fn;
    __syncthreads();
    if (tid == 0) {
      double t = 0.0;
#pragma unroll
      for (int w = 0; w < kRotThreads / 64; w++) t += red[w];
      a.fpart[blockIdx.x] = t;
    }
  }
}

static int rotate_pgrid(int K) {
  return std::max(1, std::min(cu_count(), (K + kRK - 1) / kRK));
}

int rotate_nwg(int n, int K) {
  return n <= 128 ? rotate_pgrid(K) : ((K + kRK - 1) / kRK) * rw_shape(n, K).blocks;
}

hipError_t rotate_f64(const RotArgs& args, hipStream_t st) {
  RotArgs a = args;
  if (a.ni <= 0) a.ni = a.n;
  if (a.sd_psi && (a.n > 128 || a.ni > 128)) return hipErrorInvalidValue;
  if (a.fpart && a.n <= 128 && a.ni > 128) return hipErrorInvalidValue;
  if (a.sd_psi && (a.sd_psi != a.X || !a.dtm || !a.fpart || a.ni != a.n))
    return hipErrorInvalidValue;
  if (a.n <= 128 && a.ni <= 128) {
    const int nch = (a.ni + 15) >> 4;
    // [chunk-count variant][epilogue mode: Y read (beta != 0), SD update]
    const int v = 4 * (nch <= 1 ? 0 : nch <= 2 ? 1 : nch <= 4 ? 2 : 3) +
                  (a.beta != 0.0 ? 1 : 0) + (a.sd_psi ? 2 : 0);
#define OA_ROT(nc) k_rotate_p<nc, false, false>, k_rotate_p<nc, true, false>, \
                   k_rotate_p<nc, false, true>, k_rotate_p<nc, true, true>
    void (*const fns[16])(RotArgs) = {OA_ROT(1), OA_ROT(2), OA_ROT(4), OA_ROT(8)};
#undef OA_ROT
    const size_t sm = rot_smem(1 << (v >> 2));
    if (const hipError_t e = grant_lds((const void*)fns[v], sm); e != hipSuccess) return e;
    hipLaunchKernelGGL(fns[v], dim3(rotate_pgrid(a.K)), dim3(kRotThreads), sm, st, a);
    return hipGetLastError();
  }
  if (a.ldx % kRK) return hipErrorInvalidValue;  // whole 64-column blocks inside a row
  const RwShape sh = rw_shape(a.n, a.K);
  const bool y = a.beta != 0.0;
  void (*const fn)(RotArgs) = sh.jt == 4   ? (y ? k_rotate_w<4, true> : k_rotate_w<4, false>)
                              : sh.jt == 3 ? (y ? k_rotate_w<3, true> : k_rotate_w<3, false>)
                                           : (y ? k_rotate_w<2, true> : k_rotate_w<2, false>);
  hipLaunchKernelGGL(fn, dim3((a.K + kRK - 1) / kRK, sh.blocks), dim3(64 * sh.waves), 0, st, a);
  return hipGetLastError();
}

// ================================================================== Newton-Schulz
// Workgroup = 32 x 32 tile of the n x n matrices, wave = 16 x 16 block.
#define NT 32
constexpr int kNsKP = 128;            // k panel width
constexpr int kNsLd = kNsKP + 1;      // LDS row stride of a row panel
constexpr int kNsCl = NT + 1;         // LDS row stride of a column panel
constexpr int kNsRowPanel = NT * kNsLd;
constexpr int kNsColPanel = kNsKP * kNsCl;
constexpr size_t kNsSmem = (size_t)2 * (kNsRowPanel + kNsColPanel) * sizeof(double);

// Stage A[r0.., k0..k0+KP) (row panel) and B[k0..k0+KP, c0..) (column panel)
// All of a thread's loads are issued before any LDS store, so a panel costs
// one memory latency rather than one per element.
constexpr int kNsPer = NT * kNsKP / 256;  // elements per thread and panel
struct NsPanel {
  double va[kNsPer], vb[kNsPer];
};
__device__ __forceinline__ void ns_load(const double* __restrict__ A,
                                        const double* __restrict__ B, int n, int r0, int c0,
                                        int k0, NsPanel& p) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int u = 0; u < kNsPer; u++) {
    const int e = tid + 256 * u;
    const int r = e / kNsKP, k = e - r * kNsKP;
    p.va[u] = (r0 + r < n && k0 + k < n) ? A[(size_t)(r0 + r) * n + k0 + k] : 0.0;
    const int kb = e / NT, cc = e - kb * NT;
    p.vb[u] = (k0 + kb < n && c0 + cc < n) ? B[(size_t)(k0 + kb) * n + c0 + cc] : 0.0;
  }
}
__device__ __forceinline__ void ns_store(const NsPanel& p, double* As, double* Bs) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int u = 0; u < kNsPer; u++) {
    const int e = tid + 256 * u;
    const int r = e / kNsKP, k = e - r * kNsKP;
    As[r * kNsLd + k] = p.va[u];
    const int kb = e / NT, cc = e - kb * NT;
    Bs[kb * kNsCl + cc] = p.vb[u];
  }
}

__device__ __forceinline__ v4d ns_mma(const double* As, const double* Bs, v4d acc) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  const int wr = wave >> 1, wc = wave & 1;
  const double* ap = As + (16 * wr + l16) * kNsLd + g;
  const double* bp = Bs + g * kNsCl + 16 * wc + l16;
  // four independent accumulator chains keep the matrix pipe busy
  v4d p[4] = {acc, vzero(), vzero(), vzero()};
#pragma unroll
  for (int kk = 0; kk < kNsKP; kk += 16)
#pragma unroll
    for (int u = 0; u < 4; u++)
      p[u] = mfma16(ap[kk + 4 * u], bp[(kk + 4 * u) * kNsCl], p[u]);
  return (p[0] + p[1]) + (p[2] + p[3]);
}

// One (or two) tile products through LDS panels: acc1 = A1 B1 and, if A2,
// acc2 = A2 B2, for the workgroup's tile (r0, c0).
__device__ __forceinline__ void ns_tile2(const double* A1, const double* B1, const double* A2,
                                         const double* B2, int n, int r0, int c0, double* sm,
                                         v4d& acc1, v4d& acc2) {
  double* As1 = sm;
  double* Bs1 = As1 + kNsRowPanel;
  double* As2 = Bs1 + kNsColPanel;
  double* Bs2 = As2 + kNsRowPanel;
  acc1 = vzero();
  acc2 = vzero();
  for (int k0 = 0; k0 < n; k0 += kNsKP) {
    NsPanel p;
    ns_load(A1, B1, n, r0, c0, k0, p);
    __syncthreads();  // the previous panels are consumed
    ns_store(p, As1, Bs1);
    if (A2) {
      ns_load(A2, B2, n, r0, c0, k0, p);
      ns_store(p, As2, Bs2);
    }
    __syncthreads();
    acc1 = ns_mma(As1, Bs1, acc1);
    if (A2) acc2 = ns_mma(As2, Bs2, acc2);
  }
}

__device__ __forceinline__ void blk_coords(int nt, int& row0, int& col0) {
  const int wave = threadIdx.x >> 6;
  const int ti = blockIdx.x / nt, tj = blockIdx.x - (blockIdx.x / nt) * nt;
  row0 = ti * NT + (wave >> 1) * 16;
  col0 = tj * NT + (wave & 1) * 16;
}

// store alpha*acc + gamma*I; returns this lane's sum of (Told - new)^2
__device__ __forceinline__ double blk_store(double* __restrict__ C, const v4d& acc, int n,
                                            int row0, int col0, double alpha, double gamma,
                                            const double* __restrict__ Told) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  double e = 0.0;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int row = row0 + g + 4 * v, col = col0 + l16;
    if (row < n && col < n) {
      const double val = alpha * acc[v] + (row == col ? gamma : 0.0);
      C[(size_t)row * n + col] = val;
      if (Told) {
        const double d = Told[(size_t)row * n + col] - val;
        e += d * d;
      }
    }
  }
  return e;
}

__device__ __forceinline__ double wg_sum(double v) {
  __shared__ double red[4];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const double t = red[0] + red[1] + red[2] + red[3];
  __syncthreads();
  return t;
}

// rms change of iteration `it` from the per-workgroup partials (same order
// in every workgroup, so every workgroup takes the same decision)
__device__ __forceinline__ double ns_err(const double* __restrict__ errpart, int it, int nwg,
                                         int n) {
  __shared__ double bcast;
  if (threadIdx.x == 0) {
    double s = 0.0;
    const double* ep = errpart + (size_t)it * nwg;
    for (int w = 0; w < nwg; w++) s += ep[w];
    bcast = sqrt(s / ((double)n * n));
  }
  __syncthreads();
  const double e = bcast;
  __syncthreads();
  return e;
}

// One launch for the whole iteration (cooperative, all workgroups resident):
// X0 = S/2, T0 = I; loop { C = 3I - T X; X' = X C / 2; T' = C T / 2 } with
// two grid barriers per iteration; stops when the rms change of T <= tol.
__global__ __launch_bounds__(256) void k_ns_coop(NsArgs a) {
  namespace cg = cooperative_groups;
  extern __shared__ __align__(16) double ns_smem[];
  cg::grid_group grid = cg::this_grid();
  const int n = a.n, nt = (n + NT - 1) / NT, nwg = nt * nt;
  const int r0 = (blockIdx.x / nt) * NT, c0 = (blockIdx.x % nt) * NT;
  int row0, col0;
  blk_coords(nt, row0, col0);
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int row = row0 + g + 4 * v, col = col0 + l16;
    if (row < n && col < n) {
      a.X0[(size_t)row * n + col] = 0.5 * a.S[(size_t)row * n + col];  // B = S/2 (ortho.C:236-239)
      a.T0[(size_t)row * n + col] = (row == col) ? 1.0 : 0.0;
    }
  }
  grid.sync();
  double* X[2] = {a.X0, a.X1};
  double* T[2] = {a.T0, a.T1};
  int conv = 0;
  double err = 0.0;
  for (int it = 1; it <= a.max_iter; it++) {
    const int o = (it - 1) & 1, w = it & 1;
    v4d p1, p2;
    ns_tile2(T[o], X[o], nullptr, nullptr, n, r0, c0, ns_smem, p1, p2);
    blk_store(a.C, p1, n, row0, col0, -1.0, 3.0, nullptr);
    grid.sync();
    ns_tile2(X[o], a.C, a.C, T[o], n, r0, c0, ns_smem, p1, p2);
    blk_store(X[w], p1, n, row0, col0, 0.5, 0.0, nullptr);
    const double e = blk_store(T[w], p2, n, row0, col0, 0.5, 0.0, T[o]);
    const double es = wg_sum(e);
    if (threadIdx.x == 0) a.errpart[(size_t)it * nwg + blockIdx.x] = es;
    grid.sync();
    err = ns_err(a.errpart, it, nwg, n);
    if (err <= a.tol) {
      conv = it;
      break;
    }
  }
  const int last = conv ? conv : a.max_iter;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.res->ns_iter = conv ? conv : -a.max_iter;
    a.res->ns_err = err;
  }
  const double* Tf = T[last & 1];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int row = row0 + g + 4 * v, col = col0 + l16;
    if (row < n && col < n) a.Tout[(size_t)row * n + col] = Tf[(size_t)row * n + col];
  }
}

// One workgroup for the whole iteration, a plain launch (n <= kNsOneMax): X, T
// and C stay in LDS (zero past n, odd row stride), a wave computes 16 x 16 tiles;
// the new X = X C / 2 and T = C T / 2 wait in registers until every wave has read the
// old ones.  (C X / 2 is the same matrix, but with C = 3I - T X an error of X then
// grows by up to half the square root of S's eigenvalue ratio in every iteration.)  Bound by
// the matrix pipe of one CU at n = 64 and by the dependent products and three
// barriers per iteration below; no operand leaves the CU.  The stage of a step
// (4 to 5 iterations) takes 15 us at 16 states, and 64 states 37; the cooperative
// and single-workgroup forms through global memory took 49 and 50.
__global__ __launch_bounds__(1024) void k_ns_one(NsArgs a) {
  constexpr int LD = kNsOneMax + 1;
  extern __shared__ __align__(16) double ns_smem[];
  __shared__ double red[16];
  double *X = ns_smem, *T = X + kNsOneMax * LD, *C = T + kNsOneMax * LD;
  const int n = a.n, nt = (n + 15) >> 4, np = 16 * nt, tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int nw = blockDim.x >> 6;
  for (int e = tid; e < np * np; e += blockDim.x) {
    const int r = e / np, c = e - r * np;
    const bool in = r < n && c < n;
    X[r * LD + c] = in ? 0.5 * a.S[(size_t)r * n + c] : 0.0;  // B = S/2 (ortho.C:236-239)
    T[r * LD + c] = in && r == c ? 1.0 : 0.0;
  }
  __syncthreads();
  // rows 16 ti.. of A times columns 16 tj.. of B
  auto product = [&](const double* A, const double* B, int ti, int tj) {
    const double* ap = A + (16 * ti + l16) * LD + g;
    const double* bp = B + g * LD + 16 * tj + l16;
    v4d p0 = vzero(), p1 = vzero();
    for (int k = 0; k < np; k += 16) {  // two accumulator chains
      p0 = mfma16(ap[k], bp[k * LD], p0);
      p1 = mfma16(ap[k + 4], bp[(k + 4) * LD], p1);
      p0 = mfma16(ap[k + 8], bp[(k + 8) * LD], p0);
      p1 = mfma16(ap[k + 12], bp[(k + 12) * LD], p1);
    }
    return p0 + p1;
  };
  int conv = 0;
  double err = 0.0;
  for (int it = 1; it <= a.max_iter; it++) {
    for (int t = wave; t < nt * nt; t += nw) {  // C = 3I - T X
      const int ti = t / nt, tj = t - ti * nt;
      const v4d p = product(T, X, ti, tj);
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = 16 * ti + g + 4 * v, c = 16 * tj + l16;
        C[r * LD + c] = (r == c && r < n ? 3.0 : 0.0) - p[v];
      }
    }
    __syncthreads();
    // tiles q = wave and wave + nw of the 2 nt^2: the X tiles, then the T tiles
    v4d p[2];
    double e = 0.0;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int q = wave + i * nw, t = q < nt * nt ? q : q - nt * nt;
      if (q >= 2 * nt * nt) continue;
      const int ti = t / nt, tj = t - ti * nt;
      p[i] = product(q < nt * nt ? X : C, q < nt * nt ? C : T, ti, tj) * 0.5;
      if (q >= nt * nt)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const double d = T[(16 * ti + g + 4 * v) * LD + 16 * tj + l16] - p[i][v];
          e += d * d;
        }
    }
    for (int off = 32; off > 0; off >>= 1) e += __shfl_down(e, off, 64);
    if (lane == 0) red[wave] = e;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int q = wave + i * nw, t = q < nt * nt ? q : q - nt * nt;
      if (q >= 2 * nt * nt) continue;
      const int ti = t / nt, tj = t - ti * nt;
      double* D = q < nt * nt ? X : T;
#pragma unroll
      for (int v = 0; v < 4; v++) D[(16 * ti + g + 4 * v) * LD + 16 * tj + l16] = p[i][v];
    }
    double sum = 0.0;
    for (int w = 0; w < nw; w++) sum += red[w];
    err = sqrt(sum / ((double)n * n));
    __syncthreads();
    if (err <= a.tol) {
      conv = it;
      break;
    }
  }
  if (tid == 0) {
    a.res->ns_iter = conv ? conv : -a.max_iter;
    a.res->ns_err = err;
  }
  for (int e = tid; e < n * n; e += blockDim.x) {
    const int r = e / n, c = e - r * n;
    a.Tout[e] = T[r * LD + c];
  }
}

// threads of a k_ns_one launch: a wave per two of the 2 nt^2 tiles, at most 16
static int ns_one_threads(int n) {
  const int nt = (n + 15) / 16;
  return 64 * std::min(16, nt * nt);
}
constexpr size_t kNsOneSmem = (size_t)3 * kNsOneMax * (kNsOneMax + 1) * sizeof(double);

// ---- fallback: two launches per iteration with a device-side early exit

// 16x16 block (row0, col0) of A B straight from global memory
__device__ __forceinline__ v4d blk_gemm(const double* __restrict__ A,
                                        const double* __restrict__ B, int n, int row0,
                                        int col0) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int r = row0 + l16, cc = col0 + l16;
  v4d acc = vzero();
  for (int k0 = 0; k0 < n; k0 += 4) {
    const int k = k0 + g;
    const double av = (r < n && k < n) ? A[(size_t)r * n + k] : 0.0;
    const double bv = (k < n && cc < n) ? B[(size_t)k * n + cc] : 0.0;
    acc = mfma16(av, bv, acc);
  }
  return acc;
}

__global__ void k_ns_init(const double* __restrict__ S, double* __restrict__ X0,
                          double* __restrict__ T0, int n, StepDev* res) {
  const size_t nn = (size_t)n * n;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < nn;
       e += (size_t)gridDim.x * blockDim.x) {
    X0[e] = S[e] * 0.5;
    const size_t i = e / n, j = e - i * n;
    T0[e] = (i == j) ? 1.0 : 0.0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    res->ns_iter = 0;
    res->ns_err = 0.0;
  }
}

// FP64 iterations this launch sequence may run: max_iter, less the FP32
// iterations before it in the mixed-precision form
__device__ __forceinline__ int ns_limit(int max_iter, int mixed, const StepDev* res) {
  return mixed ? max_iter - *(volatile const int*)&res->ns32_iter : max_iter;
}

// True when iteration `it` must not run (converged before it, or past the
// limit).  Thread 0 decides and broadcasts, so the whole workgroup takes the
// same path.
__device__ bool ns_skip(const double* __restrict__ errpart, int it, int nwg, int n, double tol,
                        StepDev* res, bool record, int lim) {
  __shared__ int skip;
  if (threadIdx.x == 0) {
    int f = 0;
    if (it > lim || *(volatile int*)&res->ns_iter != 0) {
      f = 1;
    } else if (it > 1) {
      double s = 0.0;
      const double* ep = errpart + (size_t)(it - 1) * nwg;
      for (int w = 0; w < nwg; w++) s += ep[w];
      const double err = sqrt(s / ((double)n * n));
      if (err <= tol) {
        f = 1;
        if (record && blockIdx.x == 0) {
          res->ns_iter = it - 1;
          res->ns_err = err;
        }
      }
    }
    skip = f;
  }
  __syncthreads();
  return skip != 0;
}

__global__ __launch_bounds__(256) void k_ns_step1(const double* __restrict__ T,
                                                  const double* __restrict__ X,
                                                  double* __restrict__ C, int n, int it,
                                                  double tol, const double* errpart,
                                                  StepDev* res, int max_iter, int mixed) {
  const int nt = (n + NT - 1) / NT, nwg = nt * nt;
  if (ns_skip(errpart, it, nwg, n, tol, res, true, ns_limit(max_iter, mixed, res))) return;
  int row0, col0;
  blk_coords(nt, row0, col0);
  blk_store(C, blk_gemm(T, X, n, row0, col0), n, row0, col0, -1.0, 3.0, nullptr);
}

__global__ __launch_bounds__(256) void k_ns_step23(const double* __restrict__ Xo,
                                                   const double* __restrict__ To,
                                                   const double* __restrict__ C,
                                                   double* __restrict__ Xn,
                                                   double* __restrict__ Tn, int n, int it,
                                                   double tol, double* errpart, StepDev* res,
                                                   int max_iter, int mixed) {
  const int nt = (n + NT - 1) / NT, nwg = nt * nt;
  if (ns_skip(errpart, it, nwg, n, tol, res, false, ns_limit(max_iter, mixed, res))) return;
  int row0, col0;
  blk_coords(nt, row0, col0);
  blk_store(Xn, blk_gemm(Xo, C, n, row0, col0), n, row0, col0, 0.5, 0.0, nullptr);
  const double e = blk_store(Tn, blk_gemm(C, To, n, row0, col0), n, row0, col0, 0.5, 0.0, To);
  const double es = wg_sum(e);
  if (threadIdx.x == 0) errpart[(size_t)it * nwg + blockIdx.x] = es;
}

__global__ void k_ns_final(const double* __restrict__ errpart, int nwg, int n, int max_iter,
                           double tol, StepDev* res, int mixed) {
  if (threadIdx.x != 0) return;
  if (res->ns_iter != 0) return;
  const int lim = ns_limit(max_iter, mixed, res);
  double s = 0.0;
  const double* ep = errpart + (size_t)lim * nwg;
  for (int w = 0; w < nwg; w++) s += ep[w];
  const double err = sqrt(s / ((double)n * n));
  res->ns_err = err;
  res->ns_iter = (err <= tol) ? lim : -lim;
}

__global__ void k_ns_copy(const double* __restrict__ T0, const double* __restrict__ T1,
                          double* __restrict__ Tout, int n, const StepDev* res) {
  const int it = res->ns_iter < 0 ? -res->ns_iter : res->ns_iter;
  const double* src = (it & 1) ? T1 : T0;
  const size_t nn = (size_t)n * n;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < nn;
       e += (size_t)gridDim.x * blockDim.x)
    Tout[e] = src[e];
}

// X = (S/2) T in FP64, before each FP64 iteration of the mixed-precision
// form.  The coupled iteration keeps X = (S/2) T and sees S only through X,
// so it cannot remove an error of T that does not commute with S (an FP32
// T's): it converges to within that error (measured 1e-10 .. 1e-7).  With X
// rebuilt from the exact S, the iteration is T' = (3I - T (S/2) T) T / 2,
// which corrects such errors quadratically.
__global__ __launch_bounds__(256) void k_ns_x_from_t(const double* __restrict__ S,
                                                     const double* __restrict__ T,
                                                     double* __restrict__ X, int n, int it,
                                                     double tol, const double* errpart,
                                                     StepDev* res, int max_iter) {
  const int nt = (n + NT - 1) / NT, nwg = nt * nt;
  if (ns_skip(errpart, it, nwg, n, tol, res, false, ns_limit(max_iter, 1, res))) return;
  int row0, col0;
  blk_coords(nt, row0, col0);
  blk_store(X, blk_gemm(S, T, n, row0, col0), n, row0, col0, 0.5, 0.0, nullptr);
}

// init: X0 = S/2, T0 = I; else X0 and T0 are already set (the FP64 phase of
// the mixed-precision iteration)
static hipError_t ns_run_launches(const NsArgs& a, hipStream_t st, bool init = true,
                                  int mixed = 0) {
  const int n = a.n;
  const int nt = (n + NT - 1) / NT;
  const int nwg = nt * nt;
  const size_t nn = (size_t)n * n;
  int eb = (int)((nn + 255) / 256);
  if (eb > 512) eb = 512;
  if (init) hipLaunchKernelGGL(k_ns_init, dim3(eb), dim3(256), 0, st, a.S, a.X0, a.T0, n, a.res);
  double* X[2] = {a.X0, a.X1};
  double* T[2] = {a.T0, a.T1};
  for (int it = 1; it <= a.max_iter; it++) {
    const int o = (it - 1) & 1, w = it & 1;
    if (mixed)
      hipLaunchKernelGGL(k_ns_x_from_t, dim3(nwg), dim3(256), 0, st, a.S, T[o], X[o], n, it,
                         a.tol, a.errpart, a.res, a.max_iter);
    hipLaunchKernelGGL(k_ns_step1, dim3(nwg), dim3(256), 0, st, T[o], X[o], a.C, n, it, a.tol,
                       a.errpart, a.res, a.max_iter, mixed);
    hipLaunchKernelGGL(k_ns_step23, dim3(nwg), dim3(256), 0, st, X[o], T[o], a.C, X[w], T[w], n,
                       it, a.tol, a.errpart, a.res, a.max_iter, mixed);
  }
  hipLaunchKernelGGL(k_ns_final, dim3(1), dim3(64), 0, st, a.errpart, nwg, n, a.max_iter, a.tol,
                     a.res, mixed);
  hipLaunchKernelGGL(k_ns_copy, dim3(eb), dim3(256), 0, st, a.T0, a.T1, a.Tout, n, a.res);
  return hipGetLastError();
}

// ---- FP32 iterations of the mixed-precision Newton-Schulz
//
// The recurrence of get_iter_Tmat (cp_lowdin.C:201-241) on FP32 X, T, C with
// v_mfma_f32_16x16x4f32, two launches per iteration as above, until the rms
// change of T is <= kNs32Switch; the last FP32 T is then widened into the
// FP64 T0, and FP64 iterations with X = (S/2) T rebuilt from the exact S
// continue to the step's tolerance (k_ns_x_from_t): they remove the FP32
// error quadratically, and T meets the same tolerance as an FP64 run.
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4f mfma16f(float a, float b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// 16x16 block (row0, col0) of A B in FP32.  A lane holds A[r][k] and B[k][c]
// with r, c = lane % 16 and k = lane / 16, as in FP64; the FP32 accumulator
// element v of lane l is D[4 (l/16) + v][l % 16] (FP64: D[l/16 + 4 v]).
__device__ __forceinline__ v4f blk_gemm32(const float* __restrict__ A,
                                          const float* __restrict__ B, int n, int row0,
                                          int col0) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int r = row0 + l16, cc = col0 + l16;
  v4f acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < n; k0 += 4) {
    const int k = k0 + g;
    const float av = (r < n && k < n) ? A[(size_t)r * n + k] : 0.f;
    const float bv = (k < n && cc < n) ? B[(size_t)k * n + cc] : 0.f;
    acc = mfma16f(av, bv, acc);
  }
  return acc;
}

// C = alpha acc + gamma I on the block; returns sum (Told - C)^2 if Told
__device__ __forceinline__ double blk_store32(float* __restrict__ C, const v4f& acc, int n,
                                              int row0, int col0, float alpha, float gamma,
                                              const float* __restrict__ Told) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  double e = 0.0;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int row = row0 + 4 * g + v, col = col0 + l16;
    if (row < n && col < n) {
      const float val = alpha * acc[v] + (row == col ? gamma : 0.f);
      C[(size_t)row * n + col] = val;
      if (Told) {
        const double d = (double)Told[(size_t)row * n + col] - (double)val;
        e += d * d;
      }
    }
  }
  return e;
}

__global__ void k_ns32_init(const double* __restrict__ S, float* __restrict__ X0,
                            float* __restrict__ T0, int n, StepDev* res) {
  const size_t nn = (size_t)n * n;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < nn;
       e += (size_t)gridDim.x * blockDim.x) {
    X0[e] = (float)(S[e] * 0.5);
    const size_t i = e / n, j = e - i * n;
    T0[e] = (i == j) ? 1.f : 0.f;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) res->ns32_iter = 0;
}

// True when FP32 iteration `it` must not run: the switch test passed before
// it (recorded in ns32_iter by the first workgroup of step 1).
__device__ bool ns32_skip(const double* __restrict__ errpart, int it, int nwg, int n,
                          StepDev* res, bool record) {
  __shared__ int skip;
  if (threadIdx.x == 0) {
    int f = 0;
    if (*(volatile int*)&res->ns32_iter != 0) {
      f = 1;
    } else if (it > 1) {
      double s = 0.0;
      const double* ep = errpart + (size_t)(it - 1) * nwg;
      for (int w = 0; w < nwg; w++) s += ep[w];
      if (sqrt(s / ((double)n * n)) <= kNs32Switch) {
        f = 1;
        if (record && blockIdx.x == 0) res->ns32_iter = it - 1;
      }
    }
    skip = f;
  }
  __syncthreads();
  return skip != 0;
}

__global__ __launch_bounds__(256) void k_ns32_step1(const float* __restrict__ T,
                                                    const float* __restrict__ X,
                                                    float* __restrict__ C, int n, int it,
                                                    const double* errpart, StepDev* res) {
  const int nt = (n + NT - 1) / NT, nwg = nt * nt;
  if (ns32_skip(errpart, it, nwg, n, res, true)) return;
  int row0, col0;
  blk_coords(nt, row0, col0);
  blk_store32(C, blk_gemm32(T, X, n, row0, col0), n, row0, col0, -1.f, 3.f, nullptr);
}

__global__ __launch_bounds__(256) void k_ns32_step23(const float* __restrict__ Xo,
                                                     const float* __restrict__ To,
                                                     const float* __restrict__ C,
                                                     float* __restrict__ Xn,
                                                     float* __restrict__ Tn, int n, int it,
                                                     double* errpart, StepDev* res) {
  const int nt = (n + NT - 1) / NT, nwg = nt * nt;
  if (ns32_skip(errpart, it, nwg, n, res, false)) return;
  int row0, col0;
  blk_coords(nt, row0, col0);
  blk_store32(Xn, blk_gemm32(Xo, C, n, row0, col0), n, row0, col0, 0.5f, 0.f, nullptr);
  const double e =
      blk_store32(Tn, blk_gemm32(C, To, n, row0, col0), n, row0, col0, 0.5f, 0.f, To);
  const double es = wg_sum(e);
  if (threadIdx.x == 0) errpart[(size_t)it * nwg + blockIdx.x] = es;
}

// T of the last FP32 iterate (all max32 ran when none passed the switch
// test) widened into the FP64 T0
__global__ void k_ns32_widen(const float* __restrict__ T0f, const float* __restrict__ T1f,
                             double* __restrict__ T0, int n, int max_iter, StepDev* res) {
  int k = *(volatile int*)&res->ns32_iter;
  if (k == 0) k = max_iter;
  const float* T = (k & 1) ? T1f : T0f;
  const size_t nn = (size_t)n * n;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < nn;
       e += (size_t)gridDim.x * blockDim.x)
    T0[e] = (double)T[e];
}


__global__ void k_ns32_final(int max_iter, StepDev* res) {
  if (threadIdx.x == 0 && res->ns32_iter == 0) res->ns32_iter = max_iter;
  if (threadIdx.x == 0) {
    res->ns_iter = 0;
    res->ns_err = 0.0;
  }
}

hipError_t ns_run_mixed(const NsArgs& a, const Ns32Bufs& b, hipStream_t st) {
  const int n = a.n;
  const int nt = (n + NT - 1) / NT;
  const int nwg = nt * nt;
  const size_t nn = (size_t)n * n;
  int eb = (int)((nn + 255) / 256);
  if (eb > 512) eb = 512;
  hipLaunchKernelGGL(k_ns32_init, dim3(eb), dim3(256), 0, st, a.S, b.X0, b.T0, n, a.res);
  float* X[2] = {b.X0, b.X1};
  float* T[2] = {b.T0, b.T1};
  const int max32 = a.max_iter > 1 ? a.max_iter - 1 : 1;  // leaves at least one FP64 iteration
  for (int it = 1; it <= max32; it++) {
    const int o = (it - 1) & 1, w = it & 1;
    hipLaunchKernelGGL(k_ns32_step1, dim3(nwg), dim3(256), 0, st, T[o], X[o], b.C, n, it,
                       a.errpart, a.res);
    hipLaunchKernelGGL(k_ns32_step23, dim3(nwg), dim3(256), 0, st, X[o], T[o], b.C, X[w], T[w],
                       n, it, a.errpart, a.res);
  }
  // the widening reads ns32_iter before k_ns32_final sets "all ran"
  hipLaunchKernelGGL(k_ns32_widen, dim3(eb), dim3(256), 0, st, b.T0, b.T1, a.T0, n, max32,
                     a.res);
  hipLaunchKernelGGL(k_ns32_final, dim3(1), dim3(64), 0, st, max32, a.res);
  return ns_run_launches(a, st, false, 1);
}

// ---- block-row variant: one grid barrier per iteration
//
// Workgroup (b, h) owns rows R = [16b, 16b + 16) and the 16-column tiles
// ct = h, h + split, h + 2 split, ... of X and T (split = gridDim.y).  With
// C = 3I - T X the new X = X C / 2 of the recurrence is D X / 2, D = 3I - X T,
// and the new tiles
//   T'[R,ct] = C[R,:] T[:,ct] / 2,  X'[R,ct] = D[R,:] X[:,ct] / 2
// need only rows of C and D, which every workgroup of the row block computes
// whole, one after the other in the same LDS rows, and the previous X and T.
// (C X / 2, which would need no D, multiplies rounding errors: see k_ns_one.)
// X and T go through global memory (double buffered) for the other
// workgroups.  Iteration 1 starts from T0 = I and X0 = S/2 (ortho.C:236-239):
// there C = D = 3I - S/2 and T1 = C/2 need no products, so no barrier precedes
// it.  After each barrier the next iteration's operands are loaded before
// the convergence test reads the error partials, so the two latencies
// overlap.  MFMA operands: A from LDS, B from global memory in batches of KB
// k-steps, branch-free (clamped addresses, masked values): a load that only
// some paths use is waited for on its own.
constexpr int kNrWaves = 8;
constexpr int kNrMaxWg = 256;  // error partials staged in LDS
// k-steps per B batch (two batches in registers at a time)
__host__ __device__ constexpr int nr_kb(int n) { return n <= 32 ? 8 : 16; }
// LDS row length: whole batches of k-steps (columns past n zero), + 2
// against bank conflicts
__host__ __device__ constexpr int nr_ld(int n) {
  return 4 * ((((n + 3) >> 2) + nr_kb(n) - 1) / nr_kb(n) * nr_kb(n)) + 2;
}
size_t ns_rows_smem(int n) { return (size_t)2 * 16 * nr_ld(n) * sizeof(double); }

// b[u] = scale * B[k][col] for the k-steps k0 .. k0 + KB - 1 of this lane
// group (k = 4 (k0 + u) + g): each load covers four rows of 16 contiguous
// columns.  k past n is clamped to the last row (finite values that meet
// zero A columns), col past n to the last column (results not stored): no
// per-k masks, which the compiler would hoist as scalar pairs and spill.
// Buffer loads: a scalar resource and one 32-bit offset register per load
// (n * n * 8 < 2^31), where flat addressing holds a register pair each.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t nr_rsrc(const double* p, int n) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(p), (short)0, n * n * 8,
                                           0x00020000);  // raw buffer, gfx9 data format
}

template <int KB>
__device__ __forceinline__ void nr_load(double (&b)[KB], rsrc_t B, int col, int n, int k0,
                                        double scale) {
  const int g = (threadIdx.x & 63) >> 4;
  const int colc = min(col, n - 1);
#pragma unroll
  for (int u = 0; u < KB; u++) {
    const int k = min((k0 + u) * 4 + g, n - 1);
    const double v = __builtin_bit_cast(
        double, __builtin_amdgcn_raw_buffer_load_b64(B, (k * n + colc) * 8, 0, 0));
    b[u] = scale * v;
  }
}

// acc += A[16 LDS rows][k] b over one batch (A columns past n are zero)
template <int KB>
__device__ __forceinline__ v4d nr_mma(const double* __restrict__ Al, int ld, const double (&b)[KB],
                                      int k0, v4d acc) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const double* __restrict__ a = Al + l16 * ld + 4 * k0 + g;
#pragma unroll
  for (int u = 0; u < KB; u++) acc = mfma16(a[4 * u], b[u], acc);
  return acc;
}

// A[16 LDS rows][0, n) B[0, n)[col tile]; b holds the first batch on entry
template <int KB>
__device__ __forceinline__ v4d nr_product(const double* __restrict__ Al, int ld, double (&b)[KB],
                                          rsrc_t B, int col, int n, double scale) {
  const int nk = (n + 3) >> 2;
  v4d acc = vzero();
#pragma nounroll
  for (int k0 = 0;; k0 += KB) {
    // the next batch is in flight while this one's MFMAs issue
    double nx[KB];
    const bool more = k0 + KB < nk;
    if (more) nr_load<KB>(nx, B, col, n, k0 + KB, scale);
    acc = nr_mma<KB>(Al, ld, b, k0, acc);
    if (!more) break;
#pragma unroll
    for (int u = 0; u < KB; u++) b[u] = nx[u];
  }
  return acc;
}

template <int KB>
__global__ __launch_bounds__(kNrWaves * 64) void k_ns_rows(NsArgs a) {
  namespace cg = cooperative_groups;
  static_assert(kNrWaves * 64 == 16 * 32, "A panel staging: 32 threads per row");
  extern __shared__ __align__(16) double nr_smem[];
  __shared__ double red[kNrWaves];
  __shared__ double epart[kNrMaxWg];
  __shared__ double bcast;
  cg::grid_group grid = cg::this_grid();
  const int nb = gridDim.x, split = gridDim.y;
  const int wg = blockIdx.y * nb + blockIdx.x, nwg = nb * split, h = blockIdx.y;
  const int r0 = 16 * blockIdx.x, tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int pr = tid >> 5, pk = tid & 31;  // A panel staging: row, first column
  constexpr int nthr = kNrWaves * 64;
  double bc[KB], bx[KB], ap[4];  // ap: rows R of T, columns pk + 32 q
  {
    const int n = a.n, ld = nr_ld(n);
    double* Tr = nr_smem;       // [16][ld]: rows R of the previous T, then of X
    double* Cr = Tr + 16 * ld;  // [16][ld]: rows R of C, then of D
    // iteration 1: T0 = I, C = 3I - S/2; LDS zero past n in both directions
    for (int e = tid; e < 16 * ld; e += nthr) {
      const int r = e / ld, k = e - r * ld, row = r0 + r;
      const bool in = row < n && k < n;
      const double sv = a.S[(size_t)min(row, n - 1) * n + min(k, n - 1)];
      Tr[e] = (in && row == k) ? 1.0 : 0.0;
      Cr[e] = in ? (row == k ? 3.0 : 0.0) - 0.5 * sv : 0.0;
    }
  }
  __syncthreads();
  int conv = 0;
  double err = 0.0;
  for (int it = 1; it <= a.max_iter; it++) {
    // n and what derives from it are recomputed in every iteration instead
    // of being hoisted into registers that the operand batches need
    int n = a.n;
    asm volatile("" : "+s"(n));
    const int ld = nr_ld(n), nct = (n + 15) >> 4, nown = (nct - h + split - 1) / split;
    double* Tr = nr_smem;
    double* Cr = Tr + 16 * ld;
    // X_k and T_k live in buffer k & 1
    const double *To = (it & 1) ? a.T0 : a.T1, *Xo = (it & 1) ? a.X0 : a.X1;
    double* Xw = (it & 1) ? a.X1 : a.X0;
    double* Tw = (it & 1) ? a.T1 : a.T0;
    double e = 0.0;
    // m = 0: C = 3I - T X and the own tiles of T' = C T / 2, m = 1: D = 3I - X T and
    // X' = D X / 2
#pragma nounroll
    for (int m = 0; m < 2; m++) {
      const rsrc_t rO = nr_rsrc(m ? Xo : To, n);
      if (it > 1) {
        if (m) __syncthreads();  // every wave has read the rows of C and T
        const bool rin = r0 + pr < n;
        const double* P = (m ? Xo : To) + (size_t)min(r0 + pr, n - 1) * n;
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (rin && pk + 32 * q < n) Tr[pr * ld + pk + 32 * q] = m ? P[pk + 32 * q] : ap[q];
        for (int k = pk + 128; k < n; k += 32)
          if (rin) Tr[pr * ld + k] = P[k];
        __syncthreads();
        const rsrc_t rQ = nr_rsrc(m ? To : Xo, n);
#pragma nounroll
        for (int ct = wave, i = 0; ct < nct; ct += kNrWaves, i++) {
          const int col = ct * 16 + l16;
          if (i > 0 || m) nr_load<KB>(bc, rQ, col, n, 0, 1.0);
          const v4d acc = nr_product<KB>(Tr, ld, bc, rQ, col, n, 1.0);
#pragma unroll
          for (int v = 0; v < 4; v++) {
            const int r = g + 4 * v, row = r0 + r;
            if (col < n) Cr[r * ld + col] = (row < n ? (row == col ? 3.0 : 0.0) - acc[v] : 0.0);
          }
        }
        __syncthreads();
      }
#pragma nounroll
      for (int q = wave, i = 0; q < nown; q += kNrWaves, i++) {
        const int col = (h + split * q) * 16 + l16;
        v4d acc;
        if (it == 1 && m == 0) {  // T0 = I: C T0 = C
#pragma unroll
          for (int v = 0; v < 4; v++) acc[v] = Cr[(g + 4 * v) * ld + min(col, ld - 1)];
        } else {
          const rsrc_t B = it == 1 ? nr_rsrc(a.S, n) : rO;  // X0 = S/2
          const double scale = it == 1 ? 0.5 : 1.0;
          if (i > 0 || m) nr_load<KB>(bx, B, col, n, 0, scale);
          acc = nr_product<KB>(Cr, ld, bx, B, col, n, scale);
        }
        double* D = m ? Xw : Tw;
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int r = g + 4 * v, row = r0 + r;
          if (row < n && col < n) {
            const double nv = 0.5 * acc[v];
            D[(unsigned)(row * n + col)] = nv;
            if (m == 0) {  // Tr holds the previous T
              const double d = Tr[r * ld + col] - nv;
              e += d * d;
            }
          }
        }
      }
    }
    {  // workgroup sum in a fixed order
      for (int off = 32; off > 0; off >>= 1) e += __shfl_down(e, off, 64);
      if (lane == 0) red[wave] = e;
      __syncthreads();
      if (tid == 0) {
        double t = 0.0;
        for (int i = 0; i < kNrWaves; i++) t += red[i];
        a.errpart[(size_t)it * nwg + wg] = t;
      }
    }
    grid.sync();
    // the next iteration's first operands, then the error partials
    if (it < a.max_iter) {
      const double* p = Tw + (size_t)min(r0 + pr, n - 1) * n;
#pragma unroll
      for (int q = 0; q < 4; q++) ap[q] = p[min(pk + 32 * q, n - 1)];
      nr_load<KB>(bc, nr_rsrc(Xw, n), wave * 16 + l16, n, 0, 1.0);
      nr_load<KB>(bx, nr_rsrc(Tw, n), (h + split * wave) * 16 + l16, n, 0, 1.0);
    }
    for (int i = tid; i < nwg; i += nthr) epart[i] = a.errpart[(size_t)it * nwg + i];
    __syncthreads();
    if (tid == 0) {
      double sum = 0.0;
      for (int i = 0; i < nwg; i++) sum += epart[i];
      bcast = sqrt(sum / ((double)n * n));
    }
    __syncthreads();
    err = bcast;
    if (err <= a.tol) {
      conv = it;
      break;
    }
  }
  if (wg == 0 && tid == 0) {
    a.res->ns_iter = conv ? conv : -a.max_iter;
    a.res->ns_err = err;
  }
  // this workgroup's tiles of the last iteration's T
  const double* Tl = ((conv ? conv : a.max_iter) & 1) ? a.T1 : a.T0;
  const int n = a.n, nct = (n + 15) >> 4, nown = (nct - h + split - 1) / split;
  for (int e = tid; e < 16 * nown * 16; e += nthr) {
    const int r = e / (16 * nown), t = e - r * 16 * nown;
    const int row = r0 + r, col = (h + split * (t >> 4)) * 16 + (t & 15);
    if (row < n && col < n) a.Tout[(size_t)row * n + col] = Tl[(size_t)row * n + col];
  }
}

// ---- plain launches by tiles, then one that finishes
//
// A launch boundary takes the place of the grid barrier: about 3 us against 30 us
// for entering a cooperative launch and 8 us per barrier.  C = 3I - T X in one
// launch, X' = X C / 2 and T' = C T / 2 in the next; a workgroup computes one
// tile of 16 R rows and columns, its eight waves sharing the sum over k (four to
// a product where there are two), all loads of a wave in flight at once: these
// products are bound by the latency of reading what the last launch wrote
// through another XCD's L2.  The first iteration starts from T0 = I and X0 =
// S/2 (ortho.C:236-239) and needs one launch.  The convergence test (the last
// iteration's partials, summed in the same order by every workgroup) overlaps
// the product, and only the stores depend on it.  Iterations after convergence
// return at once; where the last call's count is known one more than that is
// launched, and k_nl_tail runs any others by the same code in the
// same order, so the result does not depend on how many were launched.  T goes to
// Tout in every iteration.  The stage takes 70 us at 84, 128 and 180 states, 95 at
// 256 and 174 at 512 (4 to 6 iterations); the cooperative forms took 103, 91, 186,
// 280 and, over 32 x 32 tiles, 623.
constexpr int kNlThreads = 512;
// iterations launched where no count is known: get_iter_Tmat's limit (cp_lowdin.C:212)
constexpr int kNlLaunch = 10;
enum { kNlC, kNlXT, kNlFirst };

// What the launches of one run tell each other, in the unused error partials of
// iteration 0.  The workgroups of a launch start at different times, so a launch
// reads only what earlier launches wrote: the C launches read res->ns_iter and write
// this, the others read this and write res->ns_iter.
struct NlRun {
  int conv;             // the iteration that met the tolerance, 0: none yet
  double err;           // its change of T
  unsigned next, done;  // k_nl_tail: tiles handed out, tiles finished
};
__device__ __forceinline__ NlRun* nl_run(const NsArgs& a) {
  return reinterpret_cast<NlRun*>(a.errpart);
}

struct NlBuf {
  const double *To, *Xo;
  double *Tw, *Xw;
};
__device__ __forceinline__ NlBuf nl_buf(const NsArgs& a, int it) {  // X_k, T_k in buffer k & 1
  return (it & 1) ? NlBuf{a.T0, a.X0, a.T1, a.X1} : NlBuf{a.T1, a.X1, a.T0, a.X0};
}

// Partial sums over this wave's share s of ks of k (chunks of 16) of rows 16 R ti..
// times columns 16 R tj.. into part[e]; lane group g takes k = 4 g .. 4 g + 3 of a
// chunk.  A past column n counts as zero, addresses are clamped to the matrix.
template <int R, bool FIRST>
__device__ __forceinline__ void nl_product(const double* __restrict__ A,
                                           const double* __restrict__ B, int n, int ti, int tj,
                                           int s, int ks, double* __restrict__ part) {
  constexpr int CB = 4;  // chunks per batch of loads
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int nch = (n + 15) >> 4, q = (nch + ks - 1) / ks, end = min(nch, (s + 1) * q);
  unsigned ar[R], bc[R];
  int row[R];
#pragma unroll
  for (int i = 0; i < R; i++) {
    row[i] = 16 * (R * ti + i) + l16;
    ar[i] = (unsigned)min(row[i], n - 1) * (unsigned)n;
    bc[i] = (unsigned)min(16 * (R * tj + i) + l16, n - 1);
  }
  v4d acc[R][R];
#pragma unroll
  for (int i = 0; i < R * R; i++) acc[i / R][i % R] = vzero();
  for (int c0 = s * q; c0 < end; c0 += CB) {
    double av[R][4 * CB], bv[R][4 * CB];
#pragma unroll
    for (int u = 0; u < 4 * CB; u++) {
      const int k = 16 * (c0 + u / 4) + 4 * g + (u & 3);
      const unsigned kc = min(k, n - 1);
#pragma unroll
      for (int i = 0; i < R; i++) {
        av[i][u] = A[ar[i] + kc];
        bv[i][u] = B[kc * (unsigned)n + bc[i]];
      }
    }
#pragma unroll
    for (int u = 0; u < 4 * CB; u++) {
      const int k = 16 * (c0 + u / 4) + 4 * g + (u & 3);
      const bool in = k < n && c0 + u / 4 < end;
#pragma unroll
      for (int i = 0; i < R; i++) {
        if constexpr (FIRST) {  // C = 3I - S/2, X0 = S/2
          av[i][u] = (row[i] == k ? 3.0 : 0.0) - 0.5 * av[i][u];
          bv[i][u] = 0.5 * bv[i][u];
        }
        av[i][u] = in ? av[i][u] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < R * R; i++)
        acc[i / R][i % R] = mfma16(av[i / R][u], bv[i % R][u], acc[i / R][i % R]);
    }
  }
#pragma unroll
  for (int i = 0; i < R * R; i++)
#pragma unroll
    for (int v = 0; v < 4; v++) part[(4 * i + v) * 64 + lane] = acc[i / R][i % R][v];
}

// Tile (ti, tj) of one launch's work in iteration it.  check: stop where the
// iteration has converged.  Ends with a barrier when check is off.
template <int R, int MODE>
__device__ __forceinline__ void nl_tile(const NsArgs& a, int it, int ti, int tj, int nt,
                                        bool check, double* part) {
  __shared__ double red[8];
  constexpr int NP = MODE == kNlXT ? 2 : 1, KS = 8 / NP, E = 256 * R * R, TP = kNlThreads / NP;
  constexpr int NE = (E + TP - 1) / TP;
  const int n = a.n, nwg = nt * nt, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: so are its matrices
  const NlBuf q = nl_buf(a, it);
  const int m = tid / TP;  // which product's elements this thread finishes
  double es = 0.0;
  // the same in every workgroup (NlRun); one more wait, but idle launches take 1.2 us
  if (MODE == kNlC && check && a.res->ns_iter != 0) return;
  if (MODE == kNlXT && check) {
    const NlRun r = *nl_run(a);
    if (r.conv != 0) {
      if (ti == 0 && tj == 0 && tid == 0) {
        a.res->ns_iter = r.conv;
        a.res->ns_err = r.err;
      }
      return;
    }
  }
  if (MODE == kNlC && check)
    for (int i = tid; i < nwg; i += kNlThreads) es += a.errpart[(size_t)(it - 1) * nwg + i];
  int row[NE], col[NE];
  double old[NE];
#pragma unroll
  for (int i = 0; i < NE; i++) {
    const int e = tid % TP + i * TP, t = e >> 8;
    row[i] = e < E ? 16 * (R * ti + t / R) + ((e & 63) >> 4) + 4 * ((e >> 6) & 3) : n;
    col[i] = 16 * (R * tj + t % R) + (e & 15);
    old[i] = 0.0;
    if (MODE != kNlC)  // the T element before this iteration (first: of S)
      old[i] = (MODE == kNlFirst ? a.S : q.To)[(size_t)min(row[i], n - 1) * n + min(col[i], n - 1)];
  }
  if constexpr (MODE == kNlFirst)
    nl_product<R, true>(a.S, a.S, n, ti, tj, wave, KS, part + wave * E);
  else if constexpr (MODE == kNlC)
    nl_product<R, false>(q.To, q.Xo, n, ti, tj, wave, KS, part + wave * E);
  else
    nl_product<R, false>(wave < KS ? q.Xo : a.C, wave < KS ? a.C : q.To, n, ti, tj, wave % KS, KS,
                         part + wave * E);
  if (MODE == kNlC && check) {
    for (int off = 32; off > 0; off >>= 1) es += __shfl_down(es, off, 64);
    if (lane == 0) red[wave] = es;
  }
  __syncthreads();
  if (MODE == kNlC && check) {
    double s = 0.0;
    for (int w = 0; w < 8; w++) s += red[w];
    const double err = sqrt(s / ((double)n * n));
    if (err <= a.tol) {
      if (ti == 0 && tj == 0 && tid == 0) *nl_run(a) = {it - 1, err, 0, 0};
      return;
    }
  }
  double e2 = 0.0;
#pragma unroll
  for (int i = 0; i < NE; i++) {
    const int e = tid % TP + i * TP;
    if (row[i] >= n || col[i] >= n) continue;
    double p = 0.0;
#pragma unroll
    for (int s = 0; s < KS; s++) p += part[(m * KS + s) * E + e];
    const size_t o = (size_t)row[i] * n + col[i];
    const double one = row[i] == col[i] ? 1.0 : 0.0;
    if constexpr (MODE == kNlC) {
      a.C[o] = 3.0 * one - p;
    } else {
      double nv = 0.5 * p, before = old[i];
      if (m == 0) q.Xw[o] = nv;
      if constexpr (MODE == kNlFirst) {  // T1 = C / 2
        before = one;
        nv = 0.5 * (3.0 * one - 0.5 * old[i]);
      }
      if (MODE == kNlFirst || m == 1) {
        q.Tw[o] = nv;
        a.Tout[o] = nv;
        e2 += (before - nv) * (before - nv);
      }
    }
  }
  if constexpr (MODE != kNlC) {
    for (int off = 32; off > 0; off >>= 1) e2 += __shfl_down(e2, off, 64);
    if (lane == 0) red[wave] = e2;
    __syncthreads();
    if (tid == 0) {
      double s = 0.0;
      for (int w = 0; w < 8; w++) s += red[w];
      a.errpart[(size_t)it * nwg + ti * nt + tj] = s;
    }
    if (MODE == kNlFirst && ti == 0 && tj == 0 && tid == 0) {
      a.res->ns_iter = 0;
      a.res->ns_err = 0.0;
      *nl_run(a) = {0, 0.0, 0, 0};
    }
  }
  if (!check) __syncthreads();
}

template <int R, int MODE>
__global__ __launch_bounds__(kNlThreads) void k_nl(NsArgs a, int it) {
  extern __shared__ __align__(16) double nl_smem[];
  nl_tile<R, MODE>(a, it, blockIdx.y, blockIdx.x, gridDim.x, true, nl_smem);
}

// After `launched` iterations: records convergence of the last one, or runs the
// rest, up to max_iter.  The tiles of all C and X', T' phases are handed out in order;
// a workgroup waits for the phases before its tile's.  Those tiles have all been taken
// by workgroups that run, so every wait ends however few of them are resident: this
// needs no cooperative launch, and where nothing is left to do all return at once.  At
// most as many workgroups as tiles: each takes one tile of the phase that finds the
// end, none of a later one.  An iteration of 512 states takes 75 us here (35 launched
// by itself; 8 ms in the one workgroup that this kernel once was).
constexpr int kNlSpin = 1 << 22;  // polls of a wait: seconds, where a tile takes microseconds
template <int R>
__global__ __launch_bounds__(kNlThreads) void k_nl_tail(NsArgs a, int launched, int nt) {
  extern __shared__ __align__(16) double nl_smem[];
  __shared__ double part[kNlThreads / 64];
  __shared__ int ticket;  // -1: the wait did not end
  const int nwg = nt * nt, tid = threadIdx.x;
  NlRun* run = nl_run(a);
  if (run->conv != 0) return;  // recorded by the last launch
  // the same in every workgroup: true at the end of the iteration, recorded by one
  auto ended = [&](int it, bool record) {
    double es = 0.0;
    for (int i = tid; i < nwg; i += kNlThreads) es += a.errpart[(size_t)it * nwg + i];
    for (int off = 32; off > 0; off >>= 1) es += __shfl_down(es, off, 64);
    if ((tid & 63) == 0) part[tid >> 6] = es;
    __syncthreads();
    es = 0.0;
    for (int w = 0; w < kNlThreads / 64; w++) es += part[w];
    __syncthreads();
    const double err = sqrt(es / ((double)a.n * a.n));
    const bool lost = !(err < __builtin_huge_val());  // S, or a product, not finite
    if (!(err <= a.tol || it >= a.max_iter || lost)) return false;
    if (record) {
      if (tid == 0) {
        a.res->ns_iter = err <= a.tol ? it : -a.max_iter;
        a.res->ns_err = err;
      }
      if (lost && it < a.max_iter)  // where the iterations left would have ended
        for (size_t e = tid; e < (size_t)a.n * a.n; e += kNlThreads)
          a.Tout[e] = __builtin_nan("");
    }
    return true;
  };
  if (ended(launched, blockIdx.x == 0)) return;
  // Thread 0 finishes a tile and takes the next one in one place, and the ways through
  // the loop meet at a barrier before it: with a branch for thread 0 at the end too the
  // compiler made loops of their own for it and for the other lanes of its wave.
  const int rounds = 2 * nwg * (a.max_iter - launched) + 1;  // all tickets, and the end
  for (int round = 0; round < rounds; round++) {
    if (tid == 0) {
      if (round > 0) {  // nl_tile has ended with a barrier: every store of the tile is done
        __threadfence();
        __hip_atomic_fetch_add(&run->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      const unsigned t =
          __hip_atomic_fetch_add(&run->next, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned before = t / nwg * nwg;  // tiles of the earlier phases
      int left = kNlSpin;
      while (__hip_atomic_load(&run->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < before &&
             --left > 0)
        __builtin_amdgcn_s_sleep(8);
      __threadfence();
      ticket = left > 0 ? (int)t : -1;
    }
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(ticket), phase = t / nwg, w = t - phase * nwg, it = launched + 1 + phase / 2;
    if (t < 0) {
      if (tid == 0) {
        a.res->ns_iter = -a.max_iter;
        a.res->ns_err = __builtin_nan("");
      }
      return;
    }
    if (phase & 1) {
      nl_tile<R, kNlXT>(a, it, w / nt, w % nt, nt, false, nl_smem);
    } else {
      if (phase > 0 && ended(it - 1, w == 0)) return;
      nl_tile<R, kNlC>(a, it, w / nt, w % nt, nt, false, nl_smem);
    }
  }
}

template <int R>
static hipError_t ns_steps_r(const NsArgs& a, hipStream_t st) {
  const int nt = (a.n + 16 * R - 1) / (16 * R);
  const size_t sm = (size_t)8 * 256 * R * R * sizeof(double);
  for (const void* f : {(const void*)k_nl<R, kNlC>, (const void*)k_nl<R, kNlXT>,
                        (const void*)k_nl<R, kNlFirst>, (const void*)k_nl_tail<R>})
    if (const hipError_t e = grant_lds(f, sm); e != hipSuccess) return e;
  const int count = std::min(a.max_iter, a.hint > 0 ? a.hint + 1 : kNlLaunch);
  const dim3 grid(nt, nt), thr(kNlThreads);
  hipLaunchKernelGGL((k_nl<R, kNlFirst>), grid, thr, sm, st, a, 1);
  for (int it = 2; it <= count; it++) {
    hipLaunchKernelGGL((k_nl<R, kNlC>), grid, thr, sm, st, a, it);
    hipLaunchKernelGGL((k_nl<R, kNlXT>), grid, thr, sm, st, a, it);
  }
  hipLaunchKernelGGL(k_nl_tail<R>, dim3(std::min(nt * nt, cu_count())), thr, sm, st, a, count, nt);
  return hipGetLastError();
}
static hipError_t ns_run_steps(const NsArgs& a, hipStream_t st) {
  return ns_steps_r_of(a.n) == 1 ? ns_steps_r<1>(a, st) : ns_steps_r<2>(a, st);
}

static const void* nr_kernel(int n) {
  switch (nr_kb(n)) {
    case 8: return (const void*)k_ns_rows<8>;
    default: return (const void*)k_ns_rows<16>;
  }
}

static bool ns_smem_granted(int device) {
  int lds_max = 0;
  if (hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, device) !=
          hipSuccess ||
      (size_t)lds_max < kNsSmem)
    return false;
  return grant_lds((const void*)k_ns_coop, kNsSmem) == hipSuccess;
}

// Can all n x n tiles be resident at once for the cooperative launch?
// The block-row variant: all ceil(n/16) x split workgroups resident, both
// LDS row blocks within the device's limit, at least one column tile per
// column group.
bool ns_rows_possible(int n, int split, int device) {
  int per_cu = 0, ncu = 0, coop = 0, lds_max = 0;
  const int nb = (n + 15) / 16;
  if (n < 1 || split < 1 || split > (n + 15) / 16 || nb * split > kNrMaxWg ||
      hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess ||
      !coop)
    return false;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
      hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, device) !=
          hipSuccess)
    return false;
  const size_t smem = ns_rows_smem(n);
  const void* fn = nr_kernel(n);
  if (smem > (size_t)lds_max || grant_lds(fn, smem) != hipSuccess) return false;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, kNrWaves * 64, smem) !=
      hipSuccess)
    return false;
  return (long)per_cu * ncu >= (long)nb * split;
}

bool ns_coop_possible(int n, int device) {
  const int nt = (n + NT - 1) / NT;
  int per_cu = 0, ncu = 0, coop = 0;
  if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess ||
      !coop)
    return false;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
    return false;
  if (!ns_smem_granted(device)) return false;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k_ns_coop, 256,
                                                   kNsSmem) != hipSuccess)
    return false;
  return (long)per_cu * ncu >= (long)nt * nt;
}

hipError_t ns_run(const NsArgs& a, hipStream_t st) {
  if (!a.coop) return ns_run_launches(a, st);
  if (a.coop == kNsStepsKind) return ns_run_steps(a, st);
  if (a.coop == kNsOneKind) {
    if (a.n > kNsOneMax) return hipErrorInvalidValue;  // X, T and C would not fit in LDS
    const hipError_t e = grant_lds((const void*)k_ns_one, kNsOneSmem);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_ns_one, dim3(1), dim3(ns_one_threads(a.n)), kNsOneSmem, st, a);
    return hipGetLastError();
  }
  NsArgs args = a;
  void* params[] = {&args};
  hipError_t e;
  if (a.coop >= 2) {
    e = hipLaunchCooperativeKernel(nr_kernel(a.n), dim3((a.n + 15) / 16, ns_rows_split(a.coop)),
                                   dim3(kNrWaves * 64), params, ns_rows_smem(a.n), st);
  } else {
    const int nt = (a.n + NT - 1) / NT;
    e = hipLaunchCooperativeKernel((const void*)k_ns_coop, dim3(nt * nt), dim3(256), params,
                                   kNsSmem, st);
  }
  if (e == hipSuccess) return e;
  // The runtime refuses a cooperative launch when the device's grid-barrier
  // resource is held by another process (hipErrorIllegalState); a refused
  // launch enqueues nothing, so the same iteration runs as two launches per
  // iteration instead (its error partials fit the same buffer).
  (void)hipGetLastError();
  return ns_run_launches(a, st);
}

}  // namespace oa

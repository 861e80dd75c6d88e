// oa_gemm_bf16.hip -- split-BF16 contractions of the mixed-precision step on
// CDNA4 matrix cores (v_mfma_f32_32x32x16_bf16).
//
// Every FP64 operand x is rounded to FP32, f = fl32(x) (2^-24 relative),
// and f is split exactly into three BF16 terms, f = h + m + l (h = bf16(f),
// m = bf16(f - h), l = f - h - m, each step exact in FP32 with round to
// nearest, |m| <= 2^-8 |f|, |l| <= 2^-16 |f|).  A product keeps the six term
// products with i + j <= 2 (h*h, h*m, m*h, h*l, m*m, l*h): each BF16 x BF16
// product is exact in FP32, the dropped ones are below 2^-24 relative, and
// the MFMA sums into FP32 accumulators.  So the result carries the FP32
// rounding of its operands and FP32 accumulation error over the products
// of one K slice (gram) or of the inner dimension (rotate), no more.
// K-slice partial sums are written in FP32 and summed in FP64.  The split
// costs three packed conversions, two widenings and two FP32 subtractions
// per pair of values (splitting the FP64 residuals instead took twice the
// vector instructions, which bound the gram).
//
//   gram_bf16   : C = sum_k w(k) A[i][k] B[j][k] (Lambda = Re Psi^H F, and S on
//                 request): one workgroup per output block (128 or 256 square)
//                 and K slice, operands split once per workgroup into LDS;
//   rotate_bf16 : Y = beta Y + s(k) M^T X (+ X) for n, ni <= 128 (F -= w Psi
//                 Lambda, and Psi T on request in the form Psi + Psi (T - I)):
//                 persistent workgroups over 64-column blocks of K; the
//                 split M^T (A operand) stays in registers for the whole
//                 launch, each block of X is split once into LDS in the
//                 B-operand layout and read back conflict-free.
//
// MFMA 32x32x16 lane layout (gfx950): A operand lane l holds row l%32 and
// k = 8 (l/32) + e, B operand lane l holds column l%32 and the same k; the
// accumulator element v of lane l is D[8 (v/4) + 4 (l/32) + v%4][l%32].
// Within one MFMA the assignment of k to (lane group, element) is free as
// long as A and B agree.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "oa_common.h"
#include "oa_gemm_common.h"
#include "oa_kernels.h"

namespace oa {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

namespace {

__device__ __forceinline__ f16v mfma32(bf8 a, bf8 b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f16v fzero16() {
  f16v z;
#pragma unroll
  for (int v = 0; v < 16; v++) z[v] = 0.f;
  return z;
}

// Three BF16 terms of eight doubles (of their FP32 roundings).
struct Split {
  bf8 h, m, l;
};

__device__ __forceinline__ Split split3(const double (&x)[8]) {
  Split s;
  float r[8];
#pragma unroll
  for (int e = 0; e < 8; e++) r[e] = (float)x[e];
#pragma unroll
  for (int e = 0; e < 8; e++) s.h[e] = (__bf16)r[e];
#pragma unroll
  for (int e = 0; e < 8; e++) r[e] -= (float)s.h[e];
#pragma unroll
  for (int e = 0; e < 8; e++) s.m[e] = (__bf16)r[e];
#pragma unroll
  for (int e = 0; e < 8; e++) r[e] -= (float)s.m[e];
#pragma unroll
  for (int e = 0; e < 8; e++) s.l[e] = (__bf16)r[e];
  return s;
}

// acc += A B over the six kept term products, small terms first
__device__ __forceinline__ f16v mma6(const Split& a, const Split& b, f16v acc) {
  acc = mfma32(a.l, b.h, acc);
  acc = mfma32(a.m, b.m, acc);
  acc = mfma32(a.h, b.l, acc);
  acc = mfma32(a.m, b.h, acc);
  acc = mfma32(a.h, b.m, acc);
  return mfma32(a.h, b.h, acc);
}

}  // namespace

// ------------------------------------------------------------------ gram
// Blocks of 64 RT x 64 RT outputs (every block whole: a symmetric product's
// lower half is mirrored by the reduction), operands split once per workgroup.
// A workgroup of four waves (wave: RT x RT tiles of 32 x 32) owns a block and a
// K slice.  Per 16 k values every thread loads pairs of its rows (a row's 128
// bytes by eight lanes), splits them and puts the three terms into LDS in the
// operand layout; the MFMAs of the current chunk, the split of the next one and
// the loads of the one after overlap (double-buffered LDS, one barrier per
// chunk).  A split in every wave that uses an operand, from registers, took
// each value through the conversions up to eight times and bound the product:
// us for 128 x 65,922 reals 42 -> 27, 180 x 73,600 150 -> 65, 256 x 131,824
// 284 -> 133, 512 x 260,992 2533 -> 878 (conversions and MFMAs alternate in one
// wave per SIMD there; the bytes take 420 at the rate of a copy).
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));

template <int RT>
constexpr size_t gram_bf16_lds() {
  return (size_t)2 * 2 * 3 * (2 * RT) * 64 * sizeof(bf8);
}

// Workgroups go to the 8 XCDs round-robin: all output blocks of one K slice read
// the same operand columns, so they are put on one XCD (one L2) where the slice
// count allows.
__device__ __forceinline__ void slice_block(int& b, int& sp) {
  b = blockIdx.x;
  sp = blockIdx.y;
  if (gridDim.y % 8 == 0) {
    const int id = blockIdx.x + gridDim.x * blockIdx.y, k = id >> 3;
    b = k % gridDim.x;
    sp = (k / gridDim.x) * 8 + (id & 7);
  }
}

template <int RT>
__global__ __launch_bounds__(256, RT == 4 ? 1 : 2) void k_gram_bf16(GramArgs a,
                                                                     float* __restrict__ part,
                                                                     int nbe_b, int nlo) {
  constexpr int TT = 2 * RT;                   // 32-row tiles per operand
  constexpr int TERM = TT * 64, OPER = 3 * TERM, BUF = 2 * OPER;  // in bf8
  extern __shared__ __align__(16) unsigned char gb_smem[];
  bf8* L = reinterpret_cast<bf8*>(gb_smem);    // [buffer][operand][term][tile][lane]
  int blk, sp;
  slice_block(blk, sp);
  const int bi = blk / nbe_b, bj = blk - bi * nbe_b;
  const GSlice s = gram_slice(a, sp, nlo);
  const double* __restrict__ B = a.sym ? a.A : a.B;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const int l32 = lane & 31, g = lane >> 5;
  // staging: thread (r0, kp) takes the pair of k values 2 kp, 2 kp + 1 of row r0
  // of every tile; rows past the matrices repeat the last (outputs not stored)
  const int kp = tid & 7, r0 = tid >> 3;
  unsigned* const stage = reinterpret_cast<unsigned*>(L) + (r0 + 32 * (kp >> 2)) * 4 + (kp & 3);
  double2 raw[2 * TT];
  auto load = [&](int u, int c) __attribute__((always_inline)) {
    const bool isb = u >= TT;
    const int n = isb ? a.nb : a.n;
    const int tb = min((isb ? bj : bi) * 64 * RT + 32 * (isb ? u - TT : u), n - 1);
    const double* p = (isb ? B : a.A) + (size_t)tb * a.lda + s.base + 16 * c;
    raw[u] = *reinterpret_cast<const double2*>(p + (size_t)min(r0, n - 1 - tb) * a.lda + 2 * kp);
  };
  // split tile u of chunk c into buffer buf; edge: elements outside the region
  // [rs, re) are zeroed (only a slice's first and last chunk reach past it;
  // padding past K may hold anything)
  auto split = [&](auto edge, int u, int c, int buf) __attribute__((always_inline)) {
    double2 x = raw[u];
    if constexpr (decltype(edge)::value) {
      const int kk = s.base + 16 * c + 2 * kp;
      x.x = kk >= s.rs && kk < s.re ? x.x : 0.0;
      x.y = kk + 1 >= s.rs && kk + 1 < s.re ? x.y : 0.0;
    }
    f2 r = {(float)x.x, (float)x.y};
    // the FP32 values as such: rounding the doubles to BF16 directly, as the
    // compiler otherwise does for the first term, takes ten instructions more
    asm("" : "+v"(r.x), "+v"(r.y));
    unsigned* out = stage + (size_t)(buf * BUF + (u >= TT ? OPER : 0) + (u % TT) * 64) * 4;
#pragma unroll
    for (int t = 0; t < 3; t++) {
      const bf2 h = {(__bf16)r.x, (__bf16)r.y};
      out[(size_t)t * TERM * 4] = __builtin_bit_cast(unsigned, h);
      r.x -= (float)h.x;
      r.y -= (float)h.y;
    }
  };
  f16v acc[RT][RT];
#pragma unroll
  for (int x = 0; x < RT; x++)
#pragma unroll
    for (int y = 0; y < RT; y++) acc[x][y] = fzero16();
  // the products of chunk c0 + i, and the split of the next one
  auto chunk = [&](auto edge, int i) __attribute__((always_inline)) {
    const bf8* Ab = L + (i & 1) * BUF + wr * RT * 64 + lane;
    const bf8* Bb = L + (i & 1) * BUF + OPER + wc * RT * 64 + lane;
    const int cn = min(s.c0 + i + 1, s.c1 - 1), cl = min(s.c0 + i + 2, s.c1 - 1);
    Split sb[RT];
#pragma unroll
    for (int y = 0; y < RT; y++)
      sb[y] = {Bb[y * 64], Bb[TERM + y * 64], Bb[2 * TERM + y * 64]};
#pragma unroll
    for (int x = 0; x < RT; x++) {
      const Split sa = {Ab[x * 64], Ab[TERM + x * 64], Ab[2 * TERM + x * 64]};
      // the six term products, small terms first, over independent tiles
#pragma unroll
      for (int y = 0; y < RT; y++) acc[x][y] = mfma32(sa.l, sb[y].h, acc[x][y]);
#pragma unroll
      for (int y = 0; y < RT; y++) acc[x][y] = mfma32(sa.m, sb[y].m, acc[x][y]);
#pragma unroll
      for (int y = 0; y < RT; y++) acc[x][y] = mfma32(sa.h, sb[y].l, acc[x][y]);
#pragma unroll
      for (int y = 0; y < RT; y++) acc[x][y] = mfma32(sa.m, sb[y].h, acc[x][y]);
#pragma unroll
      for (int y = 0; y < RT; y++) acc[x][y] = mfma32(sa.h, sb[y].m, acc[x][y]);
#pragma unroll
      for (int y = 0; y < RT; y++) acc[x][y] = mfma32(sa.h, sb[y].h, acc[x][y]);
      // four tiles of the next chunk between the products; a tile's loads for
      // the chunk after it follow at once and are in flight for a whole chunk
#pragma unroll
      for (int u = 4 * x; u < 4 * x + 4; u++) {
        split(edge, u, cn, (i + 1) & 1);
        load(u, cl);
      }
    }
    __syncthreads();
  };
  const int nc = s.c1 - s.c0;
  if (nc > 0) {
#pragma unroll
    for (int u = 0; u < 2 * TT; u++) load(u, s.c0);
#pragma unroll
    for (int u = 0; u < 2 * TT; u++) {
      split(std::true_type{}, u, s.c0, 0);
      load(u, min(s.c0 + 1, s.c1 - 1));
    }
    __syncthreads();
    int i = 0;
    for (; i < nc - 2; i++) chunk(std::false_type{}, i);
    for (; i < nc; i++) chunk(std::true_type{}, i);
  }
  float* out = part + (size_t)sp * a.n * a.nb;
  const float w = (float)s.w;  // 1 or 2: exact
  const int rbase = bi * 64 * RT + wr * 32 * RT, cbase = bj * 64 * RT + wc * 32 * RT;
#pragma unroll
  for (int x = 0; x < RT; x++)
#pragma unroll
    for (int y = 0; y < RT; y++)
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int r = rbase + 32 * x + 8 * (v >> 2) + 4 * g + (v & 3);
        const int col = cbase + 32 * y + l32;
        if (r < a.n && col < a.nb) out[(size_t)r * a.nb + col] = w * acc[x][y][v];
      }
}

// Block edge in units of 64 rows: 256 rows where that pads a matrix of more
// than one block no more than 128 rows do (512 states: 878 us against 1088;
// 256: 155 against 133, 300: 233 against 142), else 128.
static int gram_bf16_rt(int n, int nb) {
  const int m = std::max(n, nb);
  return m > 256 && (m + 255) / 256 * 2 == (m + 127) / 128 ? 4 : 2;
}

// one workgroup per CU for a single block or blocks of 256 rows, else two
int gram_bf16_slices(int n, int K, int target) {
  const int rt = gram_bf16_rt(n, n), nb = (n + 64 * rt - 1) / (64 * rt);
  const int ns = std::max(2, target * (nb > 1 && rt == 2 ? 2 : 1) / (nb * nb));
  return std::min(ns, std::max(2, K / 64));  // at least four chunks per slice
}

hipError_t gram_bf16(const GramArgs& a, float* part, hipStream_t st) {
  if (a.nslice < 1 || (a.k_lo > 0 && a.k_lo < a.K && a.nslice < 2) || (a.lda & 15) ||
      a.n < 1 || a.nb < 1 || (a.sym && a.nb != a.n) || !part)
    return hipErrorInvalidValue;
  const int rt = gram_bf16_rt(a.n, a.nb), edge = 64 * rt;
  const int nbe = (a.n + edge - 1) / edge, nbe_b = (a.nb + edge - 1) / edge;
  void (*const fn)(GramArgs, float*, int, int) = rt == 4 ? k_gram_bf16<4> : k_gram_bf16<2>;
  const size_t lds = rt == 4 ? gram_bf16_lds<4>() : gram_bf16_lds<2>();
  if (const hipError_t e = grant_lds((const void*)fn, lds); e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(nbe * nbe_b, a.nslice), dim3(256), lds, st, a, part, nbe_b,
                     gram_nlo(a));
  return hipGetLastError();
}

// ------------------------------------------------------------------ rotate
constexpr int kRbK = 64;  // columns of K per block
constexpr int kRbSteps = 8;  // inner-dimension steps of 16 (ni <= 128)
// LDS: [term][column tile][step][lane] of bf8 (16 bytes)
constexpr size_t kRbSmem = (size_t)3 * 2 * kRbSteps * 64 * sizeof(bf8);

__global__ __launch_bounds__(256, 1) void k_rotate_bf16(RotArgs a) {
  extern __shared__ __align__(16) unsigned char rb_smem[];
  bf8* Xs = reinterpret_cast<bf8*>(rb_smem);
  __shared__ double red[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, g = lane >> 5;
  const int ni = a.ni, n = a.n;
  const int nsteps = (ni + 15) >> 4;
  // A operand: M^T split, rows j = 32 wave + l32, inner i = 16 s + 8 g + e
  // (M[i][j] at i*n + j; with m_minus_i, M - I)
  const int jrow = 32 * wave + l32;
  Split ms[kRbSteps];
#pragma unroll
  for (int s = 0; s < kRbSteps; s++) {
    double x[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int i = 16 * s + 8 * g + e;
      const bool ok = i < ni && jrow < n;
      const double v = a.M[(size_t)min(i, ni - 1) * n + min(jrow, n - 1)];
      x[e] = ok ? v - ((a.m_minus_i && i == jrow) ? 1.0 : 0.0) : 0.0;
    }
    ms[s] = split3(x);
  }
  const int nkb = (a.K + kRbK - 1) / kRbK;
  // staging: thread takes column kk = tid % 64 of a block and the 8-row
  // groups i8 = tid / 64 + 4 u of X; rows past ni are clamped (their M^T
  // entries are zero).  The next block's X is fetched into registers while
  // this block's products run.
  const int kk = tid & 63, w8 = tid >> 6;
  double xr[4][8];
  auto fetch = [&](int blk) __attribute__((always_inline)) {
    const int kb = min(blk, nkb - 1) * kRbK;
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int e = 0; e < 8; e++)
        xr[u][e] = a.X[(size_t)min(8 * (w8 + 4 * u) + e, ni - 1) * a.ldx + kb + kk];
  };
  fetch(blockIdx.x);
  double fsum = 0.0;
  for (int blk = blockIdx.x; blk < nkb; blk += gridDim.x) {
    const int kb = blk * kRbK;
    __syncthreads();  // the previous block's operands are consumed
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int i8 = w8 + 4 * u;
      const Split sx = split3(xr[u]);
      const int idx = ((kk >> 5) * kRbSteps + (i8 >> 1)) * 64 + (kk & 31) + 32 * (i8 & 1);
      Xs[idx] = sx.h;
      Xs[2 * kRbSteps * 64 + idx] = sx.m;
      Xs[4 * kRbSteps * 64 + idx] = sx.l;
    }
    // what the epilogue adds (beta Y + Xadd), loaded unconditionally at
    // clamped addresses; only the stores are masked
    double old[2][16];
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      const int kc = min(kb + 32 * kt + l32, a.K - 1);
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int jc = min(32 * wave + 8 * (v >> 2) + 4 * g + (v & 3), n - 1);
        const size_t o = (size_t)jc * a.ldx + kc;
        old[kt][v] = (a.beta != 0.0 ? a.beta * a.Y[o] : 0.0) + (a.Xadd ? a.Xadd[o] : 0.0);
      }
    }
    fetch(blk + gridDim.x);
    __syncthreads();
    f16v acc[2] = {fzero16(), fzero16()};
#pragma unroll
    for (int s = 0; s < kRbSteps; s++) {
      if (s < nsteps) {
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
          const int idx = (kt * kRbSteps + s) * 64 + lane;
          Split xb;
          xb.h = Xs[idx];
          xb.m = Xs[2 * kRbSteps * 64 + idx];
          xb.l = Xs[4 * kRbSteps * 64 + idx];
          acc[kt] = mma6(ms[s], xb, acc[kt]);
        }
      }
    }
    // epilogue: rows j, columns k along the lanes (256-byte stores)
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      const int k = kb + 32 * kt + l32;
      const double sk = k < a.k_lo ? a.s_lo : a.s_hi;
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int j = 32 * wave + 8 * (v >> 2) + 4 * g + (v & 3);
        const double y = sk * (double)acc[kt][v] + old[kt][v];
        if (j < n && k < a.K) {
          a.Y[(size_t)j * a.ldx + k] = y;
          fsum += y * y;
        }
      }
    }
  }
  if (a.fpart) {
    for (int o = 32; o > 0; o >>= 1) fsum += __shfl_down(fsum, o, 64);
    if (lane == 0) red[wave] = fsum;
    __syncthreads();
    if (tid == 0) a.fpart[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
  }
}

int rotate_bf16_nwg(int K) {
  return std::max(1, std::min(cu_count(), (K + kRbK - 1) / kRbK));
}

hipError_t rotate_bf16(const RotArgs& args, hipStream_t st) {
  RotArgs a = args;
  if (a.ni <= 0) a.ni = a.n;
  if (a.n > 128 || a.ni > 128 || a.sd_psi || (a.ldx % kRbK) || a.K > a.ldx || a.Xadd == a.Y)
    return hipErrorInvalidValue;
  if (const hipError_t e = grant_lds((const void*)k_rotate_bf16, kRbSmem); e != hipSuccess)
    return e;
  hipLaunchKernelGGL(k_rotate_bf16, dim3(rotate_bf16_nwg(a.K)), dim3(256), kRbSmem, st, a);
  return hipGetLastError();
}

}  // namespace oa

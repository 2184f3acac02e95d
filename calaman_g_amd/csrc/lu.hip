// lu.hip -- LU factorization with partial pivoting and the triangular solves of
// the Pade route (?getrf / ?getrs, which the reference takes from the vendor
// solver: src/expm/pade.cppm:186-188).
//
// Recursive LU (the column split of LAPACK's ?getrf2): factor the left half of
// a block column, interchange and solve its right half against the unit-lower
// triangle, subtract the product from the trailing rows, factor the right half.
// The large updates are the library's MFMA products; the recursion stops at panels of up
// to 32 columns and 128 KiB, factored by one 512-lane workgroup with its rows in
// registers: the pivot search is a shuffle reduction over the waves, and the pivot row
// reaches every lane through LDS and scalar registers, two barriers a column. A panel
// waits on that chain of steps, not on arithmetic; 1000 x 16 in FP64 takes 30 us (76 us
// with the block in LDS, its columns walked by strided lanes, five barriers a column).
// Panels too tall for the registers run the same steps on the matrix in memory.
// A panel's interchanges are applied at once to every other column of the
// matrix, which gives the same matrix as LAPACK's deferred application: the
// columns to the right are not touched in between, those to the left are final.
//
// Pivoting follows ?getf2: the pivot is the first entry of largest |.| (|re| +
// |im| for complex, as i?amax), a zero pivot leaves the column unscaled and
// sets info to its (1-based) column once, and the column is scaled by the
// reciprocal of the pivot unless the pivot is below the smallest normal number,
// when it is divided. ipiv is 1-based, as LAPACK's.
#include "clm_internal.hpp"

#include <algorithm>
#include <climits>
#include <cmath>

namespace clm {
namespace {

constexpr int kLeafThreads = 1024;
constexpr int kPanelCols = 32;
constexpr int kPanelThreads = 512;  // half the waves of 1024 lanes, each sending a pivot row's
                                    // columns to twice the rows
constexpr int kTrsmNb = 64;  // triangle order solved in LDS

// i?amax's measure: |x| for real, |re| + |im| for complex
__device__ inline double cabs1(double x) { return fabs(x); }
__device__ inline double cabs1(float x) { return fabsf(x); }
__device__ inline double cabs1(zd x) { return fabs(x.re) + fabs(x.im); }
__device__ inline double cabs1(zc x) { return double(fabsf(x.re) + fabsf(x.im)); }

__device__ inline double sub(double a, double b) { return a - b; }
__device__ inline float sub(float a, float b) { return a - b; }
__device__ inline zd sub(zd a, zd b) { return zd{a.re - b.re, a.im - b.im}; }
__device__ inline zc sub(zc a, zc b) { return zc{a.re - b.re, a.im - b.im}; }

// a - x y, two roundings a component at most
__device__ inline double msub(double a, double x, double y) { return __builtin_fma(-x, y, a); }
__device__ inline float msub(float a, float x, float y) { return __builtin_fmaf(-x, y, a); }
__device__ inline zd msub(zd a, zd x, zd y) {
  return zd{__builtin_fma(x.im, y.im, __builtin_fma(-x.re, y.re, a.re)),
            __builtin_fma(-x.im, y.re, __builtin_fma(-x.re, y.im, a.im))};
}
__device__ inline zc msub(zc a, zc x, zc y) {
  return zc{__builtin_fmaf(x.im, y.im, __builtin_fmaf(-x.re, y.re, a.re)),
            __builtin_fmaf(-x.im, y.re, __builtin_fmaf(-x.re, y.im, a.im))};
}

__device__ inline double cdiv(double a, double b) { return a / b; }
__device__ inline float cdiv(float a, float b) { return a / b; }
// complex division, Smith's method (as the reference LAPACK's ?ladiv family guards
// the ratio of the larger component)
__device__ inline zd cdiv(zd a, zd b) {
  if (fabs(b.re) >= fabs(b.im)) {
    const double r = b.im / b.re, d = b.re + b.im * r;
    return zd{(a.re + a.im * r) / d, (a.im - a.re * r) / d};
  }
  const double r = b.re / b.im, d = b.im + b.re * r;
  return zd{(a.re * r + a.im) / d, (a.im * r - a.re) / d};
}
__device__ inline zc cdiv(zc a, zc b) {
  if (fabsf(b.re) >= fabsf(b.im)) {
    const float r = b.im / b.re, d = b.re + b.im * r;
    return zc{(a.re + a.im * r) / d, (a.im - a.re * r) / d};
  }
  const float r = b.re / b.im, d = b.im + b.re * r;
  return zc{(a.re * r + a.im) / d, (a.im * r - a.re) / d};
}
template <typename T>
__device__ inline double min_normal() {
  return std::is_same_v<real_t<T>, float> ? 1.17549435e-38 : 2.2250738585072014e-308;
}

// ---- the panel in memory: a block column of m rows and w columns ----------------------------
// P: the block, in the matrix itself. row0 is
// the global row (and column) of the block's first row; ipiv and info get global
// 1-based indices.
template <typename T>
__device__ void leaf_factor(T *P, long ldp, int m, int w, int row0, int *ipiv, int *info,
                            double *red_v, int *red_i, T *pivot) {
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  for (int j = 0; j < w; ++j) {
    // pivot: the first row of largest measure among rows j .. m-1 (a NaN measure
    // ranks below every number, so it is taken only from an all-NaN column)
    double best = -1.0;
    int bi = INT_MAX;
    for (int i = j + tid; i < m; i += kLeafThreads) {
      double v = cabs1(P[i + j * ldp]);
      if (!(v == v)) v = -0.5;
      if (v > best) {  // rows ascend within a lane: the first maximum stays
        best = v;
        bi = i;
      }
    }
    for (int off = 32; off > 0; off >>= 1) {
      const double ov = __shfl_xor(best, off);
      const int oi = __shfl_xor(bi, off);
      if (ov > best || (ov == best && oi < bi)) {
        best = ov;
        bi = oi;
      }
    }
    if (lane == 0) {
      red_v[wave] = best;
      red_i[wave] = bi;
    }
    __syncthreads();
    if (tid == 0) {
      double b = red_v[0];
      int idx = red_i[0];
      for (int q = 1; q < kLeafThreads / 64; ++q) {
        const double v = red_v[q];
        const int i = red_i[q];
        if (v > b || (v == b && i < idx)) {
          b = v;
          idx = i;
        }
      }
      if (idx == INT_MAX) idx = j;  // row j always competes: not reached
      red_i[kLeafThreads / 64] = idx;
      *pivot = P[idx + j * ldp];  // published before the barrier: lane j exchanges it below
      ipiv[row0 + j] = row0 + idx + 1;
    }
    __syncthreads();
    const int p = red_i[kLeafThreads / 64];
    const T a = *pivot;
    const bool nonzero = !ops<T>::is_zero(a);
    if (nonzero) {
      if (p != j && tid < w) {  // interchange rows j and p of the block
        const T t = P[j + tid * ldp];
        P[j + tid * ldp] = P[p + tid * ldp];
        P[p + tid * ldp] = t;
      }
    } else if (tid == 0) {
      atomicMin(info, row0 + j + 1);
    }
    __syncthreads();
    if (nonzero) {
      // scale the column below the pivot (after the interchange the pivot is at row j)
      if (cabs1(a) >= min_normal<T>()) {
        const T r = cdiv(ops<T>::from_real(1.0), a);
        for (int i = j + 1 + tid; i < m; i += kLeafThreads) P[i + j * ldp] = ops<T>::mul(P[i + j * ldp], r);
      } else {
        for (int i = j + 1 + tid; i < m; i += kLeafThreads) P[i + j * ldp] = cdiv(P[i + j * ldp], a);
      }
    }
    __syncthreads();
    // rank-1 update of the block's remaining columns: a lane a row, across the columns
    if (j + 1 < w) {
      for (int i = j + 1 + tid; i < m; i += kLeafThreads) {
        const T lij = P[i + j * ldp];
        for (int c = j + 1; c < w; ++c)
          P[i + c * ldp] = sub(P[i + c * ldp], ops<T>::mul(lij, P[j + c * ldp]));
      }
    }
    __syncthreads();
  }
}

// lane l's value in every lane (l uniform)
__device__ inline float from_lane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ inline double from_lane(double v, int l) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane(static_cast<int>(b & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), l);
  return __longlong_as_double((static_cast<long long>(hi) << 32) | lo);
}
__device__ inline zc from_lane(zc v, int l) { return zc{from_lane(v.re, l), from_lane(v.im, l)}; }
__device__ inline zd from_lane(zd v, int l) { return zd{from_lane(v.re, l), from_lane(v.im, l)}; }

// The pivot measure as an integer that orders like it: the bits of a non-negative double,
// -1 for a NaN (below every number), -2 for no row
__device__ inline long long measure_key(double v) {
  return v == v ? __double_as_longlong(v) : -1ll;
}
// the largest key over a group of `width` lanes and the smallest index that has it
template <int width>
__device__ inline void group_argmax(long long &key, int &idx) {
  long long m = key;
#pragma unroll
  for (int off = width / 2; off > 0; off >>= 1) {
    const long long o = __shfl_xor(m, off);
    m = o > m ? o : m;
  }
  unsigned long long has = __ballot(key == m);
  if constexpr (width < 64) has &= (1ull << width) - 1;  // the keys repeat past the group
  if (__ballot(m != -2) == 0) has = 0;  // no row in the group
  int first = INT_MAX;
  while (has) {
    first = min(first, __builtin_amdgcn_readlane(idx, __ffsll(has) - 1));
    has &= has - 1;
  }
  key = m;
  idx = first;
}

// the panel A[row0 : n, row0 : row0 + w], w <= W, in registers: lane t holds rows t, t +
// 512, ... (R of them). leaf_factor's steps and arithmetic; the interchanges of the
// panel's own earlier columns are left to laswp_kernel. The current column is always
// register 0: the update writes column c's result to register c - 1, so the steps are one
// loop (unrolled over the columns they are 64 KB of code run once, and the panel waited
// for its instructions: 88 us for 1000 x 32). A finished column of L and row of U go
// straight to memory.
template <typename T, int W, int R>
__global__ void __launch_bounds__(kPanelThreads)
    panel_kernel(int n, T *A, long lda, int row0, int w, int *ipiv, int *info) {
  constexpr int kWaves = kPanelThreads / 64;
  // two sets by the column's parity: a set is rewritten two barriers after its last read
  __shared__ long long red_k[2][kWaves];
  __shared__ int red_i[2][kWaves];
  __shared__ T rows[2][2][W];  // the pivot row, and row j that it changes places with
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = n - row0;
  T *blk = A + row0 + static_cast<long>(row0) * lda;
  T a[R][W];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < W; ++c) {
      const int i = tid + kPanelThreads * r;
      a[r][c] = (i < m && c < w) ? blk[i + c * lda] : ops<T>::zero();
    }
#pragma unroll 1
  for (int j = 0; j < w; ++j) {
    const int set = j & 1;
    long long key = -2;
    int bi = INT_MAX;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = tid + kPanelThreads * r;
      const long long k = measure_key(cabs1(a[r][0]));
      if (i >= j && i < m && k > key) {  // rows ascend: the first maximum stays
        key = k;
        bi = i;
      }
    }
    group_argmax<64>(key, bi);
    if (lane == 0) {
      red_k[set][wave] = key;
      red_i[set][wave] = bi;
    }
    __syncthreads();
    key = red_k[set][lane % kWaves];
    bi = red_i[set][lane % kWaves];
    group_argmax<kWaves>(key, bi);
    const bool nonzero = key != 0;  // a zero pivot: no interchange, no scaling
    const int p = nonzero ? bi : j;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = tid + kPanelThreads * r;
      if (i == p) {
#pragma unroll
        for (int c = 0; c < W; ++c) rows[set][0][c] = a[r][c];
      }
      if (i == j) {
#pragma unroll
        for (int c = 0; c < W; ++c) rows[set][1][c] = a[r][c];
      }
    }
    if (tid == 0) {
      ipiv[row0 + j] = row0 + bi + 1;
      if (!nonzero) atomicMin(info, row0 + j + 1);
    }
    __syncthreads();
    // lane c of every wave takes column c of the pivot row; a column's value then goes to
    // all lanes through a scalar register
    const T prow = rows[set][0][lane % W];
    if (tid < w - j) blk[j + static_cast<long>(j + tid) * lda] = prow;
    const T pv = from_lane(prow, 0);
    const bool safe = cabs1(pv) >= min_normal<T>();
    const T rp = safe ? cdiv(ops<T>::from_real(1.0), pv) : ops<T>::zero();
    if (p != j) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (tid + kPanelThreads * r == p) {  // one lane: its own reads, no other lane's registers
#pragma unroll
          for (int c = 0; c < W; ++c) a[r][c] = rows[set][1][c];
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = tid + kPanelThreads * r;
      T l = a[r][0];
      if (nonzero) l = safe ? ops<T>::mul(l, rp) : cdiv(l, pv);
      if (i > j && i < m) blk[i + static_cast<long>(j) * lda] = l;
#pragma unroll
      for (int c = 1; c < W; ++c) a[r][c - 1] = sub(a[r][c], ops<T>::mul(l, from_lane(prow, c)));
      a[r][W - 1] = ops<T>::zero();
    }
  }
}

// the same steps on the matrix in memory, for blocks taller than the lanes hold
template <typename T>
__global__ void __launch_bounds__(kLeafThreads)
    leaf_mem_kernel(int n, T *A, long lda, int row0, int w, int *ipiv, int *info) {
  __shared__ double red_v[kLeafThreads / 64];
  __shared__ int red_i[kLeafThreads / 64 + 1];
  __shared__ T pivot;
  leaf_factor<T>(A + row0 + static_cast<long>(row0) * lda, lda, n - row0, w, row0, ipiv, info,
                 red_v, red_i, &pivot);
}

// rows k and ipiv[k] - 1 interchanged for k = k0 .. k1-1 in order, in every column c <
// ncols; in the columns of own0 .. own1-1 none (done) or only those past the column's own
// (a panel whose kernel left those): one lane a column
template <typename T>
__global__ void __launch_bounds__(256)
    laswp_kernel(int ncols, T *A, long lda, const int *ipiv, int k0, int k1, int own0, int own1,
                 bool own_done) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= ncols) return;
  T *col = A + static_cast<long>(c) * lda;
  for (int k = (c < own0 || c >= own1) ? k0 : own_done ? k1 : c + 1; k < k1; ++k) {
    const int p = ipiv[k] - 1;
    if (p != k) {
      const T t = col[k];
      col[k] = col[p];
      col[p] = t;
    }
  }
}

__global__ void fill_info_kernel(int *info, int v) {
  if (threadIdx.x == 0) *info = v;
}
// a first zero pivot was recorded as its column; none leaves INT_MAX, reported as 0
__global__ void finish_info_kernel(int *info) {
  if (threadIdx.x == 0 && *info == INT_MAX) *info = 0;
}

// ---- triangular solves: X = T^-1 B, T of order nb <= 64 -------------------------------------
__device__ inline bool finite(double x) { return isfinite(x); }
__device__ inline bool finite(float x) { return isfinite(x); }
__device__ inline bool finite(zd x) { return isfinite(x.re) && isfinite(x.im); }
__device__ inline bool finite(zc x) { return isfinite(x.re) && isfinite(x.im); }

constexpr int kTrsmWaves = 4;  // waves a workgroup: they share the triangle in LDS
constexpr int kTrsmCols = 4;   // right-hand sides a wave

// lower = true: T unit lower (forward substitution); false: T upper with its diagonal
// (backward). A lane is a row and a wave holds four right-hand sides in registers: step k
// sends row k's value to every lane and subtracts its column of T, so a solve is nb
// multiply-adds deep. (A lane a right-hand side, the rows in LDS, is nb^2 / 2 deep: 46 us
// for nb = 64 however few the columns, now 12 us lower and 24 us upper.) The division by the diagonal is a
// product with its reciprocal and one correction step; the quotient itself where that is
// not finite.
template <typename T, bool kLower>
__global__ void __launch_bounds__(64 * kTrsmWaves)
    trsm_small_kernel(int nb, int ncols, const T *Tm, long ldt, T *B, long ldb) {
  __shared__ T tri[kTrsmNb][kTrsmNb + 1];  // tri[k][i]: column k
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e = tid; e < kTrsmNb * kTrsmNb; e += 64 * kTrsmWaves) {
    const int i = e % kTrsmNb, k = e / kTrsmNb;
    tri[k][i] = (i < nb && k < nb) ? Tm[i + static_cast<long>(k) * ldt] : ops<T>::zero();
  }
  const int c0 = (blockIdx.x * kTrsmWaves + wave) * kTrsmCols;
  T x[kTrsmCols];
#pragma unroll
  for (int c = 0; c < kTrsmCols; ++c)
    x[c] = (lane < nb && c0 + c < ncols) ? B[lane + static_cast<long>(c0 + c) * ldb]
                                         : ops<T>::zero();
  __syncthreads();
  const T diag = kLower ? ops<T>::from_real(1.0) : tri[lane][lane];
  const T rdiag = kLower ? diag : cdiv(ops<T>::from_real(1.0), diag);
#pragma unroll 4
  for (int s = 0; s < nb; ++s) {
    const int k = kLower ? s : nb - 1 - s;
    const T t = tri[k][lane];
    const bool below = kLower ? lane > k : lane < k;
    T dk = diag, rk = rdiag;
    if constexpr (!kLower) {
      dk = from_lane(diag, k);
      rk = from_lane(rdiag, k);
    }
#pragma unroll
    for (int c = 0; c < kTrsmCols; ++c) {
      T xk = from_lane(x[c], k);
      if constexpr (!kLower) {
        const T num = xk;
        T q = ops<T>::mul(num, rk);
        q = ops<T>::add(q, ops<T>::mul(msub(num, q, dk), rk));
        if (!finite(q)) q = cdiv(num, dk);
        xk = q;
        if (lane == k) x[c] = q;
      }
      const T y = sub(x[c], ops<T>::mul(t, xk));
      if (below) x[c] = y;
    }
  }
#pragma unroll
  for (int c = 0; c < kTrsmCols; ++c)
    if (lane < nb && c0 + c < ncols) B[lane + static_cast<long>(c0 + c) * ldb] = x[c];
}

template <typename T>
hipError_t gemm_sub(hipStream_t st, int M, int N, int K, const T *A, long lda, const T *B, long ldb,
                    T *C, long ldc) {
  if (M <= 0 || N <= 0 || K <= 0) return hipSuccess;
  GemmArgs<T> g;
  g.M = M;
  g.N = N;
  g.K = K;
  g.A = A;
  g.lda = lda;
  g.B = B;
  g.ldb = ldb;
  g.C = C;
  g.ldc = ldc;
  g.alpha = ops<T>::from_real(-1.0);
  g.beta = ops<T>::from_real(1.0);
  g.Cin = C;
  g.ldcin = ldc;
  return launch_gemm<T>(st, g);
}

// X = L^-1 B (L unit lower of order nb) or X = U^-1 B (U upper), recursively:
// halves of the triangle with one product between them
template <typename T, bool kLower>
hipError_t trsm(hipStream_t st, int nb, int ncols, const T *Tm, long ldt, T *B, long ldb) {
  if (nb <= 0 || ncols <= 0) return hipSuccess;
  if (nb <= kTrsmNb) {
    constexpr int kCols = kTrsmWaves * kTrsmCols;
    trsm_small_kernel<T, kLower><<<(ncols + kCols - 1) / kCols, 64 * kTrsmWaves, 0, st>>>(
        nb, ncols, Tm, ldt, B, ldb);
    return hipGetLastError();
  }
  const int n1 = nb / 2, n2 = nb - n1;
  const T *T11 = Tm, *T22 = Tm + n1 + static_cast<long>(n1) * ldt;
  T *B1 = B, *B2 = B + n1;
  hipError_t e;
  if (kLower) {
    if ((e = trsm<T, true>(st, n1, ncols, T11, ldt, B1, ldb)) != hipSuccess) return e;
    if ((e = gemm_sub<T>(st, n2, ncols, n1, Tm + n1, ldt, B1, ldb, B2, ldb)) != hipSuccess) return e;
    return trsm<T, true>(st, n2, ncols, T22, ldt, B2, ldb);
  }
  if ((e = trsm<T, false>(st, n2, ncols, T22, ldt, B2, ldb)) != hipSuccess) return e;
  if ((e = gemm_sub<T>(st, n1, ncols, n2, Tm + static_cast<long>(n1) * ldt, ldt, B2, ldb, B1, ldb)) !=
      hipSuccess)
    return e;
  return trsm<T, false>(st, n1, ncols, T11, ldt, B1, ldb);
}

constexpr int kPanelMinCols = 4;
// columns of a panel of m rows: the widest power of two up to 32 whose block is at most
// 128 KiB, which the lanes hold (half of their 256 VGPRs); 0 (the steps in memory) where
// that is fewer than 4, past 4096 FP64, 2048 complex128 or 8192 FP32 rows. (Wider panels,
// and a right-looking split into them, were faster still but rounded every entry once per
// panel: FP64 n = 300 L U off by 1.8e-15 ||A|| against 1.3e-15 for the halves below.)
// In memory up to 8 columns make a panel, where one or two held in LDS did: FP64 n = 16000
// 399 -> 376 ms, complex128 n = 8000 224 -> 148, complex64 n = 9000 180 -> 143.
template <typename T>
constexpr int panel_cols(int m) {
  const long cap = static_cast<long>(131072 / sizeof(T)) / (m < 1 ? 1 : m);
  int w = 0;
  for (int c = 1; c <= kPanelCols && c <= cap; c <<= 1) w = c;
  return w >= kPanelMinCols ? w : 0;
}

// w columns at R rows a lane, the fewest that reach row n
template <typename T, int R>
hipError_t launch_panel(hipStream_t st, int n, T *A, long lda, int k, int w, int *ipiv, int *info) {
  constexpr int W = panel_cols<T>(kPanelThreads * (R / 2) + 1);  // at the fewest rows R serves
  if constexpr (W == 0) {
    return hipErrorInvalidValue;  // not reached: panel_cols gave 0
  } else {
    if (R * kPanelThreads < n - k) return launch_panel<T, 2 * R>(st, n, A, lda, k, w, ipiv, info);
    if (w <= W / 2) panel_kernel<T, W / 2, R><<<1, kPanelThreads, 0, st>>>(n, A, lda, k, w, ipiv, info);
    else panel_kernel<T, W, R><<<1, kPanelThreads, 0, st>>>(n, A, lda, k, w, ipiv, info);
    return hipGetLastError();
  }
}

template <typename T>
hipError_t factor_block(hipStream_t st, int n, T *A, long lda, int k, int w, int *ipiv, int *info) {
  const int m = n - k;
  const int pw = panel_cols<T>(m);
  hipError_t e;
  if (w <= (pw == 0 ? 8 : pw)) {
    if (pw > 0) {
      if ((e = launch_panel<T, 1>(st, n, A, lda, k, w, ipiv, info)) != hipSuccess) return e;
    } else {
      leaf_mem_kernel<T><<<1, kLeafThreads, 0, st>>>(n, A, lda, k, w, ipiv, info);
    }
    laswp_kernel<T><<<(n + 255) / 256, 256, 0, st>>>(n, A, lda, ipiv, k, k + w, k, k + w, pw == 0);
    return hipGetLastError();
  }
  const int w1 = w / 2, w2 = w - w1;
  if ((e = factor_block<T>(st, n, A, lda, k, w1, ipiv, info)) != hipSuccess) return e;
  T *A11 = A + k + static_cast<long>(k) * lda;
  T *A12 = A + k + static_cast<long>(k + w1) * lda;
  T *A21 = A + k + w1 + static_cast<long>(k) * lda;
  T *A22 = A + k + w1 + static_cast<long>(k + w1) * lda;
  if ((e = trsm<T, true>(st, w1, w2, A11, lda, A12, lda)) != hipSuccess) return e;
  if ((e = gemm_sub<T>(st, m - w1, w2, w1, A21, lda, A12, lda, A22, lda)) != hipSuccess) return e;
  return factor_block<T>(st, n, A, lda, k + w1, w2, ipiv, info);
}

}  // namespace

template <typename T>
hipError_t launch_getrf(hipStream_t st, int n, T *A, long lda, int *ipiv, int *info) {
  fill_info_kernel<<<1, 64, 0, st>>>(info, INT_MAX);
  const hipError_t e = factor_block<T>(st, n, A, lda, 0, n, ipiv, info);
  if (e != hipSuccess) return e;
  finish_info_kernel<<<1, 64, 0, st>>>(info);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_getrs(hipStream_t st, int n, int nrhs, const T *LU, long lda, const int *ipiv,
                        T *B, long ldb) {
  if (n <= 0 || nrhs <= 0) return hipSuccess;
  laswp_kernel<T><<<(nrhs + 255) / 256, 256, 0, st>>>(nrhs, B, ldb, ipiv, 0, n, 0, 0, true);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if ((e = trsm<T, true>(st, n, nrhs, LU, lda, B, ldb)) != hipSuccess) return e;
  return trsm<T, false>(st, n, nrhs, LU, lda, B, ldb);
}

#define CLM_LU_INST(T)                                                                        \
  template hipError_t launch_getrf<T>(hipStream_t, int, T *, long, int *, int *);             \
  template hipError_t launch_getrs<T>(hipStream_t, int, int, const T *, long, const int *, T *, \
                                      long);
CLM_LU_INST(double)
CLM_LU_INST(float)
CLM_LU_INST(zd)
CLM_LU_INST(zc)
#undef CLM_LU_INST

}  // namespace clm

// herm.hip -- exp(A) for a symmetric (real) or Hermitian (complex) A: the reference's
// expm_herm (src/expm/expm_herm.cppm:145-199, herm_exp_scale in
// src/expm/expm.cu:170-184), which takes the eigendecomposition from the vendor solver
// (syevd / heevd). Here there are two routes.
//
// For ||A||_1 <= 32 the uplo triangle is mirrored, shifted by mu = tr(A) / n and handed
// to the library's Taylor / Paterson-Stockmeyer exponential in double, and the result is
// multiplied by e^mu: 5 to 15 MFMA products of full tiles instead of 8 to 12 Jacobi sweeps,
// each 2k - 1 rounds of a launch that runs on k CUs only. The shift puts the spectrum
// around 0, so the polynomial's rounding is relative to its largest value e^r and not to
// the cancelling terms of a negative spectrum. Measured, complex128 n = 512 at
// ||A||_1 = 8: 35.1 ms by Jacobi -> 0.28 ms, error against 64-bit eigh 1.8e-13 -> 3.1e-15.
//
// The line at 32: over orders 3 to 300 and spectra one-sided, wide and with one outlier of
// either sign, the Taylor route's error against extended precision is at or below the
// sweeps' at every norm to 32 (n = 16, an outlier below: 2.9e-15 against 2.9e-15 at 32,
// 6.3e-15 against 2.8e-15 at 48): squarings amplify the polynomial's rounding. Beyond it,
// for a diagonal A (whose exponential the sweeps leave exact to the last place) and in a
// workspace that holds only its blocks, the eigendecomposition is this library's own
// blocked two-sided Jacobi method:
//
//   * the uplo triangle is mirrored into a full matrix H of order np = n rounded up
//     to 64 (zero padding adds eigenvalues 0 whose exponentials land outside the
//     n x n block the result keeps, so the block is exp(A) exactly as before);
//   * H is cut into 2k blocks of 32; a sweep pairs every block with every other once
//     over 2k - 1 rounds (the circle method). A round is two launches: one workgroup
//     per pair runs one cyclic Jacobi sweep over its 64 x 64 subproblem in LDS
//     (32 disjoint rotations at a time, circle order again), keeping the unitary Q;
//     then one launch applies Q_t^H H_tu Q_u to every off-diagonal tile (t < u, the
//     mirror written as its adjoint) and V <- V Q_u to the eigenvector tiles, skipping
//     pairs whose Q stayed the identity;
//   * an entry is rotated when its modulus exceeds delta = u ||H||_F / np, so when a
//     whole sweep rotates nothing every off-diagonal entry is at most delta and
//     ||off(H)||_F <= u ||H||_F (u = 2^-53 or 2^-24); one read-back per sweep;
//   * M = V diag(exp(w)) over the first n rows, then exp(A) = M V^H on the library's
//     MFMA product (V^H staged once, the product is NN).
#include "clm_internal.hpp"
#include "calaman_expm.h"

#include <algorithm>
#include <cmath>

namespace clm {
namespace {

constexpr int kB = 32;             // block width
constexpr int kP = 2 * kB;         // a pair of blocks: the subproblem order
constexpr int kLd = kP + 1;        // LDS row pitch
constexpr int kThreads = 256;      // one workgroup per tile (a lane a 4 x 4 block)
constexpr int kSolveThreads = 1024;  // one workgroup per subproblem (32 lanes a rotation)
constexpr int kInnerSweeps = 1;    // Jacobi sweeps of one subproblem per round: more
                                   // sweeps save no outer sweep at n >= 128 and every
                                   // rotation adds its rounding to V
constexpr int kMaxSweeps = 30;     // cap on the sweeps over the whole matrix

__device__ inline double conj_(double x) { return x; }
__device__ inline float conj_(float x) { return x; }
__device__ inline zd conj_(zd x) { return zd{x.re, -x.im}; }
__device__ inline zc conj_(zc x) { return zc{x.re, -x.im}; }
__device__ inline double re_(double x) { return x; }
__device__ inline float re_(float x) { return x; }
__device__ inline double re_(zd x) { return x.re; }
__device__ inline float re_(zc x) { return x.re; }
__device__ inline double abs_(double x) { return fabs(x); }
__device__ inline double abs_(zd x) { return hypot(x.re, x.im); }
__device__ inline double abs2_(double x) { return x * x; }
__device__ inline double abs2_(zd x) { return x.re * x.re + x.im * x.im; }
__device__ inline double exp_(double x) { return exp(x); }
// The working type: the Jacobi sweeps of the single-precision types run in double
// (their rotations' rounding would otherwise reach 1e-5 of exp(A) at n = 128)
template <typename T>
struct work_type {
  using type = T;
};
template <>
struct work_type<float> {
  using type = double;
};
template <>
struct work_type<zc> {
  using type = zd;
};
template <typename T>
using work_t = typename work_type<T>::type;
__device__ inline double widen(double x) { return x; }
__device__ inline double widen(float x) { return x; }
__device__ inline zd widen(zd x) { return x; }
__device__ inline zd widen(zc x) { return zd{x.re, x.im}; }
template <typename T>
__device__ inline T narrow(work_t<T> x);  // defined for the single-precision types
template <>
__device__ inline float narrow<float>(double x) { return static_cast<float>(x); }
template <>
__device__ inline zc narrow<zc>(zd x) { return zc{static_cast<float>(x.re), static_cast<float>(x.im)}; }

template <typename T>
__device__ inline T sub_(T a, T b) {
  return ops<T>::add(a, ops<T>::scale(b, -1.0));
}
template <typename T>
__device__ inline T mac_(T acc, T a, T b) {
  return ops<T>::add(acc, ops<T>::mul(a, b));
}

// the circle method over np2 positions (np2 even): pair t of round r
__device__ inline void pair_of(int r, int t, int np2, int &p, int &q) {
  const int m = np2 - 1;
  if (t == 0) {
    p = r;
    q = m;
  } else {
    p = (r + t) % m;
    q = (r - t + m) % m;
  }
}

// H = the uplo triangle of A mirrored (real diagonal), zero-padded to np x np, in the
// working type W; V (when given) = I
template <typename T, typename W>
__global__ void __launch_bounds__(kThreads)
    mirror_kernel(int n, int np, int upper, const T *__restrict__ A, long lda, W *__restrict__ H,
                  W *__restrict__ V) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= np) return;
  W v = ops<W>::zero();
  if (i < n && j < n) {
    if (i == j) v = ops<W>::from_real(re_(A[i + static_cast<long>(i) * lda]));
    else if ((i < j) == (upper != 0)) v = widen(A[i + static_cast<long>(j) * lda]);
    else v = widen(conj_(A[j + static_cast<long>(i) * lda]));
  }
  H[i + static_cast<long>(j) * np] = v;
  if (V) V[i + static_cast<long>(j) * np] = ops<W>::from_real(i == j ? 1.0 : 0.0);
}
// E = the n x n result rounded to the caller's type
template <typename T, typename W>
__global__ void __launch_bounds__(kThreads)
    narrow_kernel(int n, const W *__restrict__ X, T *__restrict__ E, long lde) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  const int j = blockIdx.y;
  if (i < n) E[i + static_cast<long>(j) * lde] = narrow<T>(X[i + static_cast<long>(j) * n]);
}

// colsq[j] = sum_i |H(i, j)|^2
template <typename T>
__global__ void __launch_bounds__(kThreads) colsq_kernel(int np, const T *H, real_t<T> *colsq) {
  using R = real_t<T>;
  __shared__ R red[kThreads];
  const int j = blockIdx.x;
  R s = R(0);
  for (int i = threadIdx.x; i < np; i += kThreads) s += abs2_(H[i + static_cast<long>(j) * np]);
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (static_cast<int>(threadIdx.x) < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) colsq[j] = red[0];
}
// delta = u sqrt(sum colsq) / np
template <typename T>
__global__ void __launch_bounds__(kThreads)
    delta_kernel(int np, const real_t<T> *colsq, real_t<T> u, real_t<T> *delta) {
  using R = real_t<T>;
  __shared__ R red[kThreads];
  R s = R(0);
  for (int j = threadIdx.x; j < np; j += kThreads) s += colsq[j];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (static_cast<int>(threadIdx.x) < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *delta = u * sqrt(red[0]) / static_cast<R>(np);
}

__global__ void clear_count_kernel(int *c) {
  if (threadIdx.x == 0) *c = 0;
}

// local index l of a 64-wide pair (p, q) -> global index
__device__ inline int glob(int l, int p, int q) { return l < kB ? p * kB + l : q * kB + (l - kB); }

// The subproblem of pair t in round r: S = H[{p,q},{p,q}] in LDS, one cyclic sweep of
// rotations J = [[c, e s], [-conj(e) s, c]] (e = S_ij / |S_ij|, t = sign(tau) /
// (|tau| + sqrt(1 + tau^2)), tau = (S_jj - S_ii) / (2 |S_ij|), c = 1 / sqrt(1 + t^2),
// s = t c: the real symmetric Jacobi rotation conjugated by the phase of S_ij),
// S <- J^H S J and Q <- Q J. 32 lanes serve one rotation of a round: each computes
// the rotation itself from the same three entries (no broadcast), updates two of
// the pair's 64 columns of rows i, j, then -- after every row update -- two rows of
// columns i, j of S and of Q. Two barriers a round. Writes S back and Q to Qbuf[t]
// when anything rotated.
template <typename W>
__global__ void __launch_bounds__(kSolveThreads)
    solve_kernel(int np, W *H, const real_t<W> *delta, int round, W *Qbuf, int *flags,
                 int *count) {
  using R = real_t<W>;
  __shared__ W S[kP][kLd];
  __shared__ W Q[kP][kLd];
  __shared__ int sweep_rot;
  const int np2 = np / kB;
  const int t = blockIdx.x;
  int p, q;
  pair_of(round, t, np2, p, q);
  const long ld = np;
  for (int e = threadIdx.x; e < kP * kP; e += kSolveThreads) {
    const int r = e % kP, c = e / kP;
    S[r][c] = H[glob(r, p, q) + glob(c, p, q) * ld];
    Q[r][c] = ops<W>::from_real(r == c ? 1.0 : 0.0);
  }
  const int m = threadIdx.x >> 5;  // the rotation this lane serves (32 lanes each)
  const int sl = threadIdx.x & 31;
  const R d = *delta;
  bool any = false;
  for (int sw = 0; sw < kInnerSweeps; ++sw) {
    if (threadIdx.x == 0) sweep_rot = 0;
    __syncthreads();
    for (int r = 0; r < kP - 1; ++r) {
      int a, b;
      pair_of(r, m, kP, a, b);
      const int i = min(a, b), j = max(a, b);
      // rows i and j are this pair's alone until the barrier: the three entries are
      // read by all 32 lanes before any of them writes
      const W c = S[i][j];
      const R absc = abs_(c);
      const bool on = absc > d;  // false for NaN
      R cs = R(1), di = R(0), dj = R(0);
      W es = ops<W>::zero();
      if (on) {
        const R aii = re_(S[i][i]), ajj = re_(S[j][j]);
        const R tau = (ajj - aii) / (R(2) * absc);
        const R at = fabs(tau);
        const R tt = at > R(1e150) ? R(0.5) / tau
                                   : (tau >= R(0) ? R(1) : R(-1)) / (at + sqrt(R(1) + tau * tau));
        cs = R(1) / sqrt(R(1) + tt * tt);
        es = ops<W>::scale(c, tt * cs / absc);
        di = aii - tt * absc;
        dj = ajj + tt * absc;
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // rows i, j: S <- J^H S
          const int col = sl + 32 * h;
          const W xi = S[i][col], xj = S[j][col];
          S[i][col] = sub_(ops<W>::scale(xi, cs), ops<W>::mul(es, xj));
          S[j][col] = mac_(ops<W>::scale(xj, cs), conj_(es), xi);
        }
        if (sl == 0) atomicAdd(&sweep_rot, 1);
      }
      __syncthreads();
      if (on) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // columns i, j: S <- S J, Q <- Q J
          const int row = sl + 32 * h;
          const W xi = S[row][i], xj = S[row][j];
          W ni = sub_(ops<W>::scale(xi, cs), ops<W>::mul(conj_(es), xj));
          W nj = mac_(ops<W>::scale(xj, cs), es, xi);
          if (row == i) {
            ni = ops<W>::from_real(di);
            nj = ops<W>::zero();
          } else if (row == j) {
            ni = ops<W>::zero();
            nj = ops<W>::from_real(dj);
          }
          S[row][i] = ni;
          S[row][j] = nj;
          const W qi = Q[row][i], qj = Q[row][j];
          Q[row][i] = sub_(ops<W>::scale(qi, cs), ops<W>::mul(conj_(es), qj));
          Q[row][j] = mac_(ops<W>::scale(qj, cs), es, qi);
        }
      }
      __syncthreads();
    }
    const bool quiet = sweep_rot == 0;
    __syncthreads();  // every lane has read the count before the next sweep clears it
    if (quiet) break;
    any = true;
  }
  if (any) {
    W *Qt = Qbuf + static_cast<long>(t) * kP * kP;
    for (int e = threadIdx.x; e < kP * kP; e += kSolveThreads) {
      const int r = e % kP, c = e / kP;
      H[glob(r, p, q) + glob(c, p, q) * ld] = S[r][c];
      Qt[r + c * kP] = Q[r][c];
    }
  }
  if (threadIdx.x == 0) {
    flags[t] = any ? 1 : 0;
    if (any) atomicAdd(count, 1);
  }
}

// acc = X * Y over 64 x 64 tiles in LDS (adj: X^H * Y); a lane a 4 x 4 block of the
// result: rows lane % 16 + 16 a (16 consecutive rows per k across a lane group, so
// the X reads fall on distinct banks), columns 4 (lane / 16) + b (one Y element a
// lane group: a broadcast)
template <typename T, bool kAdjX>
__device__ inline void tile_product(const T (*X)[kLd], const T (*Y)[kLd], T (&acc)[4][4]) {
  const int r0 = threadIdx.x % 16, c0 = 4 * (threadIdx.x / 16);
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = ops<T>::zero();
  for (int k = 0; k < kP; ++k) {
    T x[4], y[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) x[a] = kAdjX ? conj_(X[k][r0 + 16 * a]) : X[r0 + 16 * a][k];
#pragma unroll
    for (int b = 0; b < 4; ++b) y[b] = Y[k][c0 + b];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = mac_(acc[a][b], x[a], y[b]);
  }
}
template <typename T>
__device__ inline void tile_store(T (*X)[kLd], const T (&acc)[4][4]) {
  const int r0 = threadIdx.x % 16, c0 = 4 * (threadIdx.x / 16);
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) X[r0 + 16 * a][c0 + b] = acc[a][b];
}

// One launch per round: jobs [0, k(k-1)/2) are the tiles (t, u), t < u, of H:
// H_tu <- Q_t^H H_tu Q_u and H_ut = H_tu^H; jobs past them are V's tiles (64 rows,
// pair u): V <- V Q_u. Tiles whose Q are both the identity are skipped.
template <typename T>
__global__ void __launch_bounds__(kThreads)
    update_kernel(int np, T *H, T *V, int round, const T *Qbuf, const int *flags) {
  __shared__ T X[kP][kLd];
  __shared__ T Y[kP][kLd];
  const int np2 = np / kB, k = np2 / 2;
  const int nA = k * (k - 1) / 2;
  const long ld = np;
  int job = blockIdx.x;
  T acc[4][4];
  if (job < nA) {
    int t = 0, rem = job;
    while (rem >= k - 1 - t) {
      rem -= k - 1 - t;
      ++t;
    }
    const int u = t + 1 + rem;
    const bool ft = flags[t] != 0, fu = flags[u] != 0;
    if (!ft && !fu) return;
    int pt, qt, pu, qu;
    pair_of(round, t, np2, pt, qt);
    pair_of(round, u, np2, pu, qu);
    for (int e = threadIdx.x; e < kP * kP; e += kThreads) {
      const int r = e % kP, c = e / kP;
      X[r][c] = H[glob(r, pt, qt) + glob(c, pu, qu) * ld];
    }
    if (fu) {
      const T *Qu = Qbuf + static_cast<long>(u) * kP * kP;
      for (int e = threadIdx.x; e < kP * kP; e += kThreads) Y[e % kP][e / kP] = Qu[e];
      __syncthreads();
      tile_product<T, false>(X, Y, acc);
      __syncthreads();
      tile_store<T>(X, acc);
    }
    if (ft) {
      const T *Qt = Qbuf + static_cast<long>(t) * kP * kP;
      for (int e = threadIdx.x; e < kP * kP; e += kThreads) Y[e % kP][e / kP] = Qt[e];
      __syncthreads();
      tile_product<T, true>(Y, X, acc);
      __syncthreads();
      tile_store<T>(X, acc);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < kP * kP; e += kThreads) {
      const int r = e % kP, c = e / kP;
      H[glob(r, pt, qt) + glob(c, pu, qu) * ld] = X[r][c];
    }
    for (int e = threadIdx.x; e < kP * kP; e += kThreads) {  // the adjoint, rows of it coalesced
      const int c = e % kP, r = e / kP;
      H[glob(c, pu, qu) + glob(r, pt, qt) * ld] = conj_(X[r][c]);
    }
    return;
  }
  job -= nA;
  const int u = job % k, rb = job / k;
  if (flags[u] == 0) return;
  int pu, qu;
  pair_of(round, u, np2, pu, qu);
  const T *Qu = Qbuf + static_cast<long>(u) * kP * kP;
  for (int e = threadIdx.x; e < kP * kP; e += kThreads) {
    const int r = e % kP, c = e / kP;
    X[r][c] = V[rb * kP + r + glob(c, pu, qu) * ld];
    Y[r][c] = Qu[e];
  }
  __syncthreads();
  tile_product<T, false>(X, Y, acc);
  __syncthreads();
  tile_store<T>(X, acc);
  __syncthreads();
  for (int e = threadIdx.x; e < kP * kP; e += kThreads) {
    const int r = e % kP, c = e / kP;
    V[rb * kP + r + glob(c, pu, qu) * ld] = X[r][c];
  }
}

// w = the real diagonal of H; M = V diag(exp(w)) over rows < n (leading dimension n)
template <typename T>
__global__ void __launch_bounds__(kThreads)
    exp_scale_kernel(int n, int np, const T *H, const T *V, T *M) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= n) return;
  const real_t<T> w = re_(H[j + static_cast<long>(j) * np]);
  M[i + static_cast<long>(j) * n] = ops<T>::scale(V[i + static_cast<long>(j) * np], exp_(w));
}
// W = V(0:n, :)^H (np x n, leading dimension np)
template <typename T>
__global__ void __launch_bounds__(kThreads) adjoint_rows_kernel(int n, int np, const T *V, T *W) {
  const int k = blockIdx.x * kThreads + threadIdx.x;
  const int j = blockIdx.y;
  if (k < np && j < n) W[k + static_cast<long>(j) * np] = conj_(V[j + static_cast<long>(k) * np]);
}

__global__ void set_info_kernel(int *info, int v) {
  if (threadIdx.x == 0) *info = v;
}

// ---- the Taylor route -------------------------------------------------------------------
constexpr double kTaylorMaxNorm1 = 32.0;
// the largest workspace a size query asks for on this route's account (it takes 7/3 of the
// sweeps' in the double types, 8/3 in the single ones): past it, from orders of 23 000
// (complex64) to 35 000 (FP64), a call whose A, E and sweeps' blocks fit the card might not
// get this one; it runs the sweeps then
constexpr size_t kTaylorMaxBytes = size_t(64) << 30;

// the larger; a NaN on either side stays
__device__ inline double nan_max_(double best, double v) { return v > best || isnan(v) ? v : best; }

// stats[j] = column j's 1-norm, stats[n + j] = its part off the diagonal
template <typename W>
__global__ void __launch_bounds__(kThreads) column_stats_kernel(int n, const W *H, double *stats) {
  __shared__ double all[kThreads], off[kThreads];
  const int j = blockIdx.x;
  double a = 0.0, o = 0.0;
  for (int i = threadIdx.x; i < n; i += kThreads) {
    const double v = abs_(H[i + static_cast<long>(j) * n]);
    a += v;
    if (i != j) o += v;
  }
  all[threadIdx.x] = a;
  off[threadIdx.x] = o;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (static_cast<int>(threadIdx.x) < w) {
      all[threadIdx.x] += all[threadIdx.x + w];
      off[threadIdx.x] += off[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    stats[j] = all[0];
    stats[n + j] = off[0];
  }
}
// out = {||H||_1, the largest off-diagonal column sum, tr(H) / n}
template <typename W>
__global__ void __launch_bounds__(kThreads)
    fold_stats_kernel(int n, const W *H, const double *stats, double *out) {
  __shared__ double red[3][kThreads];
  const int t = threadIdx.x;
  double a = 0.0, o = 0.0, d = 0.0;
  for (int j = t; j < n; j += kThreads) {
    a = nan_max_(a, stats[j]);
    o = nan_max_(o, stats[n + j]);
    d += re_(H[j + static_cast<long>(j) * n]);
  }
  red[0][t] = a;
  red[1][t] = o;
  red[2][t] = d;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (t < w) {
      red[0][t] = nan_max_(red[0][t], red[0][t + w]);
      red[1][t] = nan_max_(red[1][t], red[1][t + w]);
      red[2][t] += red[2][t + w];
    }
    __syncthreads();
  }
  if (t == 0) {
    out[0] = red[0][0];
    out[1] = red[1][0];
    out[2] = red[2][0] / n;
  }
}
// H -= mu I
template <typename W>
__global__ void __launch_bounds__(kThreads) shift_kernel(int n, W *H, double mu) {
  const int j = blockIdx.x * kThreads + threadIdx.x;
  if (j < n) {
    W *d = H + j + static_cast<long>(j) * n;
    *d = ops<W>::from_real(re_(*d) - mu);
  }
}
// E = f X in the caller's type (X may be E)
template <typename T, typename W>
__global__ void __launch_bounds__(kThreads)
    unshift_kernel(int n, double f, const W *X, long ldx, T *E, long lde) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  const long j = blockIdx.y;
  if (i >= n) return;
  const W x = ops<W>::scale(X[i + j * ldx], f);
  if constexpr (std::is_same_v<T, W>) E[i + j * lde] = x;
  else E[i + j * lde] = narrow<T>(x);
}

inline clm_status_t general_bytes(double, int n, size_t *b) { return clm_expm_buffer_size_d(n, b); }
inline clm_status_t general_bytes(zd, int n, size_t *b) { return clm_expm_buffer_size_z(n, b); }
inline clm_status_t general_expm(clm_ctx *ctx, hipStream_t st, int n, const double *A, double *E,
                                 int lde, void *work, size_t bytes) {
  return clm_expm_d(ctx, st, n, A, n, E, lde, work, bytes, nullptr, nullptr);
}
inline clm_status_t general_expm(clm_ctx *ctx, hipStream_t st, int n, const zd *A, zd *E, int lde,
                                 void *work, size_t bytes) {
  return clm_expm_z(ctx, st, n, reinterpret_cast<const clm_double_complex *>(A), n,
                    reinterpret_cast<clm_double_complex *>(E), lde, work, bytes, nullptr, nullptr);
}

template <typename T>
struct HermTaylorWs {
  using W = work_t<T>;
  W *H = nullptr, *X = nullptr;  // X: the result of a single-precision call, in double
  double *stats = nullptr, *out = nullptr;
  char *work = nullptr;
  size_t work_bytes = 0;
  size_t carve(void *base, int n) {
    const size_t nn = static_cast<size_t>(n) * n;
    Layout L(base);
    H = L.take<W>(nn);
    if constexpr (!std::is_same_v<T, W>) X = L.take<W>(nn);
    stats = L.take<double>(2 * static_cast<size_t>(n));
    out = L.take<double>(3);
    (void)general_bytes(W{}, n, &work_bytes);
    work = L.take<char>(work_bytes);
    return L.total();
  }
};

// *done = whether the Taylor route applied (and then E holds the result)
template <typename T>
clm_status_t herm_taylor(clm_ctx *ctx, int device, hipStream_t st, int upper, int n, const T *A,
                         int lda, T *E, int lde, void *work, int *info, bool *done) {
  using W = work_t<T>;
  HermTaylorWs<T> ws;
  ws.carve(work, n);
  const dim3 grid((n + kThreads - 1) / kThreads, n);
  mirror_kernel<T, W><<<grid, kThreads, 0, st>>>(n, n, upper, A, lda, ws.H, nullptr);
  column_stats_kernel<W><<<n, kThreads, 0, st>>>(n, ws.H, ws.stats);
  fold_stats_kernel<W><<<1, kThreads, 0, st>>>(n, ws.H, ws.stats, ws.out);
  CLM_TRY_HIP(hipGetLastError());
  double v[3] = {};
  CLM_TRY(read_device_values<double>(st, device, ws.out, 3, v));
  *done = v[0] <= kTaylorMaxNorm1 && v[1] > 0.0;  // false for NaN
  if (!*done) return CLM_STATUS_SUCCESS;
  const double mu = v[2];
  shift_kernel<W><<<(n + kThreads - 1) / kThreads, kThreads, 0, st>>>(n, ws.H, mu);
  CLM_TRY_HIP(hipGetLastError());
  W *X;
  int ldx;
  if constexpr (std::is_same_v<T, W>) {
    X = E;
    ldx = lde;
  } else {
    X = ws.X;
    ldx = n;
  }
  CLM_TRY(general_expm(ctx, st, n, ws.H, X, ldx, ws.work, ws.work_bytes));
  unshift_kernel<T, W><<<grid, kThreads, 0, st>>>(n, std::exp(mu), X, ldx, E, lde);
  if (info) set_info_kernel<<<1, 64, 0, st>>>(info, 0);
  CLM_TRY_HIP(hipGetLastError());
  return CLM_STATUS_SUCCESS;
}

template <typename T>
struct HermWs {
  T *H = nullptr, *V = nullptr, *W = nullptr, *Q = nullptr;
  int *flags = nullptr, *count = nullptr;
  real_t<T> *delta = nullptr, *colsq = nullptr;
  size_t carve(void *base, int n) {
    const size_t np = static_cast<size_t>((n + kP - 1) / kP) * kP;
    const size_t k = np / kP;
    Layout L(base);
    H = L.take<T>(np * np);
    V = L.take<T>(np * np);
    W = L.take<T>(np * np);
    Q = L.take<T>(k * kP * kP);
    flags = L.take<int>(k);
    count = L.take<int>(1);
    delta = L.take<real_t<T>>(1);
    colsq = L.take<real_t<T>>(np);
    return L.total();
  }
};

template <typename T>
clm_status_t herm_bytes(int n, size_t *bytes) {
  if (bytes == nullptr || n < 1 || n > kMaxDim) return CLM_STATUS_INVALID_VALUE;
  HermWs<work_t<T>> ws;
  HermTaylorWs<T> tw;
  const size_t sweeps = ws.carve(nullptr, n), taylor = tw.carve(nullptr, n);
  *bytes = taylor > kTaylorMaxBytes ? sweeps : std::max(sweeps, taylor);
  return CLM_STATUS_SUCCESS;
}

template <typename T>
clm_status_t expm_herm_impl(clm_ctx *ctx, hipStream_t st, int uplo, int n, const T *A, int lda,
                            T *E, int lde, void *work, size_t bytes, int *info) {
  using W = work_t<T>;
  using R = real_t<W>;
  if (n < 1 || n > kMaxDim || lda < n || lde < n || A == nullptr || E == nullptr ||
      work == nullptr || (uplo != CLM_FILL_MODE_LOWER && uplo != CLM_FILL_MODE_UPPER))
    return CLM_STATUS_INVALID_VALUE;
  HermWs<W> ws;
  if (bytes < ws.carve(nullptr, n)) return CLM_STATUS_ALLOC_FAILED;
  clm_ctx *c = nullptr;
  CLM_TRY(resolve_ctx(ctx, &c));
  // a workspace of the Jacobi blocks alone (the size before the Taylor route) stays good
  if (HermTaylorWs<T> tw; bytes >= tw.carve(nullptr, n)) {
    bool done = false;
    CLM_TRY(herm_taylor<T>(ctx, c->device, st, uplo == CLM_FILL_MODE_UPPER, n, A, lda, E, lde, work,
                           info, &done));
    if (done) return CLM_STATUS_SUCCESS;
  }
  ws.carve(work, n);
  const int np = (n + kP - 1) / kP * kP;
  const int np2 = np / kB, k = np2 / 2;
  const dim3 grid_sq((np + kThreads - 1) / kThreads, np);
  mirror_kernel<T, W><<<grid_sq, kThreads, 0, st>>>(n, np, uplo == CLM_FILL_MODE_UPPER, A, lda,
                                                    ws.H, ws.V);
  colsq_kernel<W><<<np, kThreads, 0, st>>>(np, ws.H, ws.colsq);
  // the unit roundoff of the working precision, 2^-53
  delta_kernel<W><<<1, kThreads, 0, st>>>(np, ws.colsq, R(1.1102230246251565e-16), ws.delta);
  CLM_TRY_HIP(hipGetLastError());
  bool converged = false;
  const int jobs = k * (k - 1) / 2 + k * k;
  for (int sweep = 0; sweep < kMaxSweeps && !converged; ++sweep) {
    clear_count_kernel<<<1, 64, 0, st>>>(ws.count);
    for (int r = 0; r < np2 - 1; ++r) {
      solve_kernel<W><<<k, kSolveThreads, 0, st>>>(np, ws.H, ws.delta, r, ws.Q, ws.flags, ws.count);
      update_kernel<W><<<jobs, kThreads, 0, st>>>(np, ws.H, ws.V, r, ws.Q, ws.flags);
    }
    CLM_TRY_HIP(hipGetLastError());
    double rotated = 0;
    CLM_TRY(read_device_values<int>(st, c->device, ws.count, 1, &rotated));
    converged = rotated == 0;
  }
  if (info) {
    set_info_kernel<<<1, 64, 0, st>>>(info, converged ? 0 : 1);
    CLM_TRY_HIP(hipGetLastError());
  }
  // M = V diag(exp(w)) (rows < n) over W's storage first, then V(0:n,:)^H over H's (the
  // eigenvalues have been read by then), then exp(A) = M V^H: into E directly, or, for
  // the single-precision types, into V's storage and rounded into E
  W *M = ws.W;
  exp_scale_kernel<W><<<dim3((n + kThreads - 1) / kThreads, np), kThreads, 0, st>>>(n, np, ws.H,
                                                                                   ws.V, M);
  CLM_TRY_HIP(hipGetLastError());
  W *Vh = ws.H;
  adjoint_rows_kernel<W><<<dim3((np + kThreads - 1) / kThreads, n), kThreads, 0, st>>>(n, np, ws.V,
                                                                                       Vh);
  CLM_TRY_HIP(hipGetLastError());
  constexpr bool kSame = std::is_same_v<T, W>;
  GemmArgs<W> g;
  g.M = n;
  g.N = n;
  g.K = np;
  g.A = M;
  g.lda = n;
  g.B = Vh;
  g.ldb = np;
  if constexpr (kSame) {
    g.C = E;
    g.ldc = lde;
  } else {
    g.C = ws.V;
    g.ldc = n;
  }
  g.alpha = ops<W>::from_real(1.0);
  g.beta = ops<W>::zero();
  CLM_TRY_HIP(launch_gemm<W>(st, g));
  if constexpr (!kSame) {
    narrow_kernel<T, W><<<dim3((n + kThreads - 1) / kThreads, n), kThreads, 0, st>>>(n, ws.V, E,
                                                                                     lde);
    CLM_TRY_HIP(hipGetLastError());
  }
  return CLM_STATUS_SUCCESS;
}

}  // namespace
}  // namespace clm

using clm::zc;
using clm::zd;

extern "C" {

clm_status_t clm_expm_herm_buffer_size_s(int n, size_t *b) { return clm::herm_bytes<float>(n, b); }
clm_status_t clm_expm_herm_buffer_size_d(int n, size_t *b) { return clm::herm_bytes<double>(n, b); }
clm_status_t clm_expm_herm_buffer_size_c(int n, size_t *b) { return clm::herm_bytes<zc>(n, b); }
clm_status_t clm_expm_herm_buffer_size_z(int n, size_t *b) { return clm::herm_bytes<zd>(n, b); }

clm_status_t clm_expm_herm_s(clm_ctx *ctx, clm_stream_t stream, int uplo, int n, const float *dA,
                             int lda, float *dE, int lde, void *dWork, size_t lwork_bytes,
                             int *dInfo) {
  return clm::expm_herm_impl<float>(ctx, static_cast<hipStream_t>(stream), uplo, n, dA, lda, dE,
                                    lde, dWork, lwork_bytes, dInfo);
}
clm_status_t clm_expm_herm_d(clm_ctx *ctx, clm_stream_t stream, int uplo, int n, const double *dA,
                             int lda, double *dE, int lde, void *dWork, size_t lwork_bytes,
                             int *dInfo) {
  return clm::expm_herm_impl<double>(ctx, static_cast<hipStream_t>(stream), uplo, n, dA, lda, dE,
                                     lde, dWork, lwork_bytes, dInfo);
}
clm_status_t clm_expm_herm_c(clm_ctx *ctx, clm_stream_t stream, int uplo, int n,
                             const clm_float_complex *dA, int lda, clm_float_complex *dE, int lde,
                             void *dWork, size_t lwork_bytes, int *dInfo) {
  return clm::expm_herm_impl<zc>(ctx, static_cast<hipStream_t>(stream), uplo, n,
                                 reinterpret_cast<const zc *>(dA), lda, reinterpret_cast<zc *>(dE),
                                 lde, dWork, lwork_bytes, dInfo);
}
clm_status_t clm_expm_herm_z(clm_ctx *ctx, clm_stream_t stream, int uplo, int n,
                             const clm_double_complex *dA, int lda, clm_double_complex *dE, int lde,
                             void *dWork, size_t lwork_bytes, int *dInfo) {
  return clm::expm_herm_impl<zd>(ctx, static_cast<hipStream_t>(stream), uplo, n,
                                 reinterpret_cast<const zd *>(dA), lda, reinterpret_cast<zd *>(dE),
                                 lde, dWork, lwork_bytes, dInfo);
}

}  // extern "C"

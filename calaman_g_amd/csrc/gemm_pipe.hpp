// gemm_pipe.hpp -- the product of a workgroup tile with its operands fetched several K
// slices ahead, for the launches that leave the chip short of waves.
//
// A 16-byte vector is staged per lane and step (2 FP64 / complex64, 4 FP32, 1
// complex128 elements), at element alignment: column-major operands of an odd order
// start their columns off 16 bytes, and the vector memory path takes such loads
// whole. The last tile of a ragged row or column of tiles is moved back to end at the
// matrix's edge (it recomputes rows of its neighbour and stores its own only), so every
// tile of a matrix at least a tile wide is full; the last K slice, and matrices
// narrower than a tile, read the last full vector of a line and shift it (zeros past
// the end).
//
// The slices of the next kAhead steps are in flight in registers while one is
// multiplied from LDS (two stages, one barrier a slice): with one wave per SIMD
// nothing else hides the 1-2 us a slice takes to arrive.
//
// The MFMA operands are exchanged (D = B^T A^T on the transposed 16 x 16 tile): the
// same products, summed in the same order (k ascending, four per step), with the
// result's rows on consecutive lanes, so C, Cin and the Paterson-Stockmeyer blocks
// are touched in 64- to 256-byte column pieces straight from the registers.
#pragma once

#include "gemm_tile.hpp"

namespace clm {
namespace pipe {

using tile::CxReal;
using tile::Mfma;

typedef unsigned u4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(4))) U4 {
  u4 v;
};

template <typename T>
constexpr bool is_cx = std::is_same_v<T, zd> || std::is_same_v<T, zc>;
template <typename T>
struct Plane {
  using type = T;
};
template <>
struct Plane<zd> {
  using type = double;
};
template <>
struct Plane<zc> {
  using type = float;
};
template <typename T>
using plane_t = typename Plane<T>::type;

template <typename T>
__device__ __forceinline__ u4 load16(const T *p) {
  return reinterpret_cast<const U4 *>(p)->v;
}

// elements i .. i + EV - 1 of a line of len elements (len >= 1), zeros past its end;
// no element outside the line is read
template <typename T>
__device__ __forceinline__ u4 edge16(const T *line, int i, int len) {
  constexpr int EV = 16 / sizeof(T);
  const u4 zero = {0u, 0u, 0u, 0u};
  if constexpr (EV == 1) {
    const u4 v = load16(line + min(i, len - 1));
    return i < len ? v : zero;
  } else if (len >= EV) {
    const int at = min(i, len - EV), sh = i - at;  // sh elements of the vector precede i
    const u4 v = load16(line + at);
    u4 r;
    if constexpr (EV == 2) {
      r[0] = sh == 0 ? v[0] : sh == 1 ? v[2] : 0u;
      r[1] = sh == 0 ? v[1] : sh == 1 ? v[3] : 0u;
      r[2] = sh == 0 ? v[2] : 0u;
      r[3] = sh == 0 ? v[3] : 0u;
    } else {
      r[0] = sh == 0 ? v[0] : sh == 1 ? v[1] : sh == 2 ? v[2] : sh == 3 ? v[3] : 0u;
      r[1] = sh == 0 ? v[1] : sh == 1 ? v[2] : sh == 2 ? v[3] : 0u;
      r[2] = sh == 0 ? v[2] : sh == 1 ? v[3] : 0u;
      r[3] = sh == 0 ? v[3] : 0u;
    }
    return r;
  } else {  // a line shorter than a vector
    u4 r = zero;
    constexpr int W = sizeof(T) / 4;
#pragma unroll
    for (int e = 0; e < EV; ++e)
      if (i + e < len) {
        const unsigned *w = reinterpret_cast<const unsigned *>(line + i + e);
#pragma unroll
        for (int q = 0; q < W; ++q) r[e * W + q] = w[q];
      }
    return r;
  }
}

// A BM x BN tile of NT lanes over K slices of BK. LDS stage: A's planes (k-major, m
// contiguous), then B's (n-major, k contiguous), real and imaginary planes apart.
template <typename T, int BM_, int BN_, int BK_, int NT_>
struct Shape {
  using S = plane_t<T>;
  static constexpr int BM = BM_, BN = BN_, BK = BK_, NT = NT_;
  static constexpr int EV = 16 / sizeof(T);
  static constexpr int NP = is_cx<T> ? 2 : 1;
  // A row pitch: one k row of BM values; the 16 lanes of a k read 16 consecutive ones
  static constexpr int LDA = BM + (sizeof(S) == 8 ? 2 : 4);
  // B row pitch: 2 banks (mod 32) past a multiple of 32 banks, so the 16 rows one k step
  // reads fall on distinct bank pairs
  static constexpr int LDB = BK + (sizeof(S) == 8 ? 1 : 2);
  static constexpr int A_V = BM * BK / EV / NT, B_V = BN * BK / EV / NT;
  static constexpr int A_PLANE = BK * LDA, B_PLANE = BN * LDB;
  static constexpr int STAGE = NP * (A_PLANE + B_PLANE);
  static_assert(A_V >= 1 && B_V >= 1 && A_V * EV * NT == BM * BK && B_V * EV * NT == BN * BK,
                "a slice splits evenly over the lanes");
};

template <typename SH, typename T>
__device__ __forceinline__ void fetch(const GemmArgs<T> &g, bool full, int m0, int n0, int k0,
                                      int tid, u4 (&ra)[SH::A_V], u4 (&rb)[SH::B_V]) {
  constexpr int EV = SH::EV;
  if (full && k0 + SH::BK <= g.K) {
#pragma unroll
    for (int it = 0; it < SH::A_V; ++it) {
      const int idx = tid + it * SH::NT;
      const int m = (idx % (SH::BM / EV)) * EV, k = idx / (SH::BM / EV);
      ra[it] = load16(g.A + (m0 + m) + static_cast<long>(k0 + k) * g.lda);
    }
#pragma unroll
    for (int it = 0; it < SH::B_V; ++it) {
      const int idx = tid + it * SH::NT;
      const int k = (idx % (SH::BK / EV)) * EV, n = idx / (SH::BK / EV);
      rb[it] = load16(g.B + (k0 + k) + static_cast<long>(n0 + n) * g.ldb);
    }
  } else {
    const u4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int it = 0; it < SH::A_V; ++it) {
      const int idx = tid + it * SH::NT;
      const int m = (idx % (SH::BM / EV)) * EV, k = k0 + idx / (SH::BM / EV);
      const u4 v = edge16(g.A + static_cast<long>(min(k, g.K - 1)) * g.lda, m0 + m, g.M);
      ra[it] = k < g.K ? v : zero;
    }
#pragma unroll
    for (int it = 0; it < SH::B_V; ++it) {
      const int idx = tid + it * SH::NT;
      const int k = (idx % (SH::BK / EV)) * EV, n = n0 + idx / (SH::BK / EV);
      rb[it] = edge16(g.B + static_cast<long>(min(n, g.N - 1)) * g.ldb, k0 + k, g.K);
    }
  }
}

template <typename SH, typename T>
__device__ __forceinline__ void stage(plane_t<T> *L, int tid, const u4 (&ra)[SH::A_V],
                                      const u4 (&rb)[SH::B_V]) {
  using S = plane_t<T>;
  constexpr int EV = SH::EV;
  S *As = L, *Bs = L + SH::NP * SH::A_PLANE;
#pragma unroll
  for (int it = 0; it < SH::A_V; ++it) {
    const int idx = tid + it * SH::NT;
    const int m = (idx % (SH::BM / EV)) * EV, k = idx / (SH::BM / EV);
    S *at = As + k * SH::LDA + m;
    if constexpr (SH::NP == 1) {
      *reinterpret_cast<u4 *>(at) = ra[it];
    } else if constexpr (sizeof(S) == 8) {
      at[0] = __hiloint2double(ra[it][1], ra[it][0]);
      at[SH::A_PLANE] = __hiloint2double(ra[it][3], ra[it][2]);
    } else {
      *reinterpret_cast<uint2 *>(at) = make_uint2(ra[it][0], ra[it][2]);
      *reinterpret_cast<uint2 *>(at + SH::A_PLANE) = make_uint2(ra[it][1], ra[it][3]);
    }
  }
#pragma unroll
  for (int it = 0; it < SH::B_V; ++it) {
    const int idx = tid + it * SH::NT;
    const int k = (idx % (SH::BK / EV)) * EV, n = idx / (SH::BK / EV);
    S *at = Bs + n * SH::LDB + k;
    if constexpr (SH::NP == 1) {
      if constexpr (sizeof(S) == 8) {
        at[0] = __hiloint2double(rb[it][1], rb[it][0]);
        at[1] = __hiloint2double(rb[it][3], rb[it][2]);
      } else {
        reinterpret_cast<uint2 *>(at)[0] = make_uint2(rb[it][0], rb[it][1]);
        reinterpret_cast<uint2 *>(at)[1] = make_uint2(rb[it][2], rb[it][3]);
      }
    } else if constexpr (sizeof(S) == 8) {
      at[0] = __hiloint2double(rb[it][1], rb[it][0]);
      at[SH::B_PLANE] = __hiloint2double(rb[it][3], rb[it][2]);
    } else {
      *reinterpret_cast<uint2 *>(at) = make_uint2(rb[it][0], rb[it][2]);
      *reinterpret_cast<uint2 *>(at + SH::B_PLANE) = make_uint2(rb[it][1], rb[it][3]);
    }
  }
}

// the accumulators of a wave's TM x TN MFMA tiles
template <typename T, int TM, int TN>
struct Acc {
  typename Mfma<plane_t<T>>::acc re[TM][TN], im[is_cx<T> ? TM : 1][is_cx<T> ? TN : 1];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        re[i][j] = Mfma<plane_t<T>>::zero();
        if constexpr (is_cx<T>) im[i][j] = Mfma<plane_t<T>>::zero();
      }
  }
  __device__ __forceinline__ T at(int i, int j, int r) const {
    using S = plane_t<T>;
    if constexpr (is_cx<T>) return T{S(re[i][j][r]), S(im[i][j][r])};
    else return S(re[i][j][r]);
  }
};

// the products of the k steps [K0, K1) of a staged slice, k ascending
template <typename SH, typename T, int TM, int TN, int K0, int K1>
__device__ __forceinline__ void multiply(const plane_t<T> *L, int lane, int wm0, int wn0,
                                         Acc<T, TM, TN> &c) {
  using S = plane_t<T>;
  using M = Mfma<S>;
  const S *As = L + (lane >> 4) * SH::LDA + wm0 + (lane & 15);
  const S *Bs = L + SH::NP * SH::A_PLANE + (wn0 + (lane & 15)) * SH::LDB + (lane >> 4);
#pragma unroll
  for (int kk = K0; kk < K1; kk += 4) {
    S a[TM], b[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) a[i] = As[kk * SH::LDA + 16 * i];
#pragma unroll
    for (int j = 0; j < TN; ++j) b[j] = Bs[16 * j * SH::LDB + kk];
    if constexpr (!is_cx<T>) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) c.re[i][j] = M::mma(b[j], a[i], c.re[i][j]);
    } else {
      S ai[TM], nai[TM], bi[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        ai[i] = As[SH::A_PLANE + kk * SH::LDA + 16 * i];
        nai[i] = -ai[i];
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) bi[j] = Bs[SH::B_PLANE + 16 * j * SH::LDB + kk];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          c.re[i][j] = M::mma(b[j], a[i], c.re[i][j]);
          c.im[i][j] = M::mma(bi[j], a[i], c.im[i][j]);
          c.re[i][j] = M::mma(bi[j], nai[i], c.re[i][j]);
          c.im[i][j] = M::mma(b[j], ai[i], c.im[i][j]);
        }
    }
  }
}

// C's tile from the accumulators, epilogue_store's arithmetic in its order: a lane holds
// row lane % 16 of four columns of every MFMA tile. Every term's reads for a row of
// tiles are issued together. Rows below mlo and columns below nlo are a neighbour's.
template <typename T, int TM, int TN>
__device__ __forceinline__ void store_tile(const GemmArgs<T> &g, int lane, int m0, int n0,
                                           int mlo, int nlo, const Acc<T, TM, TN> &c) {
  using S = plane_t<T>;
  using O = ops<T>;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = m0 + 16 * i + (lane & 15);
    const bool rok = row >= mlo && row < g.M;
    T v[TN][4];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[j][r] = O::mul(g.alpha, c.at(i, j, r));
    auto each = [&](auto f) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int col = n0 + 16 * j + Mfma<S>::row(lane, r);
          f(j, r, col, rok && col >= nlo && col < g.N);
        }
    };
    if (g.Cin) {
      T x[TN][4];
      each([&](int j, int r, int col, bool ok) {
        if (ok) x[j][r] = g.Cin[row + static_cast<long>(col) * g.ldcin];
      });
      each([&](int j, int r, int, bool) { v[j][r] = O::add(v[j][r], O::mul(g.beta, x[j][r])); });
    }
    if (g.nterms > 0) {
      T e[TN][4];
      const T c0 = g.coef[0];
      each([&](int j, int r, int col, bool) { e[j][r] = row == col ? c0 : O::zero(); });
      for (int t = 1; t < g.nterms; ++t) {
        const T *X = t == 1 ? g.X1 : g.bank + static_cast<long>(t - 2) * g.bank_stride;
        const long ldx = t == 1 ? g.ldx1 : g.ldbank;
        const T ct = g.coef[t];
        T x[TN][4];
        each([&](int j, int r, int col, bool ok) {
          if (ok) x[j][r] = X[row + static_cast<long>(col) * ldx];
        });
        each([&](int j, int r, int, bool) { e[j][r] = O::mad(ct, x[j][r], e[j][r]); });
      }
      each([&](int j, int r, int, bool) { v[j][r] = O::add(v[j][r], e[j][r]); });
    }
    each([&](int j, int r, int col, bool ok) {
      if (ok) g.C[row + static_cast<long>(col) * g.ldc] = v[j][r];
    });
  }
}

// Tile (tm, tn) of the product; L holds two stages. The caller's LDS must be free
// on entry and is free after a barrier on return.
template <typename SH, typename T, int WM, int WN, int kAhead, int kMid = SH::BK / 2>
__device__ __forceinline__ void tile_product(const GemmArgs<T> &g, int tm, int tn,
                                             plane_t<T> *L) {
  constexpr int TM = WM / 16, TN = WN / 16, WAVES_M = SH::BM / WM;
  static_assert((SH::BM / WM) * (SH::BN / WN) == SH::NT / 64, "one wave a WM x WN sub-tile");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm0 = (wave % WAVES_M) * WM, wn0 = (wave / WAVES_M) * WN;
  const int mlo = tm * SH::BM, nlo = tn * SH::BN;
  const bool full = g.M >= SH::BM && g.N >= SH::BN;
  const int m0 = full ? min(mlo, g.M - SH::BM) : mlo, n0 = full ? min(nlo, g.N - SH::BN) : nlo;
  const int KT = (g.K + SH::BK - 1) / SH::BK;
  Acc<T, TM, TN> acc;
  acc.clear();
  u4 ra[kAhead][SH::A_V], rb[kAhead][SH::B_V];
#pragma unroll
  for (int d = 0; d < kAhead; ++d)
    if (d < KT) fetch<SH>(g, full, m0, n0, d * SH::BK, tid, ra[d], rb[d]);
  if (KT > 0) stage<SH, T>(L, tid, ra[0], rb[0]);
  // the slice kt + 1 is in register set (kt + 1) % kAhead; set kt % kAhead takes slice
  // kt + kAhead once slice kt is in LDS
  for (int kb = 0; kb < KT; kb += 2 * kAhead) {
#pragma unroll
    for (int u = 0; u < 2 * kAhead; ++u) {
      const int kt = kb + u;
      if (kt >= KT) break;
      if (kt + kAhead < KT)
        fetch<SH>(g, full, m0, n0, (kt + kAhead) * SH::BK, tid, ra[u % kAhead], rb[u % kAhead]);
      __syncthreads();
      // the next slice goes to its stage half-way through this one, so its LDS writes
      // overlap the other waves' MFMAs instead of holding up the barrier
      multiply<SH, T, TM, TN, 0, kMid>(L + (u & 1) * SH::STAGE, lane, wm0, wn0, acc);
      if (kt + 1 < KT)
        stage<SH, T>(L + ((u + 1) & 1) * SH::STAGE, tid, ra[(u + 1) % kAhead],
                     rb[(u + 1) % kAhead]);
      multiply<SH, T, TM, TN, kMid, SH::BK>(L + (u & 1) * SH::STAGE, lane, wm0, wn0, acc);
    }
  }
  store_tile<T, TM, TN>(g, lane, m0 + wm0, n0 + wn0, mlo, nlo, acc);
}

}  // namespace pipe
}  // namespace clm

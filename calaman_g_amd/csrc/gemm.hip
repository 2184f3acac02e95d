// gemm.hip -- matrix products on gfx950 MFMA for the four element types:
// FP64 and FP32 real, complex128 and complex64.
//
// C = alpha*A*B [+ beta*Cin] [+ B_blk], column-major NN, where B_blk is the
// Paterson-Stockmeyer block c0 I + c1 X1 + sum_t c_t bank[t-2] (or the Horner
// step's c I) formed in the epilogue. Fusing the block into the product's
// store is what removes the reference's separate build_block launch and its
// n^2 round trip through HBM before every Horner step
// (src/paterson_stockmeyer/interface.cppm:405-419 builds B_j, then runs the
// gemm with beta = 1 over it).
//
// Kernel shape:
//   * a tile of C per workgroup, cut into 16 x 16 MFMA tiles (v_mfma_f64_16x16x4_f64 /
//     v_mfma_f32_16x16x4_f32, 4 accumulator values per lane), one to four a wave;
//   * K advances in slices, double-buffered in LDS: later slices are fetched global ->
//     VGPR while the current one is multiplied, then written to the other LDS stage;
//     one barrier per slice;
//   * A is staged as As[k][m] (m contiguous, as it arrives from column-major
//     memory), B as Bs[n][k] at a pitch of 2 banks (mod 32), so the 16 lanes that read
//     one k of B hit distinct banks;
//   * workgroups are renumbered so each of the 8 XCDs (dispatched round robin
//     on the workgroup id) owns a contiguous run of tiles, walked in groups of
//     4 tile-rows: the A panels an XCD touches stay in its own L2;
//   * the tile is chosen per product (launch_product) so that the tiles fill the CUs.
//
// MFMA operand layout (16x16x4): A lane l holds A[l%16][l/16], B lane l holds
// B[l/16][l%16]; D lane l holds column l%16 at rows l/16 + 4r for the FP64
// instruction and rows 4(l/16) + r for the FP32 one (r = 0..3). The FP64 MFMA
// accumulates the four k terms of a step in order, as a sequential FMA chain.
#include "gemm_pipe.hpp"
#include "gemm_tile.hpp"

namespace clm {
namespace {

using namespace tile;

// Real products of whole 128 x 128 tiles and whole slices at 16-byte aligned columns.
template <typename S, int BM, int BN, int WM, int WN, int NT, int BK>
__global__ void __launch_bounds__(NT)
    rgemm_mfma(const GemmArgs<S> g, const int tiles_m, const int tiles_n) {
  using TL = RTile<S, BM, BN, NT, BK>;
  using V = typename Mfma<S>::vec;
  constexpr int WAVES_M = BM / WM;
  static_assert((BM / WM) * (BN / WN) == NT / 64, "one wave per WM x WN sub-tile");
  constexpr int TM = WM / 16, TN = WN / 16;

  __shared__ __attribute__((aligned(16))) S L[2 * (TL::A_STAGE + TL::B_STAGE)];
  S *As = L;
  S *Bs = L + 2 * TL::A_STAGE;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int wm0 = (wave % WAVES_M) * WM;
  const int wn0 = (wave / WAVES_M) * WN;

  typename Mfma<S>::acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = Mfma<S>::zero();

  V ra[TL::A_V], rb[TL::B_V];
  const int KT = (g.K + BK - 1) / BK;
  if (KT > 0) {
    rgemm_gload<S, BM, BN, NT, BK, true>(g, m0, n0, 0, tid, ra, rb);
    rgemm_sstore<S, BM, BN, NT, BK>(As, Bs, tid, ra, rb);
    __syncthreads();
    for (int kt = 0; kt < KT - 1; ++kt) {
      const int cur = kt & 1;
      rgemm_gload<S, BM, BN, NT, BK, true>(g, m0, n0, (kt + 1) * BK, tid, ra, rb);
      // the next slice goes into the other stage half-way through this one, so its
      // LDS writes overlap the other waves' MFMAs instead of idling the CU before
      // the barrier (the k-steps still run in ascending order)
      rgemm_compute<S, BM, BN, WM, WN, NT, BK, 0, BK / 2>(As + cur * TL::A_STAGE,
                                                         Bs + cur * TL::B_STAGE, lane, wm0, wn0, acc);
      rgemm_sstore<S, BM, BN, NT, BK>(As + (cur ^ 1) * TL::A_STAGE, Bs + (cur ^ 1) * TL::B_STAGE,
                                      tid, ra, rb);
      rgemm_compute<S, BM, BN, WM, WN, NT, BK, BK / 2, BK>(As + cur * TL::A_STAGE,
                                                          Bs + cur * TL::B_STAGE, lane, wm0, wn0, acc);
      __syncthreads();
    }
    const int last = (KT - 1) & 1;
    rgemm_compute<S, BM, BN, WM, WN, NT, BK>(As + last * TL::A_STAGE, Bs + last * TL::B_STAGE,
                                             lane, wm0, wn0, acc);
  }

  // the sums go column-major into the free LDS stages and the whole workgroup writes
  // them out in coalesced column pieces
  constexpr int LDT = 128 + 16 / sizeof(S);
  static_assert(BM == 128 && BN == 128 && 128 * LDT <= 2 * (TL::A_STAGE + TL::B_STAGE),
                "the tile fits the stages");
  __syncthreads();  // every wave is done with the stages
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        L[(wn0 + j * 16 + (lane & 15)) * LDT + wm0 + i * 16 + Mfma<S>::row(lane, r)] =
            S(acc[i][j][r]);
  __syncthreads();
  lds_tile_epilogue<S, NT / 64, true>(g, m0, n0, [&](int c, int r) { return L[c * LDT + r]; });
}

// One workgroup tile per workgroup, the operands fetched ahead (gemm_pipe.hpp).
template <typename T, int BM, int BN, int BK, int WM, int WN, int kAhead>
__global__ void __launch_bounds__((BM / WM) * (BN / WN) * 64)
    gemm_piped(const GemmArgs<T> g, const int tiles_m, const int tiles_n) {
  using SH = pipe::Shape<T, BM, BN, BK, (BM / WM) * (BN / WN) * 64>;
  __shared__ __attribute__((aligned(16))) pipe::plane_t<T> L[2 * SH::STAGE];
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  pipe::tile_product<SH, T, WM, WN, kAhead>(g, tm, tn, L);
}

template <typename T, int BM, int BN, int BK, int WM, int WN, int kAhead>
hipError_t launch_piped(hipStream_t stream, const GemmArgs<T> &g) {
  const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
  hipLaunchKernelGGL((gemm_piped<T, BM, BN, BK, WM, WN, kAhead>), dim3(tiles_m * tiles_n),
                     dim3((BM / WM) * (BN / WN) * 64), 0, stream, g, tiles_m, tiles_n);
  return hipGetLastError();
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

constexpr int kCus = 256;

// The workgroup tile of a product: 32 x 32 (4 waves of one MFMA tile), 64 x 64 (16 such
// waves, or 4 of 2 x 2) or the large tile (16 waves of 2 x 2 or 2 x 1 MFMA tiles). All three run the
// same k order, so the choice is speed only: the estimate is the rounds of tiles the
// 256 CUs take, times the measured time of one tile and k (ns, beyond the launch).
// A lone 32 x 32 tile per CU has one wave per SIMD and waits on its loads (`one`).
//
// Measured per product, before (64 x 64 tiles of 4 waves, one slice ahead, no vector
// loads at odd orders; 128 x 128 at n >= 2048) -> now, with a four-term block, us:
//   n       FP64           FP32           complex64      complex128
//   64      13.3 -> 4.3    11.7 -> 3.5    16.7 -> 5.3    20.4 -> 6.3
//   333     28.5 -> 9.7    24.0 -> 7.4    41.3 -> 14.0   61.8 -> 20.8
//   501     38.4 -> 12.8   32.5 -> 9.3    57.8 -> 19.3   95.1 -> 29.3
//   1000    73.8 -> 42.7   63.7 -> 26.0   104.9 -> 77.0  168.6 -> 134.5
//   1500    199 -> 153     158 -> 86      427 -> 258     826 -> 503
//   2000    306 -> 277     199 -> 157     570 -> 513     1104 -> 996
struct TileCost {
  int bm, bn;
  double one, more;
};
template <typename T>
constexpr TileCost kSmall{32, 32, 18.4, 10.8};
template <>
constexpr TileCost kSmall<float>{32, 32, 11.0, 6.2};
template <>
constexpr TileCost kSmall<zc>{32, 32, 31.0, 18.7};
template <>
constexpr TileCost kSmall<zd>{32, 32, 50.0, 36.8};
template <typename T>
constexpr TileCost kMedium{64, 64, 38.0, 38.0};
template <>
constexpr TileCost kMedium<float>{64, 64, 22.0, 22.0};
template <>
constexpr TileCost kMedium<zc>{64, 64, 73.0, 73.0};
template <>
constexpr TileCost kMedium<zd>{64, 64, 128.0, 128.0};
template <typename T>
constexpr TileCost kLarge{128, 128, 138.0, 138.0};
template <>
constexpr TileCost kLarge<float>{128, 128, 73.0, 73.0};
template <>
constexpr TileCost kLarge<zc>{128, 128, 268.0, 268.0};
template <>
constexpr TileCost kLarge<zd>{128, 64, 243.0, 243.0};

inline long tiles_of(const TileCost &t, int m, int n) {
  return static_cast<long>((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn);
}
inline double estimate(const TileCost &t, int m, int n) {
  const long rounds = (tiles_of(t, m, n) + kCus - 1) / kCus;
  return rounds == 1 ? t.one : static_cast<double>(rounds) * t.more;
}

template <typename T>
hipError_t launch_large(hipStream_t stream, const GemmArgs<T> &g) {
  if constexpr (std::is_same_v<T, zd>) {
    // 16 waves of 32 x 16 over slices of 16: 1044 -> 997 us at n = 2048 against 8 waves
    // of 32 x 32 (twice the waves over the same LDS)
    return launch_piped<T, 128, 64, 16, 32, 16, 1>(stream, g);
  } else {
    if constexpr (!std::is_same_v<T, zc>) {
      // real, whole tiles and slices at 16-byte aligned columns: no bounds anywhere and
      // 16-byte column pieces out of LDS, at n = 2048 FP64 280 against 285 us, at n = 4096
      // FP32 1063 against 1097 us, FP32 8192 x 8192 x 64 116 against 122 us
      constexpr int EV = 16 / sizeof(T);
      const bool fast = g.M % 128 == 0 && g.N % 128 == 0 && g.K % 32 == 0 && g.lda % EV == 0 &&
                        g.ldb % EV == 0 && aligned16(g.A) && aligned16(g.B);
      if (fast) {
        const int tiles_m = g.M / 128, tiles_n = g.N / 128;
        hipLaunchKernelGGL((rgemm_mfma<T, 128, 128, 32, 32, 1024, 32>), dim3(tiles_m * tiles_n),
                           dim3(1024), 0, stream, g, tiles_m, tiles_n);
        return hipGetLastError();
      }
    }
    return launch_piped<T, 128, 128, 32, 32, 32, 1>(stream, g);
  }
}

template <typename T>
hipError_t launch_product(hipStream_t stream, const GemmArgs<T> &g) {
  if (g.M <= 0 || g.N <= 0) return hipSuccess;
  const double s = estimate(kSmall<T>, g.M, g.N), m = estimate(kMedium<T>, g.M, g.N),
               l = estimate(kLarge<T>, g.M, g.N);
  if (l <= m && l <= s) return launch_large<T>(stream, g);
  if (m <= s) {
    constexpr int BK = std::is_same_v<T, float> ? 64 : 32;  // a vector a lane and slice
    if constexpr (std::is_same_v<T, float>) {
      // FP32 past two tiles a CU: 4 waves of 2 x 2 MFMA tiles, eight workgroups a CU, which
      // need no whole rounds (n = 1664 102 -> 98 us, 1728 107 -> 101, 1650 104 -> 98); up to
      // two, twice the waves of a tile hide more (n = 1024 25 us against 33)
      if (tiles_of(kMedium<T>, g.M, g.N) > 2 * kCus)
        return launch_piped<T, 64, 64, 16, 32, 32, 1>(stream, g);
    }
    return launch_piped<T, 64, 64, BK, 16, 16, 1>(stream, g);
  }
  return launch_piped<T, 32, 32, 32, 16, 16, 2>(stream, g);
}

}  // namespace

hipError_t launch_gemm_d(hipStream_t stream, const GemmArgs<double> &g) {
  return launch_product<double>(stream, g);
}
hipError_t launch_gemm_z(hipStream_t stream, const GemmArgs<zd> &g) {
  return launch_product<zd>(stream, g);
}

template <>
hipError_t launch_gemm<double>(hipStream_t stream, const GemmArgs<double> &g) {
  return launch_product<double>(stream, g);
}
template <>
hipError_t launch_gemm<float>(hipStream_t stream, const GemmArgs<float> &g) {
  return launch_product<float>(stream, g);
}
template <>
hipError_t launch_gemm<zd>(hipStream_t stream, const GemmArgs<zd> &g) {
  return launch_product<zd>(stream, g);
}
template <>
hipError_t launch_gemm<zc>(hipStream_t stream, const GemmArgs<zc> &g) {
  return launch_product<zc>(stream, g);
}

}  // namespace clm

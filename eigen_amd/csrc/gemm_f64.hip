// gemm_f64.hip -- FP64 GEMM / SYRK on CDNA4 matrix cores.
//
// C = alpha * op(A) * op(B) + beta * C, column-major with leading dimensions.
// This is the MI355X replacement for general_matrix_matrix_product::run
// (Eigen/src/Core/products/GeneralMatrixMatrix.h:49-199) and, with the
// lower-triangle filter, for general_matrix_matrix_triangular_product
// (GeneralMatrixMatrixTriangular.h:56-125).
//
// Design: C tiles of 128x128, 64x64 or 32x32 per 256-thread workgroup (four
// waves in 2x2, each a quarter of the tile in 16x16 blocks of
// v_mfma_f64_16x16x4f64), K staged through LDS in double-buffered slabs, and a
// 16x16 kernel that splits K over sixteen waves for the smallest outputs; the
// tile is picked by the output's size (pick_tile).  The MFMA is fed the
// transposed product (op(B)^T op(A)^T) so that each lane's four accumulator
// rows map to four *columns* of C and the sixteen lanes of a row group cover
// sixteen consecutive rows: the epilogue writes 128-byte runs of a column.
// Workgroups are remapped so that consecutive tiles share an XCD (the
// dispatcher deals workgroups round-robin over the 8 XCDs, each with its own
// L2) and swizzled in groups of 8 tile-rows for L2 reuse of B.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace eamd {

namespace {

// A square tile of TS x TS per workgroup.  128: eight waves of 64 x 32 in at
// most 128 registers, so two workgroups put four waves on a SIMD and one
// wave's C traffic, slab hand-over or LDS latency is another's MFMA time.
// 64 and 32: four waves in 2 x 2, for outputs that leave CUs with one
// workgroup; the K slab grows as the tile shrinks and the loads run two slabs
// ahead, since the MFMA time of one slab no longer covers a memory round trip.
template <int TS>
struct Tile {
  static constexpr int BK = TS == 128 ? 16 : (TS == 64 ? 32 : 64);
  static constexpr int LD = TS + 2;          // row length of the LDS slabs (doubles)
  static constexpr int WN = TS >= 64 ? 4 : 2;  // waves along n (two along m)
  static constexpr int NT = 128 * WN;        // threads
  static constexpr int TI = TS / 32;         // 16x16 blocks per wave along m
  static constexpr int TJ = TS / 16 / WN;    // and along n
  static constexpr int CH = BK * TS / (2 * NT);  // 16-byte words per thread and operand
  static constexpr int AHEAD = TS == 128 ? 1 : 2;  // slabs loaded ahead
};
typedef double v2d __attribute__((ext_vector_type(2)));
// a pair of doubles at any 8-byte address (global memory takes 16-byte loads
// at 4-byte alignment)
typedef double v2du __attribute__((ext_vector_type(2), aligned(8)));

__device__ __forceinline__ void tile_coords(int bid, int nblocks, int tiles_m, int tiles_n,
                                            int& tm, int& tn) {
  // XCD-aware remap: workgroup bid runs on XCD bid % 8.
  int xcd = bid & 7, loc = bid >> 3;
  int per = nblocks >> 3, rem = nblocks & 7;
  int logical = (xcd < rem) ? xcd * (per + 1) + loc : rem * (per + 1) + (xcd - rem) * per + loc;
  const int G = 8;
  int group = G * tiles_n;
  int g = logical / group;
  int first_m = g * G;
  int gm = min(tiles_m - first_m, G);
  int r = logical - g * group;
  tm = first_m + r % gm;
  tn = r / gm;
}

// Tile `idx` of the lower trapezoid {(tr, tc): tc <= tr < tr_n, tc < tc_n} of
// a tr_n x tc_n tile grid, row by row: the triangle tr < T = min(tr_n, tc_n)
// first, then full rows of tc_n tiles.
__device__ __forceinline__ void tri_tile(int idx, int tr_n, int tc_n, int& tr, int& tc) {
  const int T = min(tr_n, tc_n), tri = T * (T + 1) / 2;
  if (idx < tri) {
    int r = (int)((sqrt(8.0 * idx + 1.0) - 1.0) * 0.5);
    if ((r + 1) * (r + 2) / 2 <= idx) ++r;
    if (r * (r + 1) / 2 > idx) --r;
    tr = r;
    tc = idx - r * (r + 1) / 2;
  } else {
    const int q = idx - tri;
    tr = T + q / tc_n;
    tc = q - (q / tc_n) * tc_n;
  }
}

// Number of tiles of that trapezoid.
inline int tri_tiles(int tr_n, int tc_n) {
  const int T = std::min(tr_n, tc_n);
  return T * (T + 1) / 2 + (tr_n > T ? (tr_n - T) * tc_n : 0);
}

// One operand slab (rows of the tile x BK of K), memory to registers to LDS
// (S[k * LD + row]).  KCONT: K is the contiguous direction in memory.  A
// thread takes pairs along the contiguous direction, consecutive threads
// consecutive pairs, so a wave's load is whole cache lines (eight scattered
// words per thread kept the L1 as busy as the matrix cores).  Rows past the
// operand's last one read that row again (their products are not stored).
constexpr int kCus = 256;
constexpr int64_t kMaxPairLd = 1 << 21;  // 8 TS ld fits 32 bits
template <int TS, bool KCONT>
struct Slab {
  using Tl = Tile<TS>;
  static constexpr int CH = Tl::CH, BK = Tl::BK, LD = Tl::LD;
  const char* base;     // the next whole slab (wave-uniform)
  unsigned off[KCONT ? CH : 1];  // the thread's pairs in it, in bytes (ld <= kMaxPairLd;
  int64_t step, qstep;           // not KCONT: pair q is q * qstep further)
  bool odd;             // (not KCONT) the pair starts at the operand's last row
  v2d v[Tl::AHEAD][CH];
  static __device__ __forceinline__ void coord(int q, int& row, int& k) {
    const int c = threadIdx.x + Tl::NT * q;
    if (KCONT) {
      row = c / (BK / 2);
      k = (c % (BK / 2)) * 2;
    } else {
      k = c / (TS / 2);
      row = (c % (TS / 2)) * 2;
    }
  }
  __device__ __forceinline__ void init(const double* __restrict__ P, int64_t ld, int r0,
                                       int rows) {
    step = 8 * (KCONT ? BK : (int64_t)BK * ld);
    base = reinterpret_cast<const char*>(KCONT ? P + (int64_t)r0 * ld : P + r0);
    odd = false;
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      int rr, kk;
      coord(q, rr, kk);
      if (KCONT) {
        off[q] = 8u * ((unsigned)min(rr, rows - 1 - r0) * (unsigned)ld + (unsigned)kk);
      } else {
        // a tile whose only row is the operand's last starts a row earlier
        const int back = rows - 1 == r0 ? 1 : 0;
        if (q > 0) continue;
        base -= 8 * back;
        qstep = 8 * (int64_t)(Tl::NT / (TS / 2)) * ld;
        off[0] = 8u * ((unsigned)kk * (unsigned)ld +
                       (unsigned)max(0, min(rr, rows - 2 - r0)));
        odd = r0 + rr == rows - 1;  // the same for every q: NT is a multiple of TS / 2
      }
    }
  }
  // the next slab, all of it inside K (not KCONT: the operand has 2 rows)
  __device__ __forceinline__ void load(int st) {
#pragma unroll
    for (int q = 0; q < CH; ++q)
      v[st][q] = *reinterpret_cast<const v2du*>(KCONT ? base + off[q]
                                                      : base + q * qstep + off[0]);
    base += step;
  }
  // slab at k0 of an operand with k values of K; those past it are zero
  __device__ __forceinline__ void load_tail(const double* __restrict__ P, int64_t ld, int r0,
                                            int rows, int k0, int k, int st) {
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      int rr, kk;
      coord(q, rr, kk);
      const int gk = k0 + kk, ka = min(gk, k - 1), kb = KCONT ? min(gk + 1, k - 1) : ka;
      const int ga = min(r0 + rr, rows - 1), gb = KCONT ? ga : min(r0 + rr + 1, rows - 1);
      const double x = KCONT ? P[(int64_t)ga * ld + ka] : P[(int64_t)ka * ld + ga];
      // (a pair at the last row holds that row twice, as `odd` expects)
      const double y = KCONT ? P[(int64_t)gb * ld + kb] : P[(int64_t)kb * ld + gb];
      v[st][q].x = gk < k ? x : 0.0;
      v[st][q].y = (KCONT ? gk + 1 : gk) < k ? y : 0.0;
    }
  }
  __device__ __forceinline__ void store(double* S, int st) const {
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      int rr, kk;
      coord(q, rr, kk);
      if (KCONT) {
        S[kk * LD + rr] = v[st][q].x;
        S[(kk + 1) * LD + rr] = v[st][q].y;
      } else {
        *reinterpret_cast<v2d*>(&S[kk * LD + rr]) = v2d{odd ? v[st][q].y : v[st][q].x, v[st][q].y};
      }
    }
  }
};

// The products of one BK slab, staged in as / bs, into the wave's blocks.
// Small tiles (one or two waves per SIMD) read a step's operands from LDS
// while the step before it multiplies.
template <int TS>
__device__ __forceinline__ void slab_products(const double* as, const double* bs, int wm, int wn,
                                              int l16, int lk,
                                              v4d (&acc)[Tile<TS>::TI][Tile<TS>::TJ]) {
  constexpr int TI = Tile<TS>::TI, TJ = Tile<TS>::TJ, LD = Tile<TS>::LD;
  constexpr int KS = Tile<TS>::BK / 4, NB = TS == 128 ? 1 : 2;
  double af[NB][TI], bf[NB][TJ];
  const double* ap = as + lk * LD + wm + l16;
  const double* bp = bs + lk * LD + wn + l16;
  auto frag = [&](int kk, int buf) {
#pragma unroll
    for (int i = 0; i < TI; ++i) af[buf][i] = ap[kk * 4 * LD + i * 16];
#pragma unroll
    for (int j = 0; j < TJ; ++j) bf[buf][j] = bp[kk * 4 * LD + j * 16];
  };
  frag(0, 0);
#pragma unroll
  for (int kk = 0; kk < KS; ++kk) {
    if (NB == 2 && kk + 1 < KS) frag(kk + 1, (kk + 1) & 1);
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf[kk % NB][j], af[kk % NB][i],
                                                         acc[i][j], 0, 0, 0);
    if (NB == 1 && kk + 1 < KS) frag(kk + 1, 0);
    if (NB == 2) {
      __builtin_amdgcn_sched_group_barrier(0x100, TI + TJ, 0);  // DS reads
      __builtin_amdgcn_sched_group_barrier(0x008, TI * TJ, 0);  // MFMA
    }
  }
}

// MODE 0: full C.  MODE 1: lower triangle only (i >= j), tiles strictly above
// the diagonal are skipped.  MODE 2: upper triangle only (i <= j).
// CIN (128-wide tiles): beta == 1, alpha == +-1 and at least eight whole slabs
// of K and no partial one (the trailing updates of the blocked
// factorizations): the C tile is read in eight parts of eight words per lane,
// one part beside each of the first eight slabs' operand loads and added into
// the accumulators one slab later; the epilogue of a
// whole tile then only stores alpha * acc (alpha^2 = 1, both scalings exact).  Loading the
// whole tile before the first slab made every workgroup of a launch wait for
// 128 KB of C at once (LLT n = 8192: 13.35 -> 12.18 ms; FP64 LU n = 16384:
// 195 -> 178 ms).  Part p holds blocks (i, j) = (p / 2, 2 (p % 2) + {0, 1}).
// Smaller tiles read their C (16 or 4 words per lane) before the first slab.
template <int TS, bool TA, bool TB, int MODE, bool CIN>
__global__ __launch_bounds__(Tile<TS>::NT, TS == 128 ? 4 : 2) void dgemm_kernel(int m, int n, int k, double alpha,
                                                    const double* __restrict__ A, int64_t lda,
                                                    const double* __restrict__ B, int64_t ldb,
                                                    double beta, double* __restrict__ C,
                                                    int64_t ldc, const int* __restrict__ abort_flag) {
  using Tl = Tile<TS>;
  constexpr int BK = Tl::BK, LD = Tl::LD, TI = Tl::TI, TJ = Tl::TJ;
  using SA = Slab<TS, TA>;
  using SB = Slab<TS, !TB>;
  __shared__ __align__(16) double As[2][BK * LD];
  __shared__ __align__(16) double Bs[2][BK * LD];
  if (abort_flag && *abort_flag >= 0) return;

  const int tiles_m = (m + TS - 1) / TS, tiles_n = (n + TS - 1) / TS;
  int tm, tn;
  if (MODE == 0) {
    tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
  } else {
    // the grid holds only the tiles that meet the triangle; each XCD takes
    // a contiguous run of them (equal shares of the work)
    const int bid = blockIdx.x, nblocks = gridDim.x;
    const int xcd = bid & 7, loc = bid >> 3, per = nblocks >> 3, rem = nblocks & 7;
    const int logical =
        (xcd < rem) ? xcd * (per + 1) + loc : rem * (per + 1) + (xcd - rem) * per + loc;
    if (MODE == 1) tri_tile(logical, tiles_m, tiles_n, tm, tn);
    else tri_tile(logical, tiles_n, tiles_m, tn, tm);
  }
  const int m0 = tm * TS, n0 = tn * TS;

  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wm = (wave & 1) * (TS / 2), wn = (wave >> 1) * (TS / Tl::WN);
  int lane = threadIdx.x & 63;
  int l16 = lane & 15, lk = lane >> 4;

  const bool inner = m0 + TS <= m && n0 + TS <= n;

  v4d acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  const int ktiles = (k + BK - 1) / BK;
  // whole slabs, loaded through running pointers; the rest (a partial last
  // slab, or every slab of a one-row operand) with checks
  const bool pairs =
      (TA || m >= 2) && (!TB || n >= 2) && lda <= kMaxPairLd && ldb <= kMaxPairLd;
  const int kfull = CIN ? ktiles : (pairs ? k / BK : 0);
  SA sa;
  SB sb;
  sa.init(A, lda, m0, m);
  sb.init(B, ldb, n0, n);
  constexpr int AHEAD = Tl::AHEAD;
  // slab kt into register set st
  auto load = [&](int st) {
    sa.load(st);
    sb.load(st);
  };
  auto any = [&](int kt, int st) {
    if (kt < kfull) {
      load(st);
    } else if (kt < ktiles) {
      sa.load_tail(A, lda, m0, m, kt * BK, k, st);
      sb.load_tail(B, ldb, n0, n, kt * BK, k, st);
    }
  };
  auto store = [&](int buf, int st) {
    sa.store(As[buf], st);
    sb.store(Bs[buf], st);
  };
  any(0, 0);
  if constexpr (AHEAD == 2) any(1, 1);
  // the small tiles' C (beta != 0), requested beside the first slab
  constexpr bool kPre = TS < 128;
  double cpre[kPre ? TI : 1][kPre ? TJ : 1][4];
  if constexpr (kPre) {
    if (beta != 0.0) {
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int gi = min(m0 + wm + i * 16 + l16, m - 1);
            const int gj = min(n0 + wn + j * 16 + lk + 4 * r, n - 1);
            cpre[i][j][r] = C[(int64_t)gj * ldc + gi];
          }
    }
  }
  store(0, 0);
  __syncthreads();
  int kt = 0;
  if constexpr (CIN) {
    double cb[4];
    const char* cbase = reinterpret_cast<const char*>(C + (int64_t)(n0 + wn) * ldc + (m0 + wm));
    const unsigned coff = 8u * ((unsigned)lk * (unsigned)ldc + (unsigned)l16);
    auto cload = [&](auto P) {
      constexpr int p = decltype(P)::value, i = p / TJ, j = p % TJ;
      if (!inner) return;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        cb[r] = *reinterpret_cast<const double*>(
            cbase + 8 * ((int64_t)(j * 16 + 4 * r) * ldc + i * 16) + coff);
    };
    auto cadd = [&](auto P) {
      constexpr int p = decltype(P)::value, i = p / TJ, j = p % TJ;
      if (!inner) return;
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] += alpha * cb[r];
    };
    // slab p with C part p
    auto step = [&](auto P) {
      constexpr int p = decltype(P)::value;
      if (p < 7 || ktiles > 8) load(0);
      if constexpr (p > 0) cadd(std::integral_constant<int, p - 1>{});
      cload(P);
      __builtin_amdgcn_sched_barrier(0);
      slab_products<TS>(As[p & 1], Bs[p & 1], wm, wn, l16, lk, acc);
      __builtin_amdgcn_sched_barrier(0);
      if (p < 7 || ktiles > 8) store((p + 1) & 1, 0);
      __syncthreads();
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
    step(std::integral_constant<int, 4>{});
    step(std::integral_constant<int, 5>{});
    step(std::integral_constant<int, 6>{});
    step(std::integral_constant<int, 7>{});
    cadd(std::integral_constant<int, 7>{});
    kt = 8;
  }
  // slab kt from LDS buffer kt % 2; the register set it was loaded in is
  // free for slab kt + AHEAD, whose turn to be stored comes AHEAD - 1 slabs on
  auto slab = [&](auto L, int st) {
    constexpr bool kLoad = decltype(L)::value;
    if (kLoad) load(st);
    else any(kt + AHEAD, st);
    __builtin_amdgcn_sched_barrier(0);
    slab_products<TS>(As[kt & 1], Bs[kt & 1], wm, wn, l16, lk, acc);
    __builtin_amdgcn_sched_barrier(0);
    if (kLoad || kt + 1 < ktiles) store((kt + 1) & 1, AHEAD == 2 ? st ^ 1 : 0);
    __syncthreads();
    ++kt;
  };
  if constexpr (AHEAD == 2) {
    while (kt + 3 < kfull) {
      slab(std::true_type{}, 0);
      slab(std::true_type{}, 1);
    }
    while (kt < ktiles) {
      slab(std::false_type{}, 0);
      if (kt < ktiles) slab(std::false_type{}, 1);
    }
  } else {
    while (kt + 1 < kfull) slab(std::true_type{}, 0);
    if constexpr (CIN) {
      if (kt < ktiles) slab_products<TS>(As[kt & 1], Bs[kt & 1], wm, wn, l16, lk, acc);
    } else {
      while (kt < ktiles) slab(std::false_type{}, 0);
    }
  }

  // the lane's coordinates again, from an opaque copy: nothing of the
  // epilogue's addressing stays in registers through the K loop
  lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  l16 = lane & 15;
  lk = lane >> 4;
  // epilogue of a whole tile: plain stores, and C (where beta asks for it and
  // it is not in the accumulators or in cpre yet) read sixteen values at a
  // time; one read per value before its store is a chain of memory round
  // trips (8192 x 5000, K = 30: 185 us, and 147 with the reads together; 8192
  // x 8192, K = 64: 347 and 289)
  const bool offdiag = MODE == 0 || (MODE == 1 ? tm > tn : tn > tm);
  if (inner && offdiag && (CIN || !kPre || beta == 0.0) && ldc <= kMaxPairLd) {
    char* cbase = reinterpret_cast<char*>(C + (int64_t)(n0 + wn) * ldc + (m0 + wm));
    const unsigned coff = 8u * ((unsigned)lk * (unsigned)ldc + (unsigned)l16);
    const bool addc = !CIN && beta != 0.0;
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      double cin[4][TI];
      if (addc) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int i = 0; i < TI; ++i)
            cin[r][i] = *reinterpret_cast<const double*>(
                cbase + 8 * (int64_t)(j * 16 + 4 * r) * ldc + 128 * i + coff);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        char* cj = cbase + 8 * (int64_t)(j * 16 + 4 * r) * ldc;
#pragma unroll
        for (int i = 0; i < TI; ++i) {
          double v = alpha * acc[i][j][r];
          if (addc) v += beta * cin[r][i];
          *reinterpret_cast<double*>(cj + 128 * i + coff) = v;
        }
      }
    }
    return;
  }

  // epilogue: v_mfma_f64_16x16x4f64 leaves result row lk + 4r of the 16x16
  // tile in register r of lane (lk, l16): acc[i][j][r] = C(m0+wm+16i+l16,
  // n0+wn+16j+lk+4r)
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    const int gi = m0 + wm + i * 16 + l16;
    if (gi >= m) continue;
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gj = n0 + wn + j * 16 + lk + 4 * r;
        if (gj >= n) continue;
        if (MODE == 1 && gi < gj) continue;
        if (MODE == 2 && gi > gj) continue;
        double* c = C + (int64_t)gj * ldc + gi;
        double v = alpha * acc[i][j][r];
        if (!(CIN && inner) && beta != 0.0) {
          if constexpr (kPre) v += beta * cpre[i][j][r];
          else v += beta * *c;
        }
        *c = v;
      }
  }
}

// One 16x16 tile of C per workgroup of sixteen waves, each wave a sixteenth of
// K (in runs of 16) with its operand fragments read straight from memory: the
// smallest outputs, where larger tiles would leave the chip idle and a single
// wave's K loop would be the whole time (96 x 80 x 64: 17.6 us with one
// 128x128 tile).  In a run of 16, lane group lk takes k = 4 lk .. 4 lk + 3 of
// both operands: 32 contiguous bytes where K is the contiguous direction,
// 128-byte runs of rows where it is not.  The waves' partial tiles are summed
// through LDS in wave order.
constexpr int kThinWaves = 16;
template <bool TA, bool TB>
__global__ __launch_bounds__(64 * kThinWaves) void dgemm_thin_kernel(
    int m, int n, int k, double alpha, const double* __restrict__ A, int64_t lda,
    const double* __restrict__ B, int64_t ldb, double beta, double* __restrict__ C, int64_t ldc,
    const int* __restrict__ abort_flag) {
  __shared__ double red[kThinWaves][256];
  if (abort_flag && *abort_flag >= 0) return;
  const int tiles_m = (m + 15) / 16;
  const int tm = blockIdx.x % tiles_m, tn = blockIdx.x / tiles_m;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, lk = lane >> 4;
  // rows past the edge read the last row (their results are not stored)
  const int ar = min(tm * 16 + l16, m - 1), br = min(tn * 16 + l16, n - 1);
  const int runs = (k + 15) / 16, per = (runs + kThinWaves - 1) / kThinWaves;
  const int r1 = min(runs, (wave + 1) * per);
  // this thread's element of C, requested up front (waves 0..3)
  const int e = threadIdx.x & 255, ci = tm * 16 + (e & 15), cj = tn * 16 + (e >> 4);
  const bool mine = threadIdx.x < 256 && ci < m && cj < n;
  const double c0 = (mine && beta != 0.0) ? C[(int64_t)cj * ldc + ci] : 0.0;
  v4d acc = {0.0, 0.0, 0.0, 0.0};
  const double* ap = TA ? A + (int64_t)ar * lda + lk * 4 : A + (int64_t)(lk * 4) * lda + ar;
  const double* bp = TB ? B + (int64_t)(lk * 4) * ldb + br : B + (int64_t)br * ldb + lk * 4;
  // a whole run's operands: two 16-byte words, or four values of a row each
  auto load = [&](int r, double (&av)[4], double (&bv)[4]) {
    const int64_t kb = (int64_t)r * 16;
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      if constexpr (TA) {
        const v2d t = *reinterpret_cast<const v2du*>(ap + kb + j);
        av[j] = t.x;
        av[j + 1] = t.y;
      } else {
        av[j] = ap[(kb + j) * lda];
        av[j + 1] = ap[(kb + j + 1) * lda];
      }
      if constexpr (!TB) {
        const v2d t = *reinterpret_cast<const v2du*>(bp + kb + j);
        bv[j] = t.x;
        bv[j + 1] = t.y;
      } else {
        bv[j] = bp[(kb + j) * ldb];
        bv[j + 1] = bp[(kb + j + 1) * ldb];
      }
    }
  };
  auto mul = [&](const double (&av)[4], const double (&bv)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j], av[j], acc, 0, 0, 0);
  };
  // four whole runs in flight, then one by one
  const int rw = min(r1, k / 16);
  int r = wave * per;
  for (; r + 4 <= rw; r += 4) {
    double av[4][4], bv[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) load(r + u, av[u], bv[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) mul(av[u], bv[u]);
  }
  for (; r < rw; ++r) {
    double av[4], bv[4];
    load(r, av, bv);
    mul(av, bv);
  }
  if (r < r1) {  // the partial last run
    double av[4], bv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int kk = r * 16 + lk * 4 + j, kc = min(kk, k - 1);
      const double x = TA ? A[(int64_t)ar * lda + kc] : A[(int64_t)kc * lda + ar];
      const double y = TB ? B[(int64_t)kc * ldb + br] : B[(int64_t)br * ldb + kc];
      av[j] = kk < k ? x : 0.0;
      bv[j] = kk < k ? y : 0.0;
    }
    mul(av, bv);
  }
  // acc[q] = C(l16, lk + 4 q) of the tile
#pragma unroll
  for (int q = 0; q < 4; ++q) red[wave][(lk + 4 * q) * 16 + l16] = acc[q];
  __syncthreads();
  if (!mine) return;
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < kThinWaves; ++w) s += red[w][e];
  double v = alpha * s;
  if (beta != 0.0) v += beta * c0;
  C[(int64_t)cj * ldc + ci] = v;
}

// The tile expected to finish first (0: the 16x16 kernel).  A CU's time for one
// tile is about k c + o whether one or several workgroups share it, and the
// launch takes as many rounds as its busiest CU has tiles; c and o in ns,
// fitted to sweeps (both sides of some lines, in us): 1000 x 777 x 1301 has
// 128: 185, 64: 60, 32: 74; 2000 x 500 x 256 has 48, 16, 18; 2048^3 has 317,
// 374, 476; 500 x 500 x 8000 has 1064, 326, 122; 300^3 has 45, 17, 8 and 16x16:
// 6; 128 x 128 x 2000 has 269, 85, 30 and 10.
int pick_tile(int m, int n, int k, int mode) {
  struct Cost {
    int ts;
    double c, o;
  };
  static const Cost costs[] = {{128, 130.0, 6000.0}, {64, 45.0, 1500.0}, {32, 14.8, 1000.0},
                               {0, 3.7, 700.0}};
  int best = 128;
  double t_best = 1e300;
  for (const Cost& q : costs) {
    if (mode != 0 && q.ts < 64) break;
    const int ts = q.ts ? q.ts : 16;
    const int64_t tm = ceil_div(m, ts), tn = ceil_div(n, ts);
    const int64_t tiles = mode == 0 ? tm * tn
                                    : (mode == 1 ? tri_tiles((int)tm, (int)tn)
                                                 : tri_tiles((int)tn, (int)tm));
    const double t = (double)((tiles + kCus - 1) / kCus) * (k * q.c + q.o);
    if (t < t_best) {
      t_best = t;
      best = q.ts;
    }
  }
  return best;
}

template <int TS, bool TA, bool TB, int MODE, bool CIN>
void launch_tile(hipStream_t s, int m, int n, int k, double alpha, const double* A, int64_t lda,
                 const double* B, int64_t ldb, double beta, double* C, int64_t ldc,
                 const int* abort_flag) {
  const int tm = ceil_div(m, TS), tn = ceil_div(n, TS);
  const int tiles = MODE == 0 ? tm * tn : (MODE == 1 ? tri_tiles(tm, tn) : tri_tiles(tn, tm));
  hipLaunchKernelGGL((dgemm_kernel<TS, TA, TB, MODE, CIN>), dim3(tiles), dim3(Tile<TS>::NT), 0, s,
                     m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, abort_flag);
}

template <bool TA, bool TB, int MODE>
void launch_t(hipStream_t s, int m, int n, int k, double alpha, const double* A, int64_t lda,
              const double* B, int64_t ldb, double beta, double* C, int64_t ldc,
              const int* abort_flag) {
  const int ts = pick_tile(m, n, k, MODE);
  if (ts == 64) {
    launch_tile<64, TA, TB, MODE, false>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                         abort_flag);
    return;
  }
  if constexpr (MODE == 0) {
    if (ts == 32) {
      launch_tile<32, TA, TB, 0, false>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                        abort_flag);
      return;
    }
    if (ts == 0) {
      hipLaunchKernelGGL((dgemm_thin_kernel<TA, TB>), dim3(ceil_div(m, 16) * ceil_div(n, 16)),
                         dim3(64 * kThinWaves), 0, s, m, n, k, alpha, A, lda, B, ldb, beta, C,
                         ldc, abort_flag);
      return;
    }
  }
  if (beta == 1.0 && (alpha == 1.0 || alpha == -1.0) && k >= 8 * Tile<128>::BK &&
      k % Tile<128>::BK == 0 && m >= 2 && n >= 2 && lda <= kMaxPairLd && ldb <= kMaxPairLd &&
      ldc <= kMaxPairLd)
    launch_tile<128, TA, TB, MODE, true>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                         abort_flag);
  else
    launch_tile<128, TA, TB, MODE, false>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                          abort_flag);
}

// C = beta*C for k == 0 or alpha == 0 (BLAS semantics: beta == 0 clears C,
// NaNs included)
__global__ void dscale_kernel(int m, int n, double beta, double* C, int64_t ldc, int tri) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t total = (int64_t)m * n;
  if (idx >= total) return;
  int i = (int)(idx % m), j = (int)(idx / m);
  if ((tri == 1 && i < j) || (tri == 2 && i > j)) return;
  double* c = C + (int64_t)j * ldc + i;
  *c = beta == 0.0 ? 0.0 : beta * *c;
}

}  // namespace

int dgemm_device(hipStream_t s, bool ta, bool tb, int64_t m, int64_t n, int64_t k, double alpha,
                 const double* A, int64_t lda, const double* B, int64_t ldb, double beta,
                 double* C, int64_t ldc, int tri, const int* abort_flag) {
  if (m <= 0 || n <= 0) return kOk;
  if (m > INT32_MAX || n > INT32_MAX || k > INT32_MAX) {
    set_error("dgemm: dimensions beyond int32 are not supported");
    return kErrUnsupported;
  }
  if (k == 0 || alpha == 0.0) {
    if (beta == 1.0) return kOk;
    int64_t total = m * n;
    hipLaunchKernelGGL(dscale_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                       (int)m, (int)n, beta, C, ldc, tri);
    EAMD_HIP(hipGetLastError());
    return kOk;
  }
  int M = (int)m, N = (int)n, K = (int)k;
#define EAMD_GEMM_DISPATCH(MODE)                                                              \
  if (!ta && !tb) launch_t<false, false, MODE>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, abort_flag); \
  else if (!ta && tb) launch_t<false, true, MODE>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, abort_flag); \
  else if (ta && !tb) launch_t<true, false, MODE>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, abort_flag); \
  else launch_t<true, true, MODE>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, abort_flag);
  if (tri == 1) {
    EAMD_GEMM_DISPATCH(1)
  } else if (tri == 2) {
    EAMD_GEMM_DISPATCH(2)
  } else {
    EAMD_GEMM_DISPATCH(0)
  }
#undef EAMD_GEMM_DISPATCH
  EAMD_HIP(hipGetLastError());
  return kOk;
}

}  // namespace eamd

// ldlt.hip -- batched LDLT (symmetric diagonal pivoting) of small FP64
// matrices, and the solve with its factors.
//
// Per system this is LDLT<MatrixXd, Lower>::compute (Eigen/src/Cholesky/
// LDLT.h:491-522, through internal::ldlt_inplace<Lower>::unblocked,
// :290-395) and ::solve (:559-593).  The factorization is the reference's
// left-looking column loop, step k:
//   p = first index of the largest |a_ii| over i >= k (maxCoeff's strict '>'
//       scan: a NaN at i = k wins, NaNs elsewhere never do);
//   the lower-only symmetric exchange of k and p;
//   temp_j = d_j l_kj (j < k); a_ik -= sum_j l_ij temp_j (i >= k);
//   l_ik = a_ik / a_kk (i > k) when a_kk != 0, else the column must be zero;
//   the sign state machine and the NumericalIssue rules of the reference.
//
// MI355X mapping.  Batches whose largest n is at most 32 take eight lanes per
// system (ldlt_small_kernel, ldlt_solve_small_kernel below).  Larger ones take
// a wave per system: the lower triangle is staged in LDS (column stride n + 1),
// lane i owns row i, so the pivot search is one butterfly max plus a ballot for
// the first lane holding it, the exchange is a set of disjoint element swaps
// done by all lanes at once, and the column update is one length-k dot product
// per lane against temp held in LDS.  Their solve has x_i in lane i: each
// permutation is one gather (every lane follows its position through the
// transpositions) and the substitutions exchange values by lane shuffles.
// No host synchronisation: both launches can be captured in a HIP graph.
#include <type_traits>

#include "../../include/eigen_amd.h"
#include "common.h"
#include "kernels.h"

namespace eamd {

namespace {

constexpr int kLdltMaxN = 64;

// info: 0 Success, 1 NumericalIssue (ComputationInfo's values), -2 for a
// size outside 0..max_n; sign: 0 PositiveSemiDef, 1 NegativeSemiDef,
// 2 ZeroSign, 3 Indefinite (internal::SignMatrix, LDLT.h:22).
template <int W>
__global__ __launch_bounds__(64) void ldlt_batch_kernel(int64_t count,
                                                        const int64_t* __restrict__ offA,
                                                        const int32_t* __restrict__ nv, int max_n,
                                                        double* __restrict__ Aall,
                                                        const int64_t* __restrict__ offT,
                                                        int32_t* __restrict__ Tall,
                                                        int32_t* __restrict__ sign_out,
                                                        int32_t* __restrict__ info) {
  constexpr int G = 64 / W;  // systems per wavefront
  // LDS per system sized by the batch's largest n, not by W: the factor is
  // latency-bound, and LDS is what limits the workgroups resident per CU
  extern __shared__ double s_lds[];
  const int stride = max_n * (max_n + 1) + max_n;  // matrix, then temp
  const int lane = threadIdx.x;
  const int sub = lane / W, sl = lane % W;
  const int64_t s = (int64_t)blockIdx.x * G + sub;
  const bool act = s < count;
  int n = act ? nv[s] : -1;
  if (act && (n < 0 || n > max_n || n > W)) {
    if (sl == 0) info[s] = -2;
    n = -1;
  }
  double* a = n >= 0 ? Aall + offA[s] : nullptr;
  int32_t* tr = n >= 0 ? Tall + offT[s] : nullptr;
  if ((n == 0 || n == 1) && sl == 0) {
    int sg = 2;
    if (n == 1) {
      tr[0] = 0;
      const double d = a[0];
      sg = d > 0.0 ? 0 : (d < 0.0 ? 1 : 2);
    }
    sign_out[s] = sg;
    info[s] = 0;
  }
  const int nl = n > 1 ? n : 0;  // steps of this system
  int nmax = nl;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) nmax = max(nmax, __shfl_xor(nmax, off));
  const int ld = nl + 1;
  double* M = s_lds + sub * stride;  // nl x nl, column stride ld
  double* temp = M + max_n * (max_n + 1);
  const unsigned long long segmask =
      W == 64 ? ~0ull : (((1ull << (W & 63)) - 1ull) << (sub * W));
  // the matrix as one contiguous run of nl * nl values, eight loads per
  // lane in flight before any is stored (the lower triangle is kept)
  const int ne = nl * nl;
  for (int e0 = 0; e0 < ne; e0 += 8 * W) {
    double vals[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + u * W + sl;
      vals[u] = e < ne ? a[e] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + u * W + sl;
      if (e < ne) {
        const int j = e / nl, i = e - j * nl;
        if (i >= j) M[i + j * ld] = vals[u];
      }
    }
  }
  __syncthreads();

  int sg = 2;
  bool ret = true, found_zero = false, stop = false, zero_exit = false;
  for (int k = 0; k < nmax; ++k) {
    const bool on = !stop && k < nl;  // the same for the W lanes of a system
    // ---- pivot: the largest |a_ii| over the system's lanes, lower index on ties
    const int ci = k + sl;
    double v = -1.0;
    if (on && ci < nl) {
      v = fabs(M[ci + ci * ld]);
      if (v != v) v = sl == 0 ? __builtin_inf() : -1.0;
    }
    // the group's largest value by a butterfly max, then the lowest lane
    // holding it from one ballot (invalid lanes hold -1, below any |a_ii|)
    double vmax = v;
#pragma unroll
    for (int off = W / 2; off >= 1; off >>= 1) vmax = fmax(vmax, __shfl_xor(vmax, off));
    const unsigned long long hit = __ballot(v == vmax) & segmask;
    const int p = k + (hit ? __builtin_ctzll(hit) - sub * W : 0);
    if (on && sl == 0) tr[k] = p;
    if (on && p != k) {
      // the lower-only exchange (LDLT.h:321-337); the four sets of
      // elements are disjoint, so every lane swaps its own at once
      if (sl < k) {
        const double t = M[k + sl * ld];
        M[k + sl * ld] = M[p + sl * ld];
        M[p + sl * ld] = t;
      }
      const int it = p + 1 + sl;
      if (it < nl) {
        const double t = M[it + k * ld];
        M[it + k * ld] = M[it + p * ld];
        M[it + p * ld] = t;
      }
      if (sl == 0) {
        const double t = M[k + k * ld];
        M[k + k * ld] = M[p + p * ld];
        M[p + p * ld] = t;
      }
      const int im = k + 1 + sl;
      if (im < p) {
        const double t = M[im + k * ld];
        M[im + k * ld] = M[p + im * ld];
        M[p + im * ld] = t;
      }
    }
    __syncthreads();
    // ---- column k: a_ik -= sum_j l_ij d_j l_kj (LDLT.h:348-354)
    if (k > 0) {
      if (on && sl < k) temp[sl] = M[sl + sl * ld] * M[k + sl * ld];
      __syncthreads();
      if (on && ci < nl) {
        double r = 0.0;
#pragma unroll 4
        for (int j = 0; j < k; ++j) r += M[ci + j * ld] * temp[j];  // loads run ahead, order kept
        M[ci + k * ld] -= r;
      }
      __syncthreads();
    }
    const double akk = on ? M[k + k * ld] : 1.0;
    const bool valid = fabs(akk) > 0.0;
    const bool zx = on && k == 0 && !valid;  // the whole diagonal is zero
    bool nz = false;
    if (zx) {
      for (int j = 0; j < nl; ++j)
        if (sl > j && sl < nl && !(M[sl + j * ld] == 0.0)) nz = true;
    } else if (on) {
      const int ib = k + 1 + sl;
      if (ib < nl) {
        if (valid)
          M[ib + k * ld] /= akk;
        else
          nz = !(M[ib + k * ld] == 0.0);
      }
    }
    const bool anynz = (__ballot(nz) & segmask) != 0ull;
    if (zx) {
      // LDLT.h:363-374: identity transpositions, success iff L is zero
      ret = !anynz;
      if (sl < nl) tr[sl] = sl;
      sg = 2;
      stop = true;
      zero_exit = true;
    } else if (on) {
      if (anynz) ret = false;
      if (found_zero && valid)
        ret = false;
      else if (!valid)
        found_zero = true;
      if (sg == 0) {
        if (akk < 0.0) sg = 3;
      } else if (sg == 1) {
        if (akk > 0.0) sg = 3;
      } else if (sg == 2) {
        if (akk > 0.0)
          sg = 0;
        else if (akk < 0.0)
          sg = 1;
      }
    }
    __syncthreads();
  }
  if (nl > 0) {
    if (!zero_exit)
      for (int j = 0; j < nl; ++j)
        if (sl >= j && sl < nl) a[sl + (int64_t)j * nl] = M[sl + j * ld];
    if (sl == 0) {
      sign_out[s] = sg;
      info[s] = ret ? 0 : 1;
    }
  }
}

// ---- max_n <= 32: eight lanes per system, eight systems in step on a wave.
// Until its own column's turn a diagonal entry holds its input value, so the
// order of the pivots, and with it every interchange, follows from the input
// diagonal alone: the transpositions are found first (selection with swaps, as
// the reference's, on values in registers), and the factorization then reads
// the triangle permuted.  That takes the search, the interchanges and their
// barriers out of the column steps, and eight systems share every
// instruction of a step (1M systems of n = 6..24: 4.41 ms with 32 lanes per
// system and the interchanges done in LDS, 1.65 ms so; 3400 VALU instructions
// and 25 KB of LDS per wave, so six waves per CU, bound it now).  Row i of the permuted matrix is
// on lane i % 8, slot i / 8; columns go in groups of eight, group g's values
// of the rows of slots r >= g in registers: first the running sums of the
// left-looking update, then L.  The sums are taken in the reference's order
// (column by column, subtracted once), so the factors do not depend on which
// kernel ran.  LDS: the packed lower triangles (the gather's source) and the
// eight rows a later group needs of a finished one.
constexpr int kSmallLanes = 8, kSmallSys = 64 / kSmallLanes;

template <int B, int E, typename F>
__device__ __forceinline__ void sfor(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    sfor<B + 1, E>(f);
  }
}

// lane N of each group of eight lanes
template <int N>
__device__ __forceinline__ int bcast8(int x) {
  const int lo = __builtin_amdgcn_update_dpp(x, x, 0x150 + N, 0xf, 0x3, false);
  return __builtin_amdgcn_update_dpp(lo, x, 0x150 + 8 + N, 0xf, 0xc, false);
}
template <int N>
__device__ __forceinline__ double bcast8(double x) {
  const long long b = __double_as_longlong(x);
  return __longlong_as_double(((long long)bcast8<N>((int)(b >> 32)) << 32) |
                              (unsigned)bcast8<N>((int)b));
}

// the partner's value in the butterfly of a group of eight: xor 1, xor 2, then
// the other quad (mirrored: its lanes agree by then)
template <int CTRL>
__device__ __forceinline__ int dpp_i(int x) {
  return __builtin_amdgcn_mov_dpp(x, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ double dpp_f(double x) {
  const long long b = __double_as_longlong(x);
  return __longlong_as_double(((long long)dpp_i<CTRL>((int)(b >> 32)) << 32) |
                              (unsigned)dpp_i<CTRL>((int)b));
}
__device__ __forceinline__ double max8(double x) {
  x = fmax(x, dpp_f<0xB1>(x));
  x = fmax(x, dpp_f<0x4E>(x));
  return fmax(x, dpp_f<0x141>(x));
}
__device__ __forceinline__ int min8(int x) {
  x = min(x, dpp_i<0xB1>(x));
  x = min(x, dpp_i<0x4E>(x));
  return min(x, dpp_i<0x141>(x));
}

// doubles of LDS: packed triangles, one group's rows per system, the order
inline size_t small_lds(int max_n) {
  const size_t tri = (size_t)max_n * (max_n + 1) / 2;
  return sizeof(double) * kSmallSys * (tri + 64) + sizeof(int) * kSmallSys * 64;
}

template <int K>
__global__ __launch_bounds__(64) void ldlt_small_kernel(
    int64_t count, const int64_t* __restrict__ offA, const int32_t* __restrict__ nv, int max_n,
    double* __restrict__ Aall, const int64_t* __restrict__ offT, int32_t* __restrict__ Tall,
    int32_t* __restrict__ sign_out, int32_t* __restrict__ info) {
  extern __shared__ __align__(16) double s_lds[];
  const int tri = max_n * (max_n + 1) / 2;
  const int lane = threadIdx.x, sl = lane % kSmallLanes, sub = lane / kSmallLanes;
  double* W = s_lds + sub * 64;                          // [8 columns][8 rows]
  double* S = s_lds + kSmallSys * 64 + sub * tri;        // packed lower, column by column
  // per position: the row it takes, and where that row's column starts in S
  int* ord = reinterpret_cast<int*>(s_lds + kSmallSys * (64 + tri)) + sub * 64;
  const unsigned long long segmask = 0xffull << (8 * sub);
  const int64_t s = (int64_t)blockIdx.x * kSmallSys + sub;
  const bool act = s < count;
  // (three independent loads: one round trip)
  const int64_t oa = act ? offA[s] : 0, ot = act ? offT[s] : 0;
  int n = act ? nv[s] : -1;
  if (act && (n < 0 || n > max_n)) {
    if (sl == 0) info[s] = -2;
    n = -1;
  }
  double* a = Aall + (n > 0 ? oa : 0);
  int32_t* tr = Tall + (n > 0 ? ot : 0);
  if ((n == 0 || n == 1) && sl == 0) {
    int sg = 2;
    if (n == 1) {
      tr[0] = 0;
      const double d = a[0];
      sg = d > 0.0 ? 0 : (d < 0.0 ? 1 : 2);
    }
    sign_out[s] = sg;
    info[s] = 0;
  }
  const int nl = n > 1 ? n : 0;
  int nmax = nl;
#pragma unroll
  for (int off = 8; off < 64; off <<= 1) nmax = max(nmax, __shfl_xor(nmax, off));
  nmax = __builtin_amdgcn_readfirstlane(nmax);
  // element (r, c), r >= c, of the packed lower triangle is at colstart(c) + r
  auto colstart = [&](int c) { return c * (2 * nl - 1 - c) / 2; };

  // ---- the triangle into LDS, every load in flight before the first store.
  // Elements outside it read (and store again) the nearest one inside.
  double v[K];  // my diagonal entries
#pragma unroll
  for (int r = 0; r < K; ++r) v[r] = 0.0;
  if (nl > 0) {
    double x[K][K][8];
    auto each = [&](auto&& f) {
      sfor<0, K>([&](auto gc) {
        constexpr int g = decltype(gc)::value;
        if (8 * g >= nmax) return;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int c = min(8 * g + q, nl - 1);
#pragma unroll
          for (int r = g; r < K; ++r)
            f(c, max(c, min(8 * r + sl, nl - 1)), x[g][r][q]);
        }
      });
    };
    each([&](int c, int i, double& y) { y = a[c * nl + i]; });
    each([&](int c, int i, double& y) { S[colstart(c) + i] = y; });
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const int i = sl + 8 * r;
    if (i < nl) v[r] = S[colstart(i) + i];
  }

  // ---- the pivots' order: position k takes the first position holding the
  // largest |a_ii| over i >= k (a NaN wins at i = k only)
  bool tie = false;
  int rank[K];
  {
    // W: the magnitudes; rank = how many are larger
#pragma unroll
    for (int r = 0; r < K; ++r) W[sl + 8 * r] = sl + 8 * r < nl ? fabs(v[r]) : -2.0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < K; ++r) rank[r] = 0;
    int same[K];
#pragma unroll
    for (int r = 0; r < K; ++r) same[r] = 0;
#pragma unroll 4
    for (int j = 0; j < nmax; ++j) {
      const double w = W[j];
#pragma unroll
      for (int r = 0; r < K; ++r) {
        const double m = fabs(v[r]);
        rank[r] += w > m ? 1 : 0;
        same[r] += w == m ? 1 : 0;
      }
    }
    // (a NaN equals nothing, not even itself)
#pragma unroll
    for (int r = 0; r < K; ++r) tie = tie || (sl + 8 * r < nl && same[r] != 1);
    __syncthreads();
  }
  if (__ballot(tie) == 0) {
    // distinct magnitudes: position k takes the entry of rank k, and the
    // transposition is where that entry is by then: it starts at its own
    // index, and while that lies before k it was moved on by that step
    int* tw = ord + 32;
#pragma unroll
    for (int r = 0; r < K; ++r) {
      ord[sl + 8 * r] = 0;
      tw[sl + 8 * r] = -1;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < K; ++r)
      if (sl + 8 * r < nl) ord[rank[r]] = sl + 8 * r;
    __syncthreads();
    int x[K];
    bool todo = false;
#pragma unroll
    for (int r = 0; r < K; ++r) {
      x[r] = sl + 8 * r < nl ? ord[sl + 8 * r] : 1 << 20;
      todo = todo || sl + 8 * r < nl;
    }
    volatile int* tv = tw;
    while (__ballot(todo) != 0) {
      todo = false;
#pragma unroll
      for (int r = 0; r < K; ++r) {
        const int k = sl + 8 * r;
        if (k < nl) {
          const int y = x[r] < k ? tv[x[r]] : -1;
          x[r] = y >= 0 ? y : x[r];
          if (x[r] >= k) tv[k] = x[r];
          else todo = true;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < K; ++r)
      if (sl + 8 * r < nl) tr[sl + 8 * r] = x[r];
  } else {
    // equal magnitudes or NaN: the selection itself, slot r of group j0 being
    // position j0 + 8 r + sl
    int id[K];
    double d[K];
#pragma unroll
    for (int r = 0; r < K; ++r) {
      id[r] = sl + 8 * r;
      d[r] = v[r];
    }
#pragma unroll 1
    for (int j0 = 0; j0 < 8 * K; j0 += 8) {
      if (j0 < nmax) {
        sfor<0, 8>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          const int k = j0 + q;
          if (k >= nmax) return;
          double vv[K], m = -2.0;
#pragma unroll
          for (int r = 0; r < K; ++r) {
            const int pos = j0 + 8 * r + sl;
            double w = fabs(d[r]);
            if (w != w) w = pos == k ? __builtin_inf() : -1.0;
            vv[r] = pos >= k && pos < nl ? w : -2.0;
            m = fmax(m, vv[r]);
          }
          m = max8(m);
          int c = 1 << 20;
#pragma unroll
          for (int r = K - 1; r >= 0; --r) c = vv[r] == m ? j0 + 8 * r + sl : c;
          const int p = min8(c);
          const bool on = k < nl;
          if (on && sl == q) tr[k] = p;
          // positions k and p change places
          int ip = 1 << 20;
          const double dv = bcast8<q>(d[0]);
          const int ik = bcast8<q>(id[0]);
#pragma unroll
          for (int r = 0; r < K; ++r) ip = j0 + 8 * r + sl == p ? id[r] : ip;
          ip = min8(ip);
#pragma unroll
          for (int r = 0; r < K; ++r) {
            const bool here = on && j0 + 8 * r + sl == p;
            d[r] = here ? dv : d[r];
            id[r] = here ? ik : id[r];
          }
          if (on && sl == q) id[0] = ip;
        });
      }
      ord[j0 + sl] = j0 + sl < nl ? id[0] : 0;
#pragma unroll
      for (int r = 0; r + 1 < K; ++r) {
        d[r] = d[r + 1];
        id[r] = id[r + 1];
      }
    }
  }
  __syncthreads();

  // ---- factorization
  int oi[K], ci[K];
#pragma unroll
  for (int r = 0; r < K; ++r) {
    oi[r] = ord[sl + 8 * r];
    ci[r] = nl > 0 ? colstart(oi[r]) : 0;
    ord[32 + sl + 8 * r] = ci[r];
  }
  __syncthreads();
  double L[K][K][8];  // [group][slot >= group][column]: sums, then L (D on the diagonal)
#pragma unroll
  for (int g = 0; g < K; ++g)
#pragma unroll
    for (int r = 0; r < K; ++r)
#pragma unroll
      for (int q = 0; q < 8; ++q) L[g][r][q] = 0.0;
  // the sign machine ends in PositiveSemiDef, NegativeSemiDef, ZeroSign or
  // Indefinite as it has seen positive, negative, no or both kinds of pivots
  bool pos = false, neg = false;
  bool ret = true, found_zero = false, zero_exit = false;
  sfor<0, K>([&](auto gc) {
    constexpr int g = decltype(gc)::value;
    if (8 * g >= nmax) return;
    int oj[8], cj[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      oj[q] = ord[8 * g + q];
      cj[q] = ord[32 + 8 * g + q];
    }
    // the group's input values, gathered ahead of its steps
    double in[K][8];
#pragma unroll
    for (int q = 0; q < 8; ++q)
#pragma unroll
      for (int r = g; r < K; ++r)
        in[r][q] = S[oi[r] <= oj[q] ? ci[r] + oj[q] : cj[q] + oi[r]];
    double dk[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) dk[q] = 0.0;
    sfor<0, 8>([&](auto qc) {
      constexpr int q = decltype(qc)::value, k = 8 * g + q;
      if (k >= nmax) return;
      const bool on = k < nl && !zero_exit;
      double x[K];
#pragma unroll
      for (int r = g; r < K; ++r) x[r] = in[r][q] - L[g][r][q];
      const double akk = bcast8<q>(x[g]);
      const bool valid = fabs(akk) > 0.0;
      dk[q] = akk;
      if (__ballot(on && !valid) == 0) {
#pragma unroll
        for (int r = g; r < K; ++r) L[g][r][q] = x[r] / akk;
      } else {
        bool nz = false;
#pragma unroll
        for (int r = g; r < K; ++r) {
          const bool below = (r > g || sl > q) && sl + 8 * r < nl;
          nz = nz || (below && !(x[r] == 0.0));
          L[g][r][q] = valid ? x[r] / akk : x[r];
        }
        const bool anynz = (__ballot(nz) & segmask) != 0ull;
        if (k == 0) {
          // the whole diagonal is zero (LDLT.h:363-374): identity
          // transpositions, success iff the matrix below it is zero
          bool any = false;
          for (int c = 0; c < nl; ++c)
            for (int r = c + 1 + sl; r < nl; r += 8) any = any || !(S[colstart(c) + r] == 0.0);
          const bool anyel = (__ballot(any) & segmask) != 0ull;
          if (on && !valid) {
            ret = !anyel;
            for (int r = sl; r < nl; r += 8) tr[r] = r;
            zero_exit = true;
          }
        }
        if (on && !valid && !zero_exit) {
          if (anynz) ret = false;
          found_zero = true;
        }
      }
      if (sl == q) L[g][g][q] = akk;
      ret = ret && !(on && found_zero && valid);
      pos = pos || (on && akk > 0.0);
      neg = neg || (on && akk < 0.0);
      // the sums of the group's later columns
      const double w = akk * L[g][g][q];
      sfor<q + 1, 8>([&](auto q2c) {
        constexpr int q2 = decltype(q2c)::value;
        const double wb = bcast8<q2>(w);
#pragma unroll
        for (int r = g; r < K; ++r) L[g][r][q2] += L[g][r][q] * wb;
      });
    });
    // the sums of the later groups' columns: group g2's rows of this group,
    // times D, pass through LDS
    sfor<g + 1, K>([&](auto g2c) {
      constexpr int g2 = decltype(g2c)::value;
      if (8 * g2 >= nmax) return;
#pragma unroll
      for (int q = 0; q < 8; ++q) W[q * 8 + sl] = dk[q] * L[g][g2][q];
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 8; ++q) {
#pragma unroll
        for (int q2 = 0; q2 < 8; ++q2) {
          const double wv = W[q * 8 + q2];
#pragma unroll
          for (int r = g2; r < K; ++r) L[g2][r][q2] += L[g][r][q] * wv;
        }
      }
      __syncthreads();
    });
    // group g's columns are final
    if (!zero_exit) {
      double* p = a + 8 * g * (nl + 1) + sl;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
#pragma unroll
        for (int r = g; r < K; ++r)
          if (sl + 8 * r < nl && (r > g || sl >= q)) p[8 * (r - g)] = L[g][r][q];
        p += nl;
        asm volatile("" : "+v"(p));
      }
    }
  });
  if (nl > 0 && sl == 0) {
    sign_out[s] = pos ? (neg ? 3 : 0) : (neg ? 1 : 2);
    info[s] = ret ? 0 : 1;
  }
}

// x <- A^{-1} b for sizes up to 8 K: eight lanes per system, eight systems in
// step on a wave, row i of L on lane i % 8 (slot i / 8) in registers for both
// sweeps: L y = P b takes x_k from its lane, L^T x = y sums a column over the
// eight lanes.  Every lane follows its rows' positions back through the
// transpositions, so P is one gather of b and P^T one scatter of x.  Every
// line of a system is touched in one go (reading the diagonal ahead of the
// columns fetched 1.4 times as much: the resident systems exceed the L2).
// 1M systems of n = 6..24: 1.94 ms with 32 lanes per system, shuffles and a
// second copy of L, 0.67 ms so.
template <int K>
__global__ __launch_bounds__(256) void ldlt_solve_small_kernel(
    int64_t count, const int64_t* __restrict__ offA, const int32_t* __restrict__ nv, int max_n,
    const double* __restrict__ Aall, const int64_t* __restrict__ offT,
    const int32_t* __restrict__ Tall, const int64_t* __restrict__ offb, double* __restrict__ B) {
  const int lane = threadIdx.x & 63, sl = lane % kSmallLanes;
  const int64_t s =
      (((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6) * kSmallSys + lane / kSmallLanes;
  const bool act = s < count;
  const int64_t oa = act ? offA[s] : 0, ot = act ? offT[s] : 0, ob = act ? offb[s] : 0;
  int n = act ? nv[s] : 0;
  if (n < 0 || n > max_n) n = 0;
  int nmax = n;
#pragma unroll
  for (int off = 8; off < 64; off <<= 1) nmax = max(nmax, __shfl_xor(nmax, off));
  nmax = __builtin_amdgcn_readfirstlane(nmax);
  double L[K][8 * K], d[K], x[K];  // L[r][k], k < 8 (r + 1): L(sl + 8 r, k), zero from k = row on
  int t[K], src[K];
#pragma unroll
  for (int r = 0; r < K; ++r) {
    t[r] = src[r] = sl + 8 * r;
    d[r] = 1.0;
    x[r] = 0.0;
  }
  if (n > 0) {
    const double* a = Aall + oa;
    const int32_t* tr = Tall + ot;
#pragma unroll
    for (int r = 0; r < K; ++r) {
      const int i = min(sl + 8 * r, n - 1);
      const int tv = tr[i];
      t[r] = sl + 8 * r < n ? tv : sl + 8 * r;
    }
    // column by column: a line's two halves (rows eight apart) back to back
    sfor<0, 8 * K>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      if (k >= nmax) return;
      const double* c = a + min(k, n - 1) * n;
#pragma unroll
      for (int r = k / 8; r < K; ++r) {
        const int i = min(sl + 8 * r, n - 1);
        const double v = c[i];
        L[r][k] = k < i && sl + 8 * r < n ? v : 0.0;
        if (r == k / 8) d[r] = k == sl + 8 * r && k < n ? v : d[r];
      }
    });
  } else {
#pragma unroll
    for (int r = 0; r < K; ++r)
#pragma unroll
      for (int k = 0; k < 8 * (r + 1); ++k) L[r][k] = 0.0;
  }
  // (P b)_i = b_src: back through the transpositions (identity past n)
  sfor<0, 8 * K>([&](auto kc) {
    constexpr int k = 8 * K - 1 - decltype(kc)::value;
    if (k >= nmax) return;
    const int tk = bcast8<k % 8>(t[k / 8]);
#pragma unroll
    for (int r = 0; r < K; ++r) src[r] = src[r] == k ? tk : (src[r] == tk ? k : src[r]);
  });
  double* xp = B + ob;
#pragma unroll
  for (int r = 0; r < K; ++r)
    if (sl + 8 * r < n) x[r] = xp[src[r]];
  sfor<0, 8 * K>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    if (k >= nmax) return;
    const double xk = bcast8<k % 8>(x[k / 8]);
#pragma unroll
    for (int r = k / 8; r < K; ++r)
      if (8 * r < nmax) x[r] -= L[r][k] * xk;
  });
  // D^+ y: rows whose |d| is not above 1 / DBL_MAX become zero
#pragma unroll
  for (int r = 0; r < K; ++r)
    x[r] = fabs(d[r]) > 1.0 / 1.7976931348623157e308 ? x[r] / d[r] : 0.0;
  sfor<1, 8 * K>([&](auto kc) {
    constexpr int k = 8 * K - 1 - decltype(kc)::value;
    if (k >= nmax) return;
    double p = 0.0;
#pragma unroll
    for (int r = k / 8; r < K; ++r)
      if (8 * r < nmax) p += L[r][k] * x[r];
    p += dpp_f<0xB1>(p);
    p += dpp_f<0x4E>(p);
    p += dpp_f<0x141>(p);
    x[k / 8] -= sl == k % 8 ? p : 0.0;
  });
#pragma unroll
  for (int r = 0; r < K; ++r)
    if (sl + 8 * r < n) xp[src[r]] = x[r];
}

// x <- A^{-1} b for sizes above 32: a wave per system (x_i in lane i), four
// waves per workgroup.  Systems of a size outside 0..max_n are
// left as they are (their factorization reported -2 and wrote no
// transpositions).
template <int W>
__global__ __launch_bounds__(256) void ldlt_solve_batch_kernel(
    int64_t count, const int64_t* __restrict__ offA, const int32_t* __restrict__ nv, int max_n,
    const double* __restrict__ Aall, const int64_t* __restrict__ offT,
    const int32_t* __restrict__ Tall, const int64_t* __restrict__ offb, double* __restrict__ B) {
  constexpr int G = 64 / W;
  const int lane = threadIdx.x & 63;
  const int sub = lane / W, sl = lane % W, base = sub * W;
  const int64_t s = (((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6) * G + sub;
  if (s >= count) return;  // whole groups: every shuffle below stays in the group
  const int n = nv[s];
  if (n <= 0 || n > max_n || n > W) return;
  const double* a = Aall + offA[s];
  double* xp = B + offb[s];
  // a lane's transposition, right-hand side and d_i, requested together
  const int trv = sl < n ? Tall[offT[s] + sl] : 0;
  double x = sl < n ? xp[sl] : 0.0;
  const double d = sl < n ? a[sl + (int64_t)sl * n] : 1.0;
  // P and P^T as gathers: every lane follows its own position through the
  // transpositions (all W of them fetched by independent shuffles), so each
  // permutation costs one shuffle of x instead of a chain of swaps
  int pk[W];
#pragma unroll
  for (int k = 0; k < W; ++k) pk[k] = __shfl(trv, base + k);
  int src_p = sl, src_pt = sl;  // x (P b)_i = b_src_p; (P^T y)_i = y_src_pt
#pragma unroll
  for (int k = W - 1; k >= 0; --k)
    if (k < n) {
      if (src_p == k)
        src_p = pk[k];
      else if (src_p == pk[k])
        src_p = k;
    }
#pragma unroll
  for (int k = 0; k < W; ++k)
    if (k < n) {
      if (src_pt == k)
        src_pt = pk[k];
      else if (src_pt == pk[k])
        src_pt = k;
    }
  x = __shfl(x, base + src_p);
  // L y = x (unit lower), column k of L per step
  for (int k = 0; k < n - 1; ++k) {
    const double xk = __shfl(x, base + k);
    if (sl > k && sl < n) x -= a[sl + (int64_t)k * n] * xk;
  }
  // D^+ y: rows whose |d| is not above 1 / DBL_MAX become zero
  if (sl < n) x = fabs(d) > 1.0 / 1.7976931348623157e308 ? x / d : 0.0;
  // L^T x = y, row i of L per step
  for (int i = n - 1; i > 0; --i) {
    const double xi = __shfl(x, base + i);
    if (sl < i) x -= a[i + (int64_t)sl * n] * xi;
  }
  // x = P^T x
  x = __shfl(x, base + src_pt);
  if (sl < n) xp[sl] = x;
}

// LDLT rank-one update in place: one wave per factor, row i on lane i % 64
// (up to four rows per lane, n <= 256).  Restates
// internal::ldlt_inplace<Lower>::update (LDLT.h:440-449): w is permuted by
// the factor's transpositions in order (tmp = P w), then updateInPlace
// (LDLT.h:404-437) runs column by column: d_j += sigma w_j^2 / alpha,
// alpha += sigma w_j^2 / d_j, w_i -= w_j l_ij, and, if gamma = d_j alpha +
// sigma w_j^2 is not zero, l_ij += (sigma w_j / gamma) w_i below the
// diagonal, stopping once alpha is not finite.  Column j's entries are read
// and written by their own lanes in step j only, and d_j is read by all
// lanes before lane j % 64 writes it.  info: 0, or -2 for a size outside
// 0..256.
constexpr int kLdltRankMaxN = 256;

// element idx of a vector kept as four register slots per lane (slot idx /
// 64 of lane idx % 64), as a wave-uniform value
__device__ __forceinline__ double lane_get(const double (&t)[4], int idx) {
  const int k = idx >> 6;
  const double sel = k == 0 ? t[0] : (k == 1 ? t[1] : (k == 2 ? t[2] : t[3]));
  const long long b = __double_as_longlong(sel);
  return __longlong_as_double(((long long)__builtin_amdgcn_readlane((int)(b >> 32), idx & 63) << 32) |
                              (unsigned)__builtin_amdgcn_readlane((int)b, idx & 63));
}

__global__ __launch_bounds__(256) void ldlt_rank_update_kernel(
    int64_t count, const int64_t* __restrict__ offA, const int32_t* __restrict__ nv,
    double* __restrict__ Aall, const int64_t* __restrict__ offT, const int32_t* __restrict__ Tall,
    const int64_t* __restrict__ offw, const double* __restrict__ Wall,
    const double* __restrict__ sigmas, int32_t* __restrict__ info) {
  constexpr int K = kLdltRankMaxN / 64;
  const int lane = threadIdx.x & 63;
  const int64_t s = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6;
  if (s >= count) return;  // whole waves
  const int n = nv[s];
  if (n < 0 || n > kLdltRankMaxN) {
    if (lane == 0) info[s] = -2;
    return;
  }
  double* A = Aall + offA[s];
  const int32_t* tr = Tall + offT[s];
  const double* w = Wall + offw[s];
  const double sigma = sigmas ? sigmas[s] : 1.0;
  double t[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = lane + 64 * k;
    t[k] = i < n ? w[i] : 0.0;
  }
  // tmp = P w: transposition k swaps entries k and tr[k], k = 0, 1, ...
  for (int k = 0; k < n; ++k) {
    const int j = tr[k];
    if (j == k || j < 0 || j >= n) continue;
    const double vk = lane_get(t, k), vj = lane_get(t, j);
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const int i = lane + 64 * q;
      t[q] = i == k ? vj : (i == j ? vk : t[q]);
    }
  }
  double alpha = 1.0;
  for (int j = 0; j < n; ++j) {
    if (!__builtin_isfinite(alpha)) break;
    const double dj = A[j + (int64_t)j * n];
    const double wj = lane_get(t, j);
    const double swj2 = sigma * wj * wj;
    const double gamma = dj * alpha + swj2;
    if (lane == (j & 63)) A[j + (int64_t)j * n] = dj + swj2 / alpha;
    alpha += swj2 / dj;
    const double c = sigma * wj / gamma;
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const int i = lane + 64 * q;
      if (i > j && i < n) {
        const double lij = A[i + (int64_t)j * n];
        t[q] -= wj * lij;
        if (gamma != 0.0) A[i + (int64_t)j * n] = lij + c * t[q];
      }
    }
  }
  if (lane == 0) info[s] = 0;
}

}  // namespace

int ldlt_rank_update_batched(eamd_handle* h, int64_t count, const int64_t* offA, const int32_t* n,
                             double* A, const int64_t* offT, const int32_t* T,
                             const int64_t* offw, const double* w, const double* sigma,
                             int32_t* info) {
  if (count <= 0) return kOk;
  const int64_t blocks = (count + 3) / 4;  // four waves (factors) per workgroup
  if (blocks > INT32_MAX) {
    set_error("ldlt rank update: %lld factors exceed one launch", (long long)count);
    return kErrUnsupported;
  }
  hipLaunchKernelGGL(ldlt_rank_update_kernel, dim3((unsigned)blocks), dim3(256), 0, h->stream,
                     count, offA, n, A, offT, T, offw, w, sigma, info);
  EAMD_HIP(hipGetLastError());
  return kOk;
}

int ldlt_batched(eamd_handle* h, int64_t count, const int64_t* offA, const int32_t* n, int max_n,
                 double* A, const int64_t* offT, int32_t* T, int32_t* sign, int32_t* info) {
  if (count == 0) return kOk;
  if (max_n < 0 || max_n > kLdltMaxN) {
    set_error("ldlt: max_n %d outside 0..%d", max_n, kLdltMaxN);
    return kErrUnsupported;
  }
  const int W = max_n <= 32 ? kSmallLanes : 64;
  const int64_t blocks = (count + 64 / W - 1) / (64 / W);
  if (blocks > INT32_MAX) {
    set_error("ldlt: %lld systems exceed one launch", (long long)count);
    return kErrUnsupported;
  }
  const dim3 grid((unsigned)blocks), block(64);
  if (max_n > 32) {
    const size_t lds = sizeof(double) * ((size_t)max_n * (max_n + 1) + max_n);
    hipLaunchKernelGGL(ldlt_batch_kernel<64>, grid, block, lds, h->stream, count, offA, n, max_n,
                       A, offT, T, sign, info);
  } else {
#define EAMD_LDLT(K)                                                                           \
  hipLaunchKernelGGL(ldlt_small_kernel<K>, grid, block, small_lds(max_n), h->stream, count,   \
                     offA, n, max_n, A, offT, T, sign, info)
    if (max_n <= 8) EAMD_LDLT(1);
    else if (max_n <= 16) EAMD_LDLT(2);
    else if (max_n <= 24) EAMD_LDLT(3);
    else EAMD_LDLT(4);
#undef EAMD_LDLT
  }
  EAMD_HIP(hipGetLastError());
  return kOk;
}

int ldlt_solve_batched(eamd_handle* h, int64_t count, const int64_t* offA, const int32_t* n,
                       int max_n, const double* A, const int64_t* offT, const int32_t* T,
                       const int64_t* offb, double* b) {
  if (count == 0) return kOk;
  if (max_n < 0 || max_n > kLdltMaxN) {
    set_error("ldlt solve: max_n %d outside 0..%d", max_n, kLdltMaxN);
    return kErrUnsupported;
  }
  const int W = max_n <= 32 ? kSmallLanes : 64;
  const int64_t per_block = 4 * (64 / W);  // four wavefronts per workgroup
  const int64_t blocks = (count + per_block - 1) / per_block;
  if (blocks > INT32_MAX) {
    set_error("ldlt solve: %lld systems exceed one launch", (long long)count);
    return kErrUnsupported;
  }
  const dim3 grid((unsigned)blocks), block(256);
  if (max_n > 32) {
    hipLaunchKernelGGL(ldlt_solve_batch_kernel<64>, grid, block, 0, h->stream, count, offA, n,
                       max_n, A, offT, T, offb, b);
  } else {
#define EAMD_LDLT(K)                                                                        \
  hipLaunchKernelGGL(ldlt_solve_small_kernel<K>, grid, block, 0, h->stream, count, offA, n, \
                     max_n, A, offT, T, offb, b)
    if (max_n <= 8) EAMD_LDLT(1);
    else if (max_n <= 16) EAMD_LDLT(2);
    else if (max_n <= 24) EAMD_LDLT(3);
    else EAMD_LDLT(4);
#undef EAMD_LDLT
  }
  EAMD_HIP(hipGetLastError());
  return kOk;
}

}  // namespace eamd

// trsv.hip -- blocked triangular solves with one right-hand side.
//
// Replaces triangular_solve_vector (TriangularSolverVector.h:88-139) and the
// one-column use of triangular_solve_matrix (TriangularSolverMatrix.h:38-184)
// inside PartialPivLU::_solve_impl (PartialPivLU.h:226-244) and
// LLT::_solve_impl (LLT.h:475-505); several columns go to trsm.hip.
//
// One workgroup per BS-row block, dispatched in dependency order.  Workgroup
// b first inverts its diagonal block in LDS (independent of the others, so
// it overlaps the wait), accumulates B_b - sum_j T_bj X_j over its
// predecessors j in order, then X_b = inv(T_bb) * (...).  Solved values are
// published as 8-byte words carrying 32 bits of payload and the call's
// epoch (an aligned 8-byte store is single-copy atomic, so a word with the
// right epoch has the right payload): consumers poll the words themselves,
// with no flag and no cache write-back or invalidate on the critical path.
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace eamd {

namespace {

// polls a wait may take before it gives up (and reports a time-out) unless
// EAMD_TRSV_SPIN sets another limit
constexpr int kSpin = 1 << 26;

template <typename T>
__device__ __forceinline__ T tload(const T* p) {
  return __hip_atomic_load(const_cast<T*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// element (r, c) of the triangular matrix in the requested layout
template <typename T, bool ROWMAJOR>
__device__ __forceinline__ const T* tptr(const T* A, int64_t ld, int r, int c) {
  return ROWMAJOR ? A + (int64_t)r * ld + c : A + r + (int64_t)c * ld;
}

typedef unsigned long long u64;

template <typename T>
struct XWords {
  static constexpr int n = sizeof(T) / 4;  // 32-bit payload words per value
};

template <typename T, bool ROWMAJOR, bool LOWER, bool UNIT, int BS>
__global__ __launch_bounds__(4 * BS) void trsv_chain_kernel(int n, const T* __restrict__ A,
                                                         int64_t lda, T* __restrict__ X,
                                                         u64* __restrict__ xw, unsigned epoch,
                                                         int* __restrict__ err, int spin_limit) {
  static_assert(BS == 64 || BS == 128, "four threads per row of a 64- or 128-row block");
  constexpr int NT = 4 * BS;   // threads
  constexpr int SEG = BS / 4;  // columns of a predecessor block per thread
  constexpr int NW = XWords<T>::n;
  constexpr int CHUNK = BS * NW;                // words of one block's solution
  constexpr int WPT = (CHUNK + NT - 1) / NT;    // words staged per thread
  __shared__ T Dinv[BS][BS + 1];
  __shared__ T Tb[BS][BS + 1];
  __shared__ T accs[BS];
  __shared__ unsigned xsw[2][CHUNK];  // staged solution of the current predecessor
  __shared__ int s_abort;
  // FP32: M = inv(T_bb) T_bl for the last predecessor l
  // is formed while the block waits, and inv(T_bb) (B_b - sum over the other
  // predecessors) before l's solution arrives, so the step after it is one
  // row of M times X_l (one barrier instead of two, no reduction through LDS)
  constexpr bool kM = sizeof(T) == 4;
  __shared__ T Tl[kM ? BS : 1][BS + 1];
  __shared__ unsigned xwv[kM ? NT / 64 : 1][BS];  // (kM) each wave's copy of X_l
  const int tid = threadIdx.x;
  const int nblk = (n + BS - 1) / BS;
  // workgroups are dispatched in dependency order
  const int w = blockIdx.x;
  const int b = LOWER ? w : nblk - 1 - w;
  const int rb0 = b * BS;
  const int bs = min(BS, n - rb0);
  const int r = tid >> 2, q = tid & 3;  // my row of the block, my quarter of each column block
  const int ndep = LOWER ? b : nblk - 1 - b;
  const int jl = LOWER ? b - 1 : b + 1;  // the last predecessor (ndep > 0)

  // ---- diagonal block into LDS and its inverse (independent of the
  // predecessors: overlaps their solves)
  for (int e = tid; e < BS * BS; e += NT) {
    const int rr = e / BS, cc = e - rr * BS;
    Tb[rr][cc] = (rr < bs && cc < bs) ? *tptr<T, ROWMAJOR>(A, lda, rb0 + rr, rb0 + cc) : T(0);
    Dinv[rr][cc] = T(0);  // the padding of a partial last block stays exactly zero
    if constexpr (kM)
      Tl[rr][cc] = (ndep > 0 && rr < bs && jl * BS + cc < n)
                       ? *tptr<T, ROWMAJOR>(A, lda, rb0 + rr, jl * BS + cc)
                       : T(0);
  }
  if (tid == 0) s_abort = 0;
  __syncthreads();
  if (tid < BS) {
    const int c = tid;
    if (c < bs) {
      if (LOWER) {
        const T d = UNIT ? T(1) : T(1) / Tb[c][c];
        Dinv[c][c] = d;
        for (int rr = c + 1; rr < bs; ++rr) {
          T sum = T(0);
          for (int qq = c; qq < rr; ++qq) sum += Tb[rr][qq] * Dinv[qq][c];
          Dinv[rr][c] = UNIT ? -sum : -sum / Tb[rr][rr];
        }
      } else {
        const T d = UNIT ? T(1) : T(1) / Tb[c][c];
        Dinv[c][c] = d;
        for (int rr = c - 1; rr >= 0; --rr) {
          T sum = T(0);
          for (int qq = rr + 1; qq <= c; ++qq) sum += Tb[rr][qq] * Dinv[qq][c];
          Dinv[rr][c] = UNIT ? -sum : -sum / Tb[rr][rr];
        }
      }
    }
  }

  // ---- off-diagonal part: thread (r, q) accumulates row r over columns
  // q*SEG .. q*SEG+SEG-1 of every predecessor block.  Per predecessor the
  // workgroup stages its solution from the exchange words into LDS (one
  // barrier); the matrix values, which do not depend on X, are prefetched
  // one predecessor ahead.
  // (kM) this thread's quarter of row r of M
  T mrow[kM ? SEG : 1];
  if constexpr (kM) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < SEG; ++i) mrow[i] = T(0);
    if (ndep > 0) {
#pragma unroll 4
      for (int k = 0; k < BS; ++k) {
        const T dk = Dinv[r][k];
#pragma unroll
        for (int i = 0; i < SEG; ++i) mrow[i] += dk * Tl[k][q * SEG + i];
      }
    }
  }
  T acc[1] = {T(0)};
  // predecessors taken in the loop (kM: all but the last)
  const int nloop = kM ? max(ndep - 1, 0) : ndep;
  const bool rvalid = r < bs;
  // the block's right-hand side, requested now: read after the loop it would
  // put a memory round trip on every link of the chain
  const T bval = (q == 0 && rvalid) ? X[rb0 + r] : T(0);
  // a row-major segment is contiguous: 16-byte loads when aligned (a quarter
  // or half of the address work of element loads, which the CU's address
  // unit otherwise limits)
  constexpr int PW = 16 / sizeof(T);  // values per 16-byte word
  const bool vec = ROWMAJOR && ((uintptr_t)A & 15) == 0 && lda % PW == 0;
  auto load_seg = [&](int d, T (&tv)[SEG]) {
    const int jb = LOWER ? d : nblk - 1 - d;
    const int cb = jb * BS + q * SEG;
    if (vec && cb + SEG <= n) {
      const T* p = tptr<T, ROWMAJOR>(A, lda, rb0 + r, cb);
#pragma unroll
      for (int i = 0; i < SEG; i += PW) {
        if (sizeof(T) == 4) {
          const v4f w = rvalid ? *reinterpret_cast<const v4f*>(p + i) : v4f{0.f, 0.f, 0.f, 0.f};
          tv[i] = (T)w.x;
          tv[i + 1] = (T)w.y;
          tv[i + 2] = (T)w.z;
          tv[i + 3] = (T)w.w;
        } else {
          typedef double v2d __attribute__((ext_vector_type(2)));
          const v2d w = rvalid ? *reinterpret_cast<const v2d*>(p + i) : v2d{0.0, 0.0};
          tv[i] = (T)w.x;
          tv[i + 1] = (T)w.y;
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < SEG; ++i)
        tv[i] = (rvalid && cb + i < n) ? *tptr<T, ROWMAJOR>(A, lda, rb0 + r, cb + i) : T(0);
    }
  };
  int bad = 0;
  // the solution of predecessor step d, from its exchange words into
  // xsw[d & 1] (my words all requested together, then only the words not
  // yet published read again), then one barrier
  auto stage = [&](int d) {
    const int jb = LOWER ? d : nblk - 1 - d;
    const int par = d & 1;
    // my words of the predecessor's solution (row, half): all
    // loads in flight together, then only the words not yet published are
    // read again
    const u64* wsrc[WPT];
    u64 wv[WPT];
    bool need[WPT];
#pragma unroll
    for (int k = 0; k < WPT; ++k) {
      const int widx = tid + k * NT;
      const int row = jb * BS + widx / NW;
      need[k] = widx < CHUNK && row < n;
      wsrc[k] = xw + (size_t)row * NW + widx % NW;
      wv[k] = need[k] ? __hip_atomic_load(const_cast<u64*>(wsrc[k]), __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT)
                      : 0ull;
      if (widx < CHUNK && !need[k]) xsw[par][widx] = 0u;
    }
    for (int spins = 0;;) {
      bool all = true;
#pragma unroll
      for (int k = 0; k < WPT; ++k)
        if (need[k]) {
          if ((unsigned)(wv[k] >> 32) == epoch) {
            xsw[par][tid + k * NT] = (unsigned)wv[k];
            need[k] = false;
          } else {
            all = false;
          }
        }
      if (all) break;
      // the limit every poll, another workgroup's give-up every 256th
      ++spins;
      if (spins > spin_limit ||
          ((spins & 255) == 0 &&
           __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
        bad = 1;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
#pragma unroll
      for (int k = 0; k < WPT; ++k)
        if (need[k])
          wv[k] = __hip_atomic_load(const_cast<u64*>(wsrc[k]), __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
    }
    if (bad) s_abort = 1;
    __syncthreads();
    if (s_abort) bad = 1;
  };
  T tcur[SEG], tnext[SEG];
  if (nloop > 0) load_seg(0, tcur);
  for (int d = 0; d < nloop && !bad; ++d) {
    if (d + 1 < nloop) load_seg(d + 1, tnext);
    const int jb = LOWER ? d : nblk - 1 - d;
    const int par = d & 1;
    stage(d);
    if (bad) break;
    const int cb = jb * BS + q * SEG;
    // (the one-pass outer loop keeps the compiler from merging the guards of
    // the products, n = 16384 in FP32: 365 us a solve, and 405 without it)
#pragma unroll
    for (int c = 0; c < 1; ++c) {
      T sum = T(0);
#pragma unroll
      for (int i = 0; i < SEG; ++i) {
        const unsigned* wp = &xsw[par][(q * SEG + i) * NW];
        T xv;
        if (NW == 2)
          xv = (T)__longlong_as_double((long long)(((u64)wp[1] << 32) | wp[0]));
        else
          xv = (T)__uint_as_float(wp[0]);
        if (cb + i < n) sum += tcur[i] * xv;
      }
      acc[c] += sum;
    }
#pragma unroll
    for (int i = 0; i < SEG; ++i) tcur[i] = tnext[i];
  }
  if (bad) {
    s_abort = 1;
    __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // the four quarters of a row sit in lanes 4r .. 4r+3 of one wave
  acc[0] += __shfl_xor(acc[0], 1);
  acc[0] += __shfl_xor(acc[0], 2);
  if (q == 0) accs[r] = rvalid ? bval - acc[0] : T(0);
  __syncthreads();
  if (s_abort) return;
  // ---- X_b = inv(T_bb) * (B_b - sum): thread (r, q) takes a quarter of the row of Dinv
  T xs = T(0);
#pragma unroll
  for (int i = 0; i < SEG; ++i) xs += Dinv[r][q * SEG + i] * accs[q * SEG + i];
  xs += __shfl_xor(xs, 1);
  xs += __shfl_xor(xs, 2);
  if constexpr (kM) {
    // X_b -= M X_l once l's solution is here: every wave polls X_l's BS
    // words itself (lane l: words l, l + 64) and publishes its own rows, so
    // no workgroup barrier sits on the chain
    if (ndep > 0) {
      constexpr int WL = BS / 64;
      const int lane = tid & 63, wv = tid >> 6;
      const u64* src[WL];
      bool need[WL];
      u64 w[WL];
#pragma unroll
      for (int k = 0; k < WL; ++k) {
        const int row = jl * BS + lane + 64 * k;
        need[k] = row < n;
        src[k] = xw + (size_t)row;
        w[k] = need[k] ? __hip_atomic_load(const_cast<u64*>(src[k]), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT)
                       : (u64)epoch << 32;
      }
      auto missing = [&]() {
        bool m = false;
#pragma unroll
        for (int k = 0; k < WL; ++k) m = m || (unsigned)(w[k] >> 32) != epoch;
        return m;
      };
      for (int spins = 0; __ballot(missing()) != 0ull;) {
        ++spins;
        if (spins > spin_limit ||
            ((spins & 255) == 0 &&
             __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
          __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          return;
        }
        __builtin_amdgcn_s_sleep(1);
#pragma unroll
        for (int k = 0; k < WL; ++k)
          if ((unsigned)(w[k] >> 32) != epoch)
            w[k] = __hip_atomic_load(const_cast<u64*>(src[k]), __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
      }
      // the wave's own LDS copy (a wave's LDS accesses execute in order)
#pragma unroll
      for (int k = 0; k < WL; ++k) xwv[wv][lane + 64 * k] = (unsigned)w[k];
      asm volatile("" ::: "memory");
      T m = T(0);
#pragma unroll
      for (int i = 0; i < SEG; ++i) m += mrow[i] * __uint_as_float(xwv[wv][q * SEG + i]);
      m += __shfl_xor(m, 1);
      m += __shfl_xor(m, 2);
      xs -= m;
    }
  }
  // publish: the result, and its exchange words for the successors
  if (q == 0 && rvalid) {
    X[rb0 + r] = xs;
    u64* dst = xw + (size_t)(rb0 + r) * NW;
    if (NW == 2) {
      const u64 bits = (u64)__double_as_longlong((double)xs);
      __hip_atomic_store(dst, ((u64)epoch << 32) | (unsigned)bits, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(dst + 1, ((u64)epoch << 32) | (unsigned)(bits >> 32), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    } else {
      __hip_atomic_store(dst, ((u64)epoch << 32) | __float_as_uint((float)xs), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

}  // namespace

// Solves op(T) X = X in place.  T is n x n; `rowmajor` selects its layout;
// lower/unit select the triangle.  X is column-major n x nrhs.  FP64 with two
// or more columns goes to the matrix-product solver: it is ahead of chains of
// four columns from the start (us, solver / chains: n = 64, 2 columns 36 / 82;
// n = 1024, 2 columns 108 / 137 and 16 columns 109 / 160; n = 8192, 4 columns
// 674 / 805 and 64 columns 822 / 4129).  FP32 columns (the refinement, which
// solves one at a time) run one chain each.
template <typename T>
int trsv_device(eamd_handle* h, int n, const T* A, int64_t lda, bool rowmajor, bool lower,
                bool unit, T* X, int64_t ldx, int nrhs) {
  if (n <= 0 || nrhs <= 0) return kOk;
  PhaseScope ps(h, kPhTrsv, sizeof(T) * (0.5 * (double)n * n + 2.0 * (double)n * nrhs),
                (double)n * n * nrhs);
  if constexpr (sizeof(T) == 8) {
    if (nrhs > 1) return trsm_blocked(h, n, A, lda, rowmajor, lower, unit, X, ldx, nrhs);
  }
  static const int spin_limit = env_int("EAMD_TRSV_SPIN", kSpin);
  // (128-row blocks measured slower: 7.4 vs 3.7 ms of FP32 solves per step at
  // n = 16384)
  constexpr int BS = 64;
  const int nblk = ceil_div(n, BS);
  // error word | exchange words (32 payload bits each)
  const size_t nwords = (size_t)nblk * BS * (sizeof(T) / 4);
  size_t need = 256 + sizeof(unsigned long long) * nwords;
  void* base = nullptr;
  bool fresh = h->ws.bytes[kWsStatus] < need;
  EAMD_CHECK(h->ws.get(kWsStatus, need, &base));
  int* err = static_cast<int*>(base);
  unsigned long long* xw =
      reinterpret_cast<unsigned long long*>(static_cast<char*>(base) + 256);
  if (fresh || h->trsv_epoch > (1 << 30)) {
    EAMD_HIP(hipMemsetAsync(base, 0, h->ws.bytes[kWsStatus], h->stream));
    h->trsv_epoch = 0;
  }
  for (int c = 0; c < nrhs; ++c) {
    const unsigned epoch = (unsigned)++h->trsv_epoch;
    T* x = X + (int64_t)c * ldx;
#define EAMD_TRSV(RM, LO, UN)                                                                 \
  hipLaunchKernelGGL((trsv_chain_kernel<T, RM, LO, UN, BS>), dim3(nblk), dim3(4 * BS), 0,     \
                     h->stream, n, A, lda, x, xw, epoch, err, spin_limit)
    if (rowmajor) {
      if (lower) { if (unit) EAMD_TRSV(true, true, true); else EAMD_TRSV(true, true, false); }
      else { if (unit) EAMD_TRSV(true, false, true); else EAMD_TRSV(true, false, false); }
    } else {
      if (lower) { if (unit) EAMD_TRSV(false, true, true); else EAMD_TRSV(false, true, false); }
      else { if (unit) EAMD_TRSV(false, false, true); else EAMD_TRSV(false, false, false); }
    }
#undef EAMD_TRSV
    EAMD_HIP(hipGetLastError());
  }
  return kOk;
}

int trsv_check_error(eamd_handle* h) {
  if (!h->ws.ptr[kWsStatus]) {
    // no chain has run: nothing to read, but the call still completes
    EAMD_HIP(hipStreamSynchronize(h->stream));
    return kOk;
  }
  int e = 0;
  EAMD_HIP(hipMemcpyAsync(&e, h->ws.ptr[kWsStatus], sizeof(int), hipMemcpyDeviceToHost,
                          h->stream));
  EAMD_HIP(hipStreamSynchronize(h->stream));
  if (e) {
    EAMD_HIP(hipMemset(h->ws.ptr[kWsStatus], 0, sizeof(int)));
    set_error("triangular solve: dependency wait timed out");
    return kErrHip;
  }
  return kOk;
}

template int trsv_device<double>(eamd_handle*, int, const double*, int64_t, bool, bool, bool,
                                 double*, int64_t, int);
template int trsv_device<float>(eamd_handle*, int, const float*, int64_t, bool, bool, bool,
                                float*, int64_t, int);

// ---------------------------------------------------------------------------
// Row interchanges of a column-major right-hand side by a transposition
// sequence (Transpositions applied in order, PermutationMatrix.h:82-88 /
// ProductEvaluators.h:927-980).  One workgroup per right-hand side column,
// the column resident in LDS (n <= kMaxLdsRows), else directly in global
// memory.  One wave takes the next 64 transpositions at a time, finds the
// first that touches a row of an earlier one (each row marked with the lowest
// lane that touches it; rows that share a mark count as the same row, which
// only shortens a step), and does those before it together: they commute.
// One after the other, a transposition was an LDS round trip and a load of its
// row: 105 us for n = 1024 and 1.68 ms for 16384, 31 and 323 us so.
namespace {
constexpr int kMaxLdsRows = 18432;
constexpr int kMarks = 1024;

template <typename T>
__global__ __launch_bounds__(256) void apply_transp_kernel(int n, const int* __restrict__ t,
                                                           int forward, T* __restrict__ X,
                                                           int64_t ldx) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ int mark[kMarks];
  T* col = reinterpret_cast<T*>(smem_raw);
  T* x = X + (int64_t)blockIdx.x * ldx;
  const bool in_lds = n <= kMaxLdsRows;
  for (int i = threadIdx.x; i < kMarks; i += 256) mark[i] = 64;
  if (in_lds)
    for (int i = threadIdx.x; i < n; i += 256) col[i] = x[i];
  __syncthreads();
  T* v = in_lds ? col : x;
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    // element j of the sequence, 64 at a time, two windows ahead
    auto window = [&](int j0) {
      const int j = j0 + lane;
      return j < n ? t[forward ? j : n - 1 - j] : 0;
    };
    int base = 0, off = 0;  // the next element is base + off
    int w0 = window(0), w1 = window(64), w2 = window(128);
    while (base + off < n) {
      const int q = off + lane, j = base + q;
      const int a = __shfl(w0, q & 63), b = __shfl(w1, q & 63);
      const int p = q < 64 ? a : b, k = forward ? j : n - 1 - j;
      const bool act = j < n && p != k;
      int* mk = &mark[k & (kMarks - 1)];
      int* mp = &mark[p & (kMarks - 1)];
      if (act) {
        atomicMin(mk, lane);
        atomicMin(mp, lane);
      }
      __threadfence_block();
      const bool conflict = act && (*(volatile int*)mk < lane || *(volatile int*)mp < lane);
      const unsigned long long m = __ballot(conflict);
      // (lane 0 conflicts with nothing, so a step takes at least one)
      int many = min(m ? __ffsll((long long)m) - 1 : 64, n - base - off);
      const bool chain = m && many < 4;
      if (act) {
        *(volatile int*)mk = 64;
        *(volatile int*)mp = 64;
        if (!chain && lane < many) {
          const T y = v[k], z = v[p];
          v[k] = z;
          v[p] = y;
        }
      }
      if (chain) {
        // neighbours that touch each other's rows (a Hessenberg matrix's
        // pivots, say): the next 32 one by one
        many = min(32, n - base - off);
        for (int e = 0; e < many; ++e) {
          const int ke = __builtin_amdgcn_readlane(k, e), pe = __builtin_amdgcn_readlane(p, e);
          if (pe != ke && lane == 0) {
            const T y = v[ke], z = v[pe];
            v[ke] = z;
            v[pe] = y;
          }
        }
      }
      __threadfence_block();
      off += many;
      if (off >= 64) {
        off -= 64;
        base += 64;
        w0 = w1;
        w1 = w2;
        w2 = window(base + 128);
      }
    }
  }
  if (in_lds) {
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 256) x[i] = col[i];
  }
}
}  // namespace

template <typename T>
int apply_transpositions(eamd_handle* h, int n, const int* t, bool forward, T* X, int64_t ldx,
                         int nrhs) {
  if (n <= 0 || nrhs <= 0) return kOk;
  size_t lds = n <= kMaxLdsRows ? sizeof(T) * (size_t)n : 0;
  auto kern = apply_transp_kernel<T>;
  EAMD_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                               150 * 1024));
  hipLaunchKernelGGL(kern, dim3(nrhs), dim3(256), lds, h->stream, n, t, forward ? 1 : 0, X, ldx);
  EAMD_HIP(hipGetLastError());
  return kOk;
}
template int apply_transpositions<double>(eamd_handle*, int, const int*, bool, double*, int64_t,
                                          int);
template int apply_transpositions<float>(eamd_handle*, int, const int*, bool, float*, int64_t,
                                         int);

}  // namespace eamd

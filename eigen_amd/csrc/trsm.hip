// trsm.hip -- triangular solves with many right-hand sides (FP64).
//
// Replaces triangular_solve_matrix (TriangularSolverMatrix.h:38-184) where
// there are enough right-hand sides for matrix products to carry the work:
// the chain of trsv.hip walks n / 64 dependent blocks for every sixteen
// columns, so 500 columns of a 2000 x 2000 triangle took 32 walks (7.1 ms).
// Here:
//   trinv64_kernel     every 64 x 64 diagonal block of T is inverted, one
//                      workgroup each, in one launch;
//   trsm_block_kernel  256 rows of X for sixteen columns per workgroup: the
//                      four 64-row steps X_i = inv(T_ii) (B_i - sum T_ij X_j)
//                      as MFMA products with X in LDS;
//   dgemm_device       the remaining rows -= T X of those 256 rows.
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace eamd {

namespace {

constexpr int SB = 64;             // rows of a diagonal block
constexpr int NBR = 256;           // rows solved per trsm_block_kernel launch
constexpr int NSUB = NBR / SB;

typedef double v2du __attribute__((ext_vector_type(2), aligned(8)));

template <bool ROWMAJOR>
__device__ __forceinline__ const double* at(const double* A, int64_t ld, int r, int c) {
  return ROWMAJOR ? A + (int64_t)r * ld + c : A + r + (int64_t)c * ld;
}

// Inverse of the 64 x 64 diagonal block blockIdx.x of T, to Dinv + 4096 b
// (row-major, zero outside its triangle and past a partial last block).  An
// upper block is turned by 180 degrees into a lower one.  The two 32 x 32
// halves of the diagonal are inverted by the two halves of wave 0, lane j
// forming column j in registers; the rest is X21 = -X22 (T21 X11) on MFMA, a
// 16 x 16 tile per wave.
template <bool ROWMAJOR, bool LOWER, bool UNIT>
__global__ __launch_bounds__(256) void trinv64_kernel(int n, const double* __restrict__ A,
                                                      int64_t lda, double* __restrict__ Dinv) {
  constexpr int LD = SB + 1;
  __shared__ double S[SB * LD];    // T (lower form), row-major
  __shared__ double X[SB * LD];    // its inverse
  __shared__ double Y[32 * 33];    // T21 X11
  const int b = blockIdx.x, r0 = b * SB, bs = min(SB, n - r0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int q = 0; q < SB * SB / 256; ++q) {
    // consecutive threads along the contiguous direction
    const int e = tid + 256 * q;
    const int r = ROWMAJOR ? e / SB : e % SB, c = ROWMAJOR ? e % SB : e / SB;
    const bool in = r < bs && c < bs && (LOWER ? r >= c : r <= c);
    const double v = in ? *at<ROWMAJOR>(A, lda, r0 + r, r0 + c) : 0.0;
    // lower form: the block's own rows and columns turned, padding behind
    // them with a unit diagonal
    const int rr = (LOWER || r >= bs) ? r : bs - 1 - r, cc = (LOWER || c >= bs) ? c : bs - 1 - c;
    S[rr * LD + cc] = r == c && (UNIT || r >= bs) ? 1.0 : v;
    X[rr * LD + cc] = 0.0;
  }
  __syncthreads();
  if (wave == 0) {
    const int h = lane & 32, j = lane & 31;
    const double* T = S + h * LD + h;
    double x[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      double sp[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < i; ++k) sp[(i - 1 - k) & 3] += T[i * LD + k] * x[k];
      const double s = (sp[0] + sp[1]) + (sp[2] + sp[3]);
      const double num = i == j ? 1.0 : -s;
      x[i] = i < j ? 0.0 : (UNIT ? num : num / T[i * LD + i]);
      asm volatile("" ::: "memory");  // the next row's LDS reads stay behind (registers)
    }
#pragma unroll
    for (int i = 0; i < 32; ++i) X[(h + i) * LD + h + j] = x[i];
  }
  __syncthreads();
  const int ti = (wave & 1) * 16, tj = (wave >> 1) * 16;
  {
    v4d a[4] = {};
#pragma unroll
    for (int k = 0; k < 32; k += 4)
      a[k / 8] = __builtin_amdgcn_mfma_f64_16x16x4f64(S[(32 + ti + l16) * LD + k + lk],
                                                      X[(k + lk) * LD + tj + l16], a[k / 8], 0, 0, 0);
    const v4d acc = (a[0] + a[1]) + (a[2] + a[3]);
#pragma unroll
    for (int r = 0; r < 4; ++r) Y[(ti + lk + 4 * r) * 33 + tj + l16] = acc[r];
  }
  __syncthreads();
  {
    v4d a[4] = {};
#pragma unroll
    for (int k = 0; k < 32; k += 4)
      a[k / 8] = __builtin_amdgcn_mfma_f64_16x16x4f64(-X[(32 + ti + l16) * LD + 32 + k + lk],
                                                      Y[(k + lk) * 33 + tj + l16], a[k / 8], 0, 0, 0);
    const v4d acc = (a[0] + a[1]) + (a[2] + a[3]);
#pragma unroll
    for (int r = 0; r < 4; ++r) X[(32 + ti + lk + 4 * r) * LD + tj + l16] = acc[r];
  }
  __syncthreads();
  double* D = Dinv + (int64_t)b * SB * SB;
#pragma unroll
  for (int q = 0; q < SB * SB / 256; ++q) {
    const int e = tid + 256 * q, r = e / SB, c = e % SB;
    const bool in = r < bs && c < bs;
    const int rr = LOWER ? r : bs - 1 - r, cc = LOWER ? c : bs - 1 - c;
    D[e] = in ? X[rr * LD + cc] : 0.0;
  }
}

// X[r0 .. r0 + 256) <- T^-1 X of that diagonal block for sixteen columns per
// workgroup.  Wave w owns rows 16 w .. 16 w + 15 of each 64-row step; T's
// values do not depend on X, so a step's are requested before the previous
// step's inverse product.  In a run of 16 of the inner dimension lane group
// lk takes four consecutive k (32 contiguous bytes of a row-major T and of
// the inverses).  One launch is latency: ten 64 x 64 x 16 products and eight
// barriers.
constexpr int XLD = 20;  // LDS row stride of X: rows four apart on disjoint banks
template <bool ROWMAJOR, bool LOWER>
__global__ __launch_bounds__(256) void trsm_block_kernel(int n, const double* __restrict__ A,
                                                         int64_t lda,
                                                         const double* __restrict__ Dinv,
                                                         double* __restrict__ X, int64_t ldx,
                                                         int nrhs, int r0) {
  __shared__ __align__(16) double Xs[NBR * XLD];
  __shared__ __align__(16) double Ys[SB * XLD];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lk = lane >> 4;
  const int c0 = blockIdx.x * 16, nc = min(16, nrhs - c0);
  const int rows = min(NBR, n - r0), nsub = (rows + SB - 1) / SB;
  // thread: row tid of every column
  {
    double v[16];
    const double* xp = X + (int64_t)c0 * ldx + r0 + tid;
#pragma unroll
    for (int c = 0; c < 16; ++c)
      v[c] = (tid < rows && c < nc) ? xp[(int64_t)c * ldx] : 0.0;
#pragma unroll
    for (int c = 0; c < 16; ++c) Xs[tid * XLD + c] = v[c];
  }
  // sub-block of solve step d
  auto sub = [&](int d) { return LOWER ? d : nsub - 1 - d; };
  double t[NSUB - 1][SB / 4];  // T(my rows, the 64 columns of each earlier step)
  auto load_t = [&](int d) {
    const int rb = r0 + sub(d) * SB;
    const int row = min(rb + wave * 16 + l16, n - 1);  // rows past n are not stored
#pragma unroll
    for (int e = 0; e < NSUB - 1; ++e) {
      if (e >= d) break;
      const int cb = r0 + sub(e) * SB;
#pragma unroll
      for (int u = 0; u < SB / 16; ++u) {
        const int k = cb + u * 16 + lk * 4;
        if (ROWMAJOR && cb + SB <= n) {
          const double* p = at<true>(A, lda, row, k);
#pragma unroll
          for (int j = 0; j < 4; j += 2) {
            const v2du w = *reinterpret_cast<const v2du*>(p + j);
            t[e][u * 4 + j] = w.x;
            t[e][u * 4 + j + 1] = w.y;
          }
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const double v = *at<ROWMAJOR>(A, lda, row, min(k + j, n - 1));
            t[e][u * 4 + j] = k + j < n ? v : 0.0;
          }
        }
      }
    }
  };
  // 16 rows of a 64 x 64 block times 64 rows of X or Y: four sums of 16
  // products each, so that a result carries the rounding of short sums (one
  // chain of 32 products in each of two sums: 1.40e-16 off exact results at
  // n = 200 .. 700, and 1.29e-16 so) and a product waits for every fourth
  auto product = [&](const double (&m)[SB / 4], const double* xb) {
    v4d a[4] = {};
#pragma unroll
    for (int u = 0; u < SB / 16; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        a[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(m[u * 4 + j], xb[(u * 16 + j) * XLD], a[j], 0,
                                                    0, 0);
    return (a[0] + a[1]) + (a[2] + a[3]);
  };
  load_t(0);
  __syncthreads();
#pragma unroll
  for (int d = 0; d < NSUB; ++d) {
    if (d >= nsub) break;
    const int s = sub(d), rb = s * SB;
    // this step's inverse rows
    double di[SB / 4];
    const double* dp = Dinv + (int64_t)(r0 / SB + s) * SB * SB + (wave * 16 + l16) * SB + lk * 4;
#pragma unroll
    for (int u = 0; u < SB / 16; ++u)
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const v2du w = *reinterpret_cast<const v2du*>(dp + u * 16 + j);
        di[u * 4 + j] = w.x;
        di[u * 4 + j + 1] = w.y;
      }
    v4d acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int e = 0; e < NSUB - 1; ++e) {
      if (e >= d) break;
      acc += product(t[e], Xs + (sub(e) * SB + lk * 4) * XLD + l16);
    }
    if (d + 1 < NSUB && d + 1 < nsub) load_t(d + 1);
    // lane (lk, l16) register r: row lk + 4 r, column l16 of the wave's tile
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = wave * 16 + lk + 4 * r;
      const double y = Xs[(rb + row) * XLD + l16] - acc[r];
      Ys[row * XLD + l16] = rb + row < rows ? y : 0.0;
    }
    __syncthreads();
    const v4d x = product(di, Ys + lk * 4 * XLD + l16);
#pragma unroll
    for (int r = 0; r < 4; ++r) Xs[(rb + wave * 16 + lk + 4 * r) * XLD + l16] = x[r];
    __syncthreads();
  }
  double* xp = X + (int64_t)c0 * ldx + r0 + tid;
#pragma unroll
  for (int c = 0; c < 16; ++c)
    if (tid < rows && c < nc) xp[(int64_t)c * ldx] = Xs[tid * XLD + c];
}

template <bool ROWMAJOR, bool LOWER>
int solve(eamd_handle* h, int n, const double* A, int64_t lda, bool unit, double* X, int64_t ldx,
          int nrhs) {
  hipStream_t s = h->stream;
  const int nblk = ceil_div(n, SB), nout = ceil_div(n, NBR);
  void* dp = nullptr;
  EAMD_CHECK(h->ws.get(kWsTri, sizeof(double) * SB * SB * (size_t)nblk, &dp));
  double* Dinv = static_cast<double*>(dp);
  if (unit)
    hipLaunchKernelGGL((trinv64_kernel<ROWMAJOR, LOWER, true>), dim3(nblk), dim3(256), 0, s, n, A,
                       lda, Dinv);
  else
    hipLaunchKernelGGL((trinv64_kernel<ROWMAJOR, LOWER, false>), dim3(nblk), dim3(256), 0, s, n,
                       A, lda, Dinv);
  for (int o = 0; o < nout; ++o) {
    const int r0 = (LOWER ? o : nout - 1 - o) * NBR, rows = std::min(NBR, n - r0);
    hipLaunchKernelGGL((trsm_block_kernel<ROWMAJOR, LOWER>), dim3(ceil_div(nrhs, 16)), dim3(256),
                       0, s, n, A, lda, (const double*)Dinv, X, ldx, nrhs, r0);
    // the rows still to be solved: T(rest, block) X(block)
    const int q0 = LOWER ? r0 + rows : 0, qn = LOWER ? n - q0 : r0;
    const double* T = ROWMAJOR ? A + (int64_t)q0 * lda + r0 : A + q0 + (int64_t)r0 * lda;
    EAMD_CHECK(dgemm_device(s, ROWMAJOR, false, qn, nrhs, rows, -1.0, T, lda, X + r0, ldx, 1.0,
                            X + q0, ldx, 0));
  }
  EAMD_HIP(hipGetLastError());
  return kOk;
}

}  // namespace

int trsm_blocked(eamd_handle* h, int n, const double* A, int64_t lda, bool rowmajor, bool lower,
                 bool unit, double* X, int64_t ldx, int nrhs) {
  if (rowmajor)
    return lower ? solve<true, true>(h, n, A, lda, unit, X, ldx, nrhs)
                 : solve<true, false>(h, n, A, lda, unit, X, ldx, nrhs);
  return lower ? solve<false, true>(h, n, A, lda, unit, X, ldx, nrhs)
               : solve<false, false>(h, n, A, lda, unit, X, ldx, nrhs);
}

}  // namespace eamd

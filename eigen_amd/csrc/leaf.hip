// leaf.hip -- the partial-pivoting column loop of the LU panel.
//
// Restates unblocked_lu (Eigen/src/LU/PartialPivLU.h:365-409) for a leaf of
// at most 32 columns of a tall row-major sub-panel: per column, the first
// maximum of |a| (strict '>' scan in row order, Visitor.h:179; a NaN wins only
// from the diagonal position), the row interchange, the division of the
// column by the pivot and the rank-1 update of the leaf.
//
// MI355X mapping.  Every thread keeps one row of the leaf (32 values) in
// registers, so the rank-1 update is register FMAs; a workgroup holds 1024
// rows (512 in FP64 when that is the whole leaf), and at most 32 (FP64: 16)
// workgroups take part.  With several workgroups, each column costs ONE memory
// round trip: every workgroup publishes its candidate (value, row) together
// with the whole candidate row, and the owner of row j publishes row j, all
// as 8-byte words carrying 32 bits of payload and the column's epoch (an
// aligned 8-byte store is single-copy atomic, so a word with the right epoch
// has the right payload: no fences).  Every workgroup then reads all
// candidates and row j in one parallel poll and resolves the winner locally.
#include <type_traits>
#include <utility>

#include "common.h"
#include "kernels.h"

namespace eamd {

namespace {

constexpr int LW = 32;       // leaf width
constexpr int kMaxG = 32;    // workgroups in the exchange
constexpr int kLeafSpin = 1 << 22;
typedef unsigned long long u64;

template <typename T>
struct Words {
  static constexpr int n = sizeof(T) / 4;  // 32-bit payload words per value
};

__device__ __forceinline__ void put_word(u64* p, unsigned payload, unsigned epoch) {
  __hip_atomic_store(p, ((u64)epoch << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T>
__device__ __forceinline__ void put_value(u64* p, T v, unsigned epoch) {
  if (sizeof(T) == 8) {
    u64 bits = (u64)__double_as_longlong((double)v);
    put_word(p, (unsigned)bits, epoch);
    put_word(p + 1, (unsigned)(bits >> 32), epoch);
  } else {
    put_word(p, __float_as_uint((float)v), epoch);
  }
}

// Bit-mask selection (a ? x : y with a mask of all ones or zeros).  Written
// on the integer bits so the compiler does not fold a chain of them back
// into a runtime-indexed access of the register array (which it would place
// in scratch memory).
__device__ __forceinline__ float mask_sel(unsigned m, float x, float y) {
  return __uint_as_float((__float_as_uint(x) & m) | (__float_as_uint(y) & ~m));
}

template <typename T>
__device__ __forceinline__ T get_value(const unsigned* w) {
  if (sizeof(T) == 8) return (T)__longlong_as_double((long long)(((u64)w[1] << 32) | w[0]));
  return (T)__uint_as_float(w[0]);
}

__device__ __forceinline__ bool beats(double s, int i, double bs, int bi) {
  return s > bs || (s == bs && i < bi);
}

__device__ __forceinline__ double score_of(double v, bool first) {
  double s = fabs(v);
  if (s != s) s = first ? INFINITY : -1.0;
  return s;
}

// Rotation of a register row by 8 slots (compile-time moves): the column
// loops work on groups of 8 columns that always sit in slots 0..7, so every
// register access has a compile-time index; after 4 rotations the row is back
// in its original order.
template <typename T>
__device__ __forceinline__ void rotate8(T (&v)[32]) {
  T t[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) t[q] = v[q];
#pragma unroll
  for (int c = 0; c < 24; ++c) v[c] = v[c + 8];
#pragma unroll
  for (int q = 0; q < 8; ++q) v[24 + q] = t[q];
}

// Lane permutations of the DPP unit, applied to a double as two halves.
template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double((long long)(((u64)(unsigned)hi << 32) | (unsigned)lo));
}

__device__ __forceinline__ double readlane_d(double x, int lane) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)b, lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double((long long)(((u64)(unsigned)hi << 32) | (unsigned)lo));
}

// Maximum over the 64 lanes of a wave (inputs never NaN): xor-1 and xor-2
// within quads, half-row and row mirrors within each 16-lane row, then the
// four row results read as uniform values.
__device__ __forceinline__ double wave_max(double s) {
  s = fmax(s, dpp_d<0xB1>(s));   // quad_perm [1,0,3,2]
  s = fmax(s, dpp_d<0x4E>(s));   // quad_perm [2,3,0,1]
  s = fmax(s, dpp_d<0x141>(s));  // row_half_mirror
  s = fmax(s, dpp_d<0x140>(s));  // row_mirror
  return fmax(fmax(readlane_d(s, 0), readlane_d(s, 16)), fmax(readlane_d(s, 32), readlane_d(s, 48)));
}

// Maximum of a 64-bit key over the 64 lanes of a wave (same lane pattern).
template <int CTRL>
__device__ __forceinline__ u64 dpp_u64(u64 x) {
  const int lo = __builtin_amdgcn_mov_dpp((int)x, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(x >> 32), CTRL, 0xf, 0xf, false);
  return ((u64)(unsigned)hi << 32) | (unsigned)lo;
}
__device__ __forceinline__ u64 readlane_u64(u64 x, int lane) {
  const int lo = __builtin_amdgcn_readlane((int)x, lane);
  const int hi = __builtin_amdgcn_readlane((int)(x >> 32), lane);
  return ((u64)(unsigned)hi << 32) | (unsigned)lo;
}
__device__ __forceinline__ u64 umax64(u64 a, u64 b) { return a > b ? a : b; }
__device__ __forceinline__ u64 wave_max_u64(u64 k) {
  k = umax64(k, dpp_u64<0xB1>(k));
  k = umax64(k, dpp_u64<0x4E>(k));
  k = umax64(k, dpp_u64<0x141>(k));
  k = umax64(k, dpp_u64<0x140>(k));
  return umax64(umax64(readlane_u64(k, 0), readlane_u64(k, 16)),
                umax64(readlane_u64(k, 32), readlane_u64(k, 48)));
}

// Slot (words): [0..1] candidate value (FP64 bits), [2] row or ~0u (no
// candidate), [3] unused, [4, 4 + LW*Words) candidate row.  The slot after
// the last workgroup's holds row j (from word 4).
template <typename T>
constexpr int slot_words() {
  return 4 + LW * Words<T>::n;
}

__device__ __forceinline__ int readlane_i(int x, int lane) {
  return __builtin_amdgcn_readlane(x, lane);
}
__device__ __forceinline__ float readlane_f(float x, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// Maximum of a 32-bit key over the 64 lanes of a wave: xor-1 and xor-2
// within quads, half-row and row mirrors within each 16-lane row, then the
// row maxima are carried into lane 63 (row_bcast:15 into rows 1 and 3,
// row_bcast:31 into rows 2 and 3).
__device__ __forceinline__ unsigned wave_max_u32(unsigned k) {
  k = max(k, (unsigned)__builtin_amdgcn_mov_dpp((int)k, 0xB1, 0xf, 0xf, false));
  k = max(k, (unsigned)__builtin_amdgcn_mov_dpp((int)k, 0x4E, 0xf, 0xf, false));
  k = max(k, (unsigned)__builtin_amdgcn_mov_dpp((int)k, 0x141, 0xf, 0xf, false));
  k = max(k, (unsigned)__builtin_amdgcn_mov_dpp((int)k, 0x140, 0xf, 0xf, false));
  k = max(k, (unsigned)__builtin_amdgcn_update_dpp((int)k, (int)k, 0x142, 0xa, 0xf, false));
  k = max(k, (unsigned)__builtin_amdgcn_update_dpp((int)k, (int)k, 0x143, 0xc, 0xf, false));
  return (unsigned)readlane_i((int)k, 63);
}

// The leaf-level permutation of a leaf's row interchanges, in registers (one
// wave): entry k (lane k < n) is leaf row pos, which receives the content of
// entry src and so holds original row row (rows 0..w-1 are entries 0..w-1,
// rows swapped in from below are appended).
struct LeafPerm {
  int pos, row, src, n;
  __device__ __forceinline__ void start(int w, int lane) {
    pos = lane < w ? lane : -1;
    row = pos;
    src = lane;
    n = w;
  }
  // Column c's interchange with entry k, the entry of position p (FROM_SEL: of
  // original row p); an untouched row p (>= w) sits at position p and becomes
  // a new entry (*fresh).
  template <bool FROM_SEL>
  __device__ __forceinline__ int step(int c, int p, int lane, bool* fresh = nullptr) {
    const u64 hit = __ballot((FROM_SEL ? row : pos) == p);
    int k;
    if (hit) {
      k = __ffsll((long long)hit) - 1;
    } else {
      k = n++;
      if (lane == k) { pos = p; row = p; src = k; }
    }
    if (fresh) *fresh = !hit;
    const int rc = readlane_i(row, c), rk = readlane_i(row, k);
    const int sc = readlane_i(src, c), sk = readlane_i(src, k);
    if (lane == c) { row = rk; src = sk; }
    if (lane == k) { row = rc; src = sc; }
    return k;
  }
};

// Composes a leaf's list (lane k < ln: leaf row tpos receives the content of
// entry tsrc) into the panel-level list ppos/psrc/pperm_n (the leaf starts at
// panel row row0; panel rows 0..pnb-1 are slots 0..pnb-1, rows below them are
// appended slots; slot s: row ppos[s] receives the content of slot psrc[s]).
// All entries at once: a touched slot's new source is the old source of its
// entry's source slot, and a newly appended slot's old source is itself.
// The panel's first leaf (row0 == 0) starts the list as the identity.  One
// wave; s_pp is LDS scratch of at least pnb + 4 ints.
__device__ void panel_compose(int tpos, int tsrc, int ln, int row0, int pnb, int lane,
                              int* pperm_n, int* ppos, int* psrc, int* s_pp) {
  const bool first = row0 == 0;
  if (first) {
    for (int e = lane; e < pnb; e += 64) {
      ppos[e] = e;
      psrc[e] = e;
    }
    // complete before the touched slots are stored over them
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  const int pn0 = first ? pnb : *pperm_n, na = pn0 - pnb, na4 = (na + 3) & ~3;
  for (int e = lane; e < na4; e += 64) s_pp[e] = e < na ? ppos[pnb + e] : -1;
  asm volatile("" ::: "memory");  // LDS accesses of one wave execute in order
  const bool mine = lane < ln;
  const int prow = row0 + tpos;
  int slot = prow;
  bool need = false;
  if (mine && prow >= pnb) {
    int f = -1;
    for (int e = 0; e < na4; e += 4) {
      const int4 q = *reinterpret_cast<const int4*>(&s_pp[e]);
      f = q.x == prow ? pnb + e : f;
      f = q.y == prow ? pnb + e + 1 : f;
      f = q.z == prow ? pnb + e + 2 : f;
      f = q.w == prow ? pnb + e + 3 : f;
    }
    slot = f;
    need = f < 0;
  }
  const u64 nb = __ballot(need);
  if (need) slot = pn0 + __popcll(nb & ((1ull << lane) - 1ull));
  int old = slot;
  if (mine && !need && !first) old = psrc[slot];
  const int src_old = __shfl(old, tsrc);
  if (mine) {
    psrc[slot] = src_old;
    if (need) ppos[slot] = prow;
  }
  if (lane == 0) *pperm_n = pn0 + __popcll(nb);
}

// All lists of a leaf from its interchanges (one wave; lane c < w: x = the row
// swapped with row c): piv[] (plus piv_offset), the leaf-level list
// lperm_n/lpos/lsrc and the panel-level one.
__device__ void leaf_lists(int x, int w, int row0, int pnb, int lane, int* piv, int piv_offset,
                           int* lperm_n, int* lpos, int* lsrc, int* pperm_n, int* ppos,
                           int* psrc, int* s_pp) {
  LeafPerm lp;
  lp.start(w, lane);
  for (int c = 0; c < w; ++c) lp.step<false>(c, readlane_i(x, c), lane);
  if (lane < w) piv[lane] = x + piv_offset;
  if (lane < lp.n) {
    lpos[lane] = lp.pos;
    lsrc[lane] = lp.src;
  }
  if (lane == 0) *lperm_n = lp.n;
  panel_compose(lp.pos, lp.src, lp.n, row0, pnb, lane, pperm_n, ppos, psrc, s_pp);
}

}  // namespace

// Outputs: piv[c] leaf-relative transposition of leaf column c; leaf
// permutation lists (rows touched, leaf-relative) lperm_n/lpos/lsrc; the
// panel-level lists pperm_n/ppos/psrc (panel-relative rows, composed across
// the leaves of a panel: on entry they hold the permutation of the previous
// leaves; `row0` is the leaf's first row inside the panel, `pnb` the panel
// width); zero_col the first exactly-zero pivot column of the leaf or -1.
// piv[] is stored plus piv_offset, and a zero pivot is also recorded in
// *fz_global (nullable) as first_zero + piv_offset when that is still < 0.
template <typename T, int BLOCK>
__global__ __launch_bounds__(BLOCK) void leaf_lu_kernel(
    T* __restrict__ P, int64_t ldp, int m, int w, int G, int* __restrict__ piv,
    int* __restrict__ lperm_n, int* __restrict__ lpos, int* __restrict__ lsrc,
    int* __restrict__ pperm_n, int* __restrict__ ppos, int* __restrict__ psrc, int row0,
    int pnb, int* __restrict__ zero_col, u64* __restrict__ xbuf, int* __restrict__ err,
    unsigned epoch_base, int piv_offset, int* __restrict__ fz_global, int spin_limit) {
  __builtin_amdgcn_s_setprio(3);  // on the critical path (see tsl_kernel)
  constexpr int NW = Words<T>::n;
  constexpr int SW = slot_words<T>();
  constexpr int NWAVE = BLOCK / 64;
  constexpr int STAGE = (kMaxG + 1) * SW;
  constexpr int KMAX = (STAGE + BLOCK - 1) / BLOCK;  // words polled per thread
  // per column, double-buffered by parity (one barrier per column): each
  // wave's best score, row index, value and row, and row j when owned here
  __shared__ double red_s[2][NWAVE];
  __shared__ int red_i[2][NWAVE];
  __shared__ double red_v[2][NWAVE];
  __shared__ T candw[2][NWAVE][LW];
  __shared__ T urow[2][LW];   // pivot row received from the exchange
  __shared__ T rowj[2][LW];   // old row j received from the exchange
  __shared__ T rowjL[2][LW];  // row j, when this workgroup owns it
  __shared__ unsigned stage[STAGE];
  __shared__ int s_abort;
  __shared__ int s_win[2];  // the exchange's winning row, by column parity
  // bookkeeping (workgroup 0): the leaf's pivots and the panel list's rows
  __shared__ int s_piv[LW];
  __shared__ __align__(16) int s_pp[256 + 4];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = blockIdx.x;
  const int i = g * BLOCK + tid;  // my leaf-relative row
  const bool valid = i < m;

  T v[LW];
  {
    const T* src = P + (int64_t)i * ldp;
#pragma unroll
    for (int c = 0; c < LW; ++c) v[c] = (valid && c < w) ? src[c] : T(0);
  }
  if (tid == 0) s_abort = 0;
  __syncthreads();

  int first_zero = -1;
  // A runtime column loop over a register row: every access to v[] uses a
  // compile-time index, with the column selected by branch-free selects and
  // masked FMAs (a runtime index into a register array would go to scratch
  // memory; a fully unrolled loop overflows the instruction cache).
  // Columns in groups of 8 that sit in register slots 0..7 (see rotate8):
  // column j = 8*g8 + jj is slot jj, a compile-time index; slots [live, 32)
  // hold columns finished in earlier groups and take no update.
  auto column = [&](auto jjc, int j, int live) __attribute__((always_inline)) -> bool {
    constexpr int jj = decltype(jjc)::value;
    const int par = j & 1;
    const unsigned epoch = epoch_base + (unsigned)j + 1u;
    const T vj = v[jj];
    // ---- 1. my candidate, the wave's (maximum score, then the lowest lane
    // holding it: lanes are in row order), then the workgroup's
    double sc = -2.0;
    if (valid && i >= j) sc = score_of((double)vj, i == j);
    const double wmax = wave_max(sc);
    const int wl = __ffsll((long long)__ballot(sc == wmax)) - 1;
    // the wave's candidate lane also stores its row, and the owner of row j
    // stores that row, before the column's single barrier
    if (lane == wl) {
      red_s[par][wave] = wmax;
      red_i[par][wave] = wmax > -2.0 ? g * BLOCK + wave * 64 + wl : 0x7fffffff;
      red_v[par][wave] = (double)vj;
#pragma unroll
      for (int c = 0; c < LW; ++c) candw[par][wave][c] = v[c];
    }
    if (i == j) {
#pragma unroll
      for (int c = 0; c < LW; ++c) rowjL[par][c] = v[c];
    }
    __syncthreads();
    double best = red_s[par][0];
    int bq = 0;
#pragma unroll
    for (int q = 1; q < NWAVE; ++q) {
      const double s2 = red_s[par][q];
      if (s2 > best) { best = s2; bq = q; }
    }
    const int bi = red_i[par][bq];
    const double bval = red_v[par][bq];
    // ---- 2. the workgroup's candidate row is the winning wave's
    const bool none = bi == 0x7fffffff;
    const T* up = candw[par][bq];  // pivot row
    const T* rp = rowjL[par];      // old row j
    int p = bi;
    if (G > 1) {
      // ---- 3. publish: header, candidate row and (owner) row j, one word per lane
      u64* myslot = xbuf + ((size_t)par * (G + 1) + g) * SW;
      u64* rj = xbuf + ((size_t)par * (G + 1) + G) * SW;
      if (tid == 0) {
        u64 bits = (u64)__double_as_longlong(bval);
        put_word(myslot, (unsigned)bits, epoch);
        put_word(myslot + 1, (unsigned)(bits >> 32), epoch);
        put_word(myslot + 2, none ? 0xffffffffu : (unsigned)bi, epoch);
        put_word(myslot + 3, 0u, epoch);
      } else if (tid >= 64 && tid < 64 + LW * NW) {
        const int q = tid - 64, c = q / NW, half = q - c * NW;
        const T val = none ? T(0) : up[c];
        unsigned pl;
        if (sizeof(T) == 8) {
          u64 bits = (u64)__double_as_longlong((double)val);
          pl = half ? (unsigned)(bits >> 32) : (unsigned)bits;
        } else {
          pl = __float_as_uint((float)val);
        }
        put_word(myslot + 4 + q, pl, epoch);
      } else if (j >= g * BLOCK && j < (g + 1) * BLOCK && tid >= 128 && tid < 128 + 4 + LW * NW) {
        const int q = tid - 128;
        unsigned pl = 0;
        if (q >= 4) {
          const int c = (q - 4) / NW, half = (q - 4) - c * NW;
          const T val = rowjL[par][c];
          if (sizeof(T) == 8) {
            u64 bits = (u64)__double_as_longlong((double)val);
            pl = half ? (unsigned)(bits >> 32) : (unsigned)bits;
          } else {
            pl = __float_as_uint((float)val);
          }
        }
        put_word(rj + q, pl, epoch);
      }
      // ---- 4. one parallel poll of every slot and of row j: each thread
      // issues the loads of its words together, then re-polls the missing ones
      const int total = (G + 1) * SW;
      const u64* base = xbuf + (size_t)par * (G + 1) * SW;
      bool done[KMAX];
#pragma unroll
      for (int k = 0; k < KMAX; ++k) done[k] = tid + k * BLOCK >= total;
      int bad = 0;
      for (int spins = 0;; ++spins) {
        u64 wv[KMAX];
#pragma unroll
        for (int k = 0; k < KMAX; ++k)
          if (!done[k])
            wv[k] = __hip_atomic_load(const_cast<u64*>(base + tid + k * BLOCK), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
        bool all = true;
#pragma unroll
        for (int k = 0; k < KMAX; ++k)
          if (!done[k]) {
            if ((unsigned)(wv[k] >> 32) == epoch) {
              stage[tid + k * BLOCK] = (unsigned)wv[k];
              done[k] = true;
            } else {
              all = false;
            }
          }
        if (all) break;
        // the limit every poll, another workgroup's give-up every 256th
        if (spins >= spin_limit ||
            ((spins & 255) == 255 &&
             __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
          bad = 1;
          break;
        }
      }
      if (bad) s_abort = 1;
      __syncthreads();
      if (s_abort) {
        if (tid == 0) __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
      }
      // ---- resolve the winner: wave 0, lane s holding slot s's candidate;
      // the highest score, then the lowest row among those (the `beats`
      // order), by two wave reductions
      if (wave == 0) {
        double sc = -2.0;
        int idx = 0x7fffffff;
        if (lane < G) {
          const unsigned* hh = &stage[lane * SW];
          const unsigned id = hh[2];
          if (id != 0xffffffffu) {
            sc = score_of(get_value<double>(hh), (int)id == j);
            idx = (int)id;
          }
        }
        const double mx = wave_max(sc);
        const int wi = (int)-wave_max(sc == mx ? -(double)idx : -4294967296.0);
        const int wslot = __ffsll((long long)__ballot(sc == mx && idx == wi)) - 1;
        if (lane < LW) {
          urow[par][lane] = get_value<T>(&stage[wslot * SW + 4 + lane * NW]);
          rowj[par][lane] = get_value<T>(&stage[G * SW + 4 + lane * NW]);
        }
        if (lane == 0) s_win[par] = wi;
      }
      __syncthreads();
      p = s_win[par];
      up = urow[par];
      rp = rowj[par];
    }
    // ---- 5. interchange in registers
    if (p != j) {
      if (i == j) {
#pragma unroll
        for (int c = 0; c < LW; ++c) v[c] = up[c];
      } else if (i == p) {
#pragma unroll
        for (int c = 0; c < LW; ++c) v[c] = rp[c];
      }
    }
    if (g == 0 && tid == 0) s_piv[j] = p;
    // ---- 6. scale and rank-1 update of the rows below j
    // branch-free (a branch around the register row makes the compiler copy
    // the whole row at the join); l = 0 leaves a row unchanged
    const T pv = up[jj];
    if (pv == T(0) && first_zero < 0) first_zero = j;
    const bool act = pv != T(0) && valid && i > j;
    const T qv = (i == p ? rp[jj] : vj) / pv;
    T l = act ? qv : T(0);
    asm volatile("" : "+v"(l));  // keep the update unconditional
    v[jj] = act ? l : v[jj];
    const unsigned lm = 0u - (unsigned)(live > 8), lm16 = 0u - (unsigned)(live > 16),
                   lm24 = 0u - (unsigned)(live > 24);
#pragma unroll
    for (int c = jj + 1; c < LW; ++c) {
      // slot c is live iff c < live; an integer mask on the loaded value keeps
      // the LDS reads unconditional
      const unsigned m = c < 8 ? ~0u : (c < 16 ? lm : (c < 24 ? lm16 : lm24));
      const T u = mask_sel(m, up[c], T(0));
      v[c] -= l * u;
    }
    return true;
  };
  const int ngroups = (w + 7) / 8;
  bool ok = true;
#pragma unroll 1
  for (int g8 = 0; g8 < ngroups && ok; ++g8) {
    const int live = LW - 8 * g8, j0 = 8 * g8;
#define EAMD_COL(JJ)                                                                   \
    if (ok && j0 + JJ < w) ok = column(std::integral_constant<int, JJ>{}, j0 + JJ, live);
    EAMD_COL(0) EAMD_COL(1) EAMD_COL(2) EAMD_COL(3) EAMD_COL(4) EAMD_COL(5) EAMD_COL(6)
    EAMD_COL(7)
#undef EAMD_COL
    rotate8(v);
  }
#pragma unroll 1
  for (int r = ngroups; r < 4; ++r) rotate8(v);
  if (s_abort) {
    // gave up (another workgroup's words never came; the call reports a
    // time-out): empty permutation lists and no zero pivot, so the kernels
    // that apply the lists after this leaf do nothing instead of indexing
    // rows with stale entries.  Workgroup 0 always takes this path when any
    // workgroup does (it needs every workgroup's words for each column).
    if (g == 0 && tid == 0) {
      *lperm_n = 0;
      *pperm_n = 0;
      *zero_col = -1;
    }
    return;
  }
  __syncthreads();
  // ---- bookkeeping (workgroup 0, wave 0): the leaf-level and panel-level
  // permutation lists, replaying the interchanges in column order
  if (g == 0 && wave == 0) {
    leaf_lists(lane < w ? s_piv[lane] : 0, w, row0, pnb, lane, piv, piv_offset, lperm_n, lpos,
               lsrc, pperm_n, ppos, psrc, s_pp);
  }
  if (valid) {
    T* dst = P + (int64_t)i * ldp;
#pragma unroll
    for (int c = 0; c < LW; ++c)
      if (c < w) dst[c] = v[c];
  }
  if (g == 0 && tid == 0) {
    *zero_col = first_zero;
    if (fz_global && first_zero >= 0 && *fz_global < 0) *fz_global = first_zero + piv_offset;
  }
}


// ---------------------------------------------------------------------------
// The FP64 leaf.  Same outputs and pivots as leaf_lu_kernel; what differs is
// what a column costs (a 512-row leaf 82 -> 34 us, 1024 rows 133 -> 57 us,
// 16384 rows 172 -> 112 us).  A thread holds one row (R = 1); up to 512 rows
// take 512 threads and up to 1024 rows 1024, without an exchange, and 16384
// rows sixteen such workgroups.  (Two rows on each of half the threads: 59 us
// for 1024 rows.)  Rows never move: an interchange
// relabels two positions, and each row is stored at its final position at the
// end, so row j needs no publishing and nothing is selected by register masks.
// The pivot search reduces the high words of |a| by DPP maxima and looks at
// the low words and positions only on a tie.  The pivot row is read from LDS
// once, one element per lane (lane c of every row of sixteen holds slots c and
// 16 + c), and the rank-1 update takes it by the FMA's own lane broadcast
// (v_fmac_f64 with row_newbcast): sixteen broadcast reads per wave and column
// were a thousand LDS cycles.  Per column: one barrier after the waves'
// candidates, then with one workgroup the pivot row through LDS and a second
// barrier, with several the exchange (the candidate's wave publishes, all
// poll, second barrier).
constexpr int kLeaf64MaxG = 16;  // 16384 rows

typedef double v2du __attribute__((ext_vector_type(2), aligned(8)));
typedef double v2d __attribute__((ext_vector_type(2)));

// Maximum over the lanes of each row of sixteen (all of them get it).
__device__ __forceinline__ unsigned row_max_u32(unsigned k) {
  k = max(k, (unsigned)__builtin_amdgcn_mov_dpp((int)k, 0xB1, 0xf, 0xf, false));
  k = max(k, (unsigned)__builtin_amdgcn_mov_dpp((int)k, 0x4E, 0xf, 0xf, false));
  k = max(k, (unsigned)__builtin_amdgcn_mov_dpp((int)k, 0x141, 0xf, 0xf, false));
  return max(k, (unsigned)__builtin_amdgcn_mov_dpp((int)k, 0x140, 0xf, 0xf, false));
}

// Of the candidates (hi, lo, pos) on lanes 0..15 (repeated in every row of
// sixteen; hi 0: none), the lane with the largest (hi, lo), lowest pos.
__device__ __forceinline__ int row_best(unsigned hi, unsigned lo, unsigned pos) {
  const unsigned mh = row_max_u32(hi);
  unsigned b = (unsigned)__ballot(hi == mh) & 0xffffu;
  if (__builtin_expect(__popc(b) != 1, 0)) {
    const unsigned ml = row_max_u32(hi == mh ? lo : 0u);
    const bool c = hi == mh && lo == ml;
    const unsigned mp = row_max_u32(c ? ~pos : 0u);
    b = (unsigned)__ballot(c && ~pos == mp) & 0xffffu;
  }
  return __builtin_amdgcn_readfirstlane(__ffs((int)b) - 1);
}

template <int NT, int R>
__global__ __launch_bounds__(NT) void leaf64_kernel(
    double* __restrict__ P, int64_t ldp, int m, int w, int G, int* __restrict__ piv,
    int* __restrict__ lperm_n, int* __restrict__ lpos, int* __restrict__ lsrc,
    int* __restrict__ pperm_n, int* __restrict__ ppos, int* __restrict__ psrc, int row0, int pnb,
    int* __restrict__ zero_col, u64* __restrict__ xbuf, int* __restrict__ err,
    unsigned epoch_base, int piv_offset, int* __restrict__ fz_global, int spin_limit) {
  __builtin_amdgcn_s_setprio(3);  // on the critical path (see tsl_kernel)
  constexpr int NWAVE = NT / 64;
  constexpr int SW = slot_words<double>();  // [0] hi, [1] lo, [2] position, [3] unused, row
  constexpr int STAGE = kLeaf64MaxG * SW, KMAX = (STAGE + NT - 1) / NT;
  __shared__ uint4 s_key[2][NWAVE];           // each wave's candidate
  __shared__ __align__(16) double s_row[LW];  // the workgroup's candidate row
  __shared__ __align__(16) unsigned stage[STAGE];
  __shared__ int s_abort;
  __shared__ int s_piv[LW];
  __shared__ __align__(16) int s_pp[256 + 4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = blockIdx.x;

  // slot r of a thread is row (g R + r) NT + tid, and pos its position (rows
  // past m: none)
  double v[R][LW];
  int pos[R];
  const double* src[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    pos[r] = (g * R + r) * NT + tid;
    src[r] = P + (int64_t)min(pos[r], m - 1) * ldp;
    if (pos[r] >= m) pos[r] = -1;
  }
  if (w == LW) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < LW; c += 2) {
        const v2du t = *reinterpret_cast<const v2du*>(src[r] + c);
        v[r][c] = t.x;
        v[r][c + 1] = t.y;
      }
  } else {
#pragma unroll
    for (int c = 0; c < LW; ++c) {
      const int cc = min(c, w - 1);
      const double on = c < w ? 1.0 : 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double t = src[r][cc];
        v[r][c] = on != 0.0 ? t : 0.0;
      }
    }
  }
  if (tid == 0) s_abort = 0;
  __syncthreads();

  int first_zero = -1;
  // column j of group j / 8 is register slot jj (see rotate8); slots [live,
  // 32) hold columns finished in earlier groups
  auto column = [&](auto jjc, int j, int live) __attribute__((always_inline)) -> bool {
    constexpr int jj = decltype(jjc)::value;
    const int par = j & 1;
    // ---- the wave's candidate: the largest |a| over rows at positions >= j by
    // its high word (plus one: zero means none)
    unsigned hi[R], lo[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const u64 b = (u64)__double_as_longlong(v[r][jj]);
      hi[r] = pos[r] >= j ? ((unsigned)(b >> 32) & 0x7fffffffu) + 1u : 0u;
      lo[r] = (unsigned)b;
    }
    unsigned mh = wave_max_u32(max(hi[0], hi[R - 1]));
    if (__builtin_expect(mh > 0x7ff00000u, 0)) {
      // infinities or NaNs: a NaN counts at position j only, as an infinity
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (v[r][jj] != v[r][jj]) {
          hi[r] = pos[r] == j ? 0x7ff00001u : 0u;
          lo[r] = 0u;
        }
      mh = wave_max_u32(max(hi[0], hi[R - 1]));
    }
    u64 b0 = __ballot(hi[0] == mh), b1 = R == 2 ? __ballot(hi[R - 1] == mh) : 0ull;
    if (__builtin_expect(__popcll(b0) + __popcll(b1) != 1 && mh != 0u, 0)) {
      // equal high words: the low words, then the lowest position
      const unsigned ml = wave_max_u32(max(hi[0] == mh ? lo[0] : 0u, hi[R - 1] == mh ? lo[R - 1] : 0u));
      const bool c0 = hi[0] == mh && lo[0] == ml, c1 = hi[R - 1] == mh && lo[R - 1] == ml;
      const unsigned mp = wave_max_u32(max(c0 ? ~(unsigned)pos[0] : 0u,
                                           c1 ? ~(unsigned)pos[R - 1] : 0u));
      b0 = __ballot(c0 && ~(unsigned)pos[0] == mp);
      b1 = R == 2 ? __ballot(c1 && ~(unsigned)pos[R - 1] == mp) : 0ull;
    }
    const bool first = b0 != 0ull;
    const int wl = __ffsll((long long)(first ? b0 : b1)) - 1;
    if (lane == wl)
      s_key[par][wave] = make_uint4(mh, first ? lo[0] : lo[R - 1],
                                    (unsigned)(first ? pos[0] : pos[R - 1]),
                                    (unsigned)lane + (first ? 0u : 64u));
    __syncthreads();
    // ---- the workgroup's candidate, found by every wave
    const uint4 e = s_key[par][lane & (NWAVE - 1)];
    // (with eight waves lanes 8..15 repeat their entries; without any candidate
    // one of them may be named)
    const int bw = row_best((lane & 15) < NWAVE ? e.x : 0u, e.y, e.z) & (NWAVE - 1);
    int p = readlane_i((int)e.z, bw);
    unsigned bhi = (unsigned)readlane_i((int)e.x, bw);
    double u0, u1;
    if (wave == bw) {
      // its lane stores its row's live slots
      const int code = readlane_i((int)e.w, bw);
#define EAMD_PUT8(R_, C_)                                            \
  _Pragma("unroll") for (int c = C_; c < C_ + 8; c += 2)              \
    *reinterpret_cast<v2d*>(&s_row[c]) = v2d{v[R_][c], v[R_][c + 1]};
#define EAMD_PUT(R_)                        \
  if (lane == (code & 63)) {                \
    EAMD_PUT8(R_, 0)                        \
    if (live > 8) { EAMD_PUT8(R_, 8) }      \
    if (live > 16) { EAMD_PUT8(R_, 16) }    \
    if (live > 24) { EAMD_PUT8(R_, 24) }    \
  }                                         \
  /* (keeps the two copies apart: merged, the row would be indexed) */ \
  asm volatile("; slot " #R_ ::: "memory");
      if (R == 1 || code < 64) {
        EAMD_PUT(0)
      } else {
        EAMD_PUT(R - 1)
      }
#undef EAMD_PUT
#undef EAMD_PUT8
    }
    if (G == 1) {
      __syncthreads();
      u0 = s_row[lane & 15];
      u1 = s_row[16 + (lane & 15)];
    } else {
      const unsigned epoch = epoch_base + (unsigned)j + 1u;
      u64* base = xbuf + (size_t)par * G * SW;
      if (wave == bw) {
        // publish: the row a word per lane, and the header
        asm volatile("" ::: "memory");  // a wave's LDS accesses execute in order
        u64* slot = base + (size_t)g * SW;
        const unsigned rw = reinterpret_cast<const unsigned*>(s_row)[lane];
        const unsigned hw = lane == 0 ? bhi
                            : lane == 1 ? (unsigned)readlane_i((int)e.y, bw)
                            : lane == 2 ? (unsigned)p
                                        : 0u;
        if (lane < 4) put_word(slot + lane, hw, epoch);
        put_word(slot + 4 + lane, rw, epoch);
      }
      // one parallel poll of every slot: each thread requests its words
      // together, then only the missing ones again
      const int total = G * SW;
      bool done[KMAX];
#pragma unroll
      for (int k = 0; k < KMAX; ++k) done[k] = tid + k * NT >= total;
      int bad = 0;
      for (int spins = 0;; ++spins) {
        u64 wv[KMAX];
#pragma unroll
        for (int k = 0; k < KMAX; ++k)
          if (!done[k])
            wv[k] = __hip_atomic_load(base + tid + k * NT, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
        bool all = true;
#pragma unroll
        for (int k = 0; k < KMAX; ++k)
          if (!done[k]) {
            if ((unsigned)(wv[k] >> 32) == epoch) {
              stage[tid + k * NT] = (unsigned)wv[k];
              done[k] = true;
            } else {
              all = false;
            }
          }
        if (all) break;
        // the limit every poll, another workgroup's give-up every 256th
        if (spins >= spin_limit ||
            ((spins & 255) == 255 &&
             __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
          bad = 1;
          break;
        }
      }
      if (bad) s_abort = 1;
      __syncthreads();
      if (__builtin_expect(s_abort, 0)) {
        if (tid == 0) __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
      }
      const unsigned* hh = &stage[min(lane & 15, G - 1) * SW];
      const unsigned sh = (lane & 15) < G ? hh[0] : 0u, slo = hh[1], sp = hh[2];
      const int ws = row_best(sh, slo, sp);
      p = readlane_i((int)sp, ws);
      const double* ur = reinterpret_cast<const double*>(&stage[ws * SW + 4]);
      u0 = ur[lane & 15];
      u1 = ur[16 + (lane & 15)];
    }
    if (g == 0 && tid == 0) s_piv[j] = p;
    // ---- positions j and p change places; the pivot row is at j and done.
    // Then scale and rank-1 update of the rows below j (l = 0 leaves a row)
    const double pv = readlane_d(u0, jj);
    if (pv == 0.0 && first_zero < 0) first_zero = j;
    double nl[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      pos[r] = pos[r] == p ? j : (pos[r] == j ? p : pos[r]);
      const bool act = pos[r] > j && pv != 0.0;
      const double q = v[r][jj] / pv;
      nl[r] = act ? -q : 0.0;
      v[r][jj] = act ? q : v[r][jj];
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if constexpr (jj < 7) fmac_bcast8<0, jj + 1>(v[r], u0, nl[r]);
    if (live > 8) {
#pragma unroll
      for (int r = 0; r < R; ++r) fmac_bcast8<8, 0>(v[r], u0, nl[r]);
      if (live > 16) {
#pragma unroll
        for (int r = 0; r < R; ++r) fmac_bcast8<16, 0>(v[r], u1, nl[r]);
        if (live > 24) {
#pragma unroll
          for (int r = 0; r < R; ++r) fmac_bcast8<24, 0>(v[r], u1, nl[r]);
        }
      }
    }
    return true;
  };
  const int ngroups = (w + 7) / 8;
  bool ok = true;
#pragma unroll 1
  for (int g8 = 0; g8 < ngroups && ok; ++g8) {
    const int live = LW - 8 * g8, j0 = 8 * g8;
#define EAMD_COL(JJ) \
    if (ok && j0 + JJ < w) ok = column(std::integral_constant<int, JJ>{}, j0 + JJ, live);
    EAMD_COL(0) EAMD_COL(1) EAMD_COL(2) EAMD_COL(3) EAMD_COL(4) EAMD_COL(5) EAMD_COL(6)
    EAMD_COL(7)
#undef EAMD_COL
#pragma unroll
    for (int r = 0; r < R; ++r) rotate8(v[r]);
  }
#pragma unroll 1
  for (int q = ngroups; q < 4; ++q)
#pragma unroll
    for (int r = 0; r < R; ++r) rotate8(v[r]);
  if (s_abort) {
    // gave up: empty lists, as leaf_lu_kernel
    if (g == 0 && tid == 0) {
      *lperm_n = 0;
      *pperm_n = 0;
      *zero_col = -1;
    }
    return;
  }
  __syncthreads();
  if (g == 0 && wave == 0) {
    leaf_lists(lane < w ? s_piv[lane] : 0, w, row0, pnb, lane, piv, piv_offset, lperm_n, lpos,
               lsrc, pperm_n, ppos, psrc, s_pp);
  }
  // every row at its final position (every workgroup has read its rows before
  // any passes the exchange of a column)
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (pos[r] < 0) continue;
    double* dst = P + (int64_t)pos[r] * ldp;
    if (w == LW) {
#pragma unroll
      for (int c = 0; c < LW; c += 2)
        *reinterpret_cast<v2du*>(dst + c) = v2du{v[r][c], v[r][c + 1]};
    } else {
#pragma unroll
      for (int c = 0; c < LW; ++c)
        if (c < w) dst[c] = v[r][c];
    }
  }
  if (g == 0 && tid == 0) {
    *zero_col = first_zero;
    if (fz_global && first_zero >= 0 && *fz_global < 0) *fz_global = first_zero + piv_offset;
  }
}

// Launches one leaf over rows [0, m) of the sub-panel at P (row-major, ldp),
// columns [0, w), w <= 32.
template <typename T>
int leaf_lu(eamd_handle* h, T* P, int64_t ldp, int m, int w, int* piv, int* lperm_n, int* lpos,
            int* lsrc, int* pperm_n, int* ppos, int* psrc, int row0, int pnb, int* zero_col,
            int piv_offset, int* fz_global) {
  if (w > LW || pnb > 256) {
    set_error("leaf width %d / panel width %d unsupported", w, pnb);
    return kErrUnsupported;
  }
  constexpr bool k64 = sizeof(T) == 8;
  constexpr int BLOCK = 1024;
  const int rows = k64 && m <= 512 ? 512 : BLOCK;
  const int G = ceil_div(m, rows), max_g = k64 ? kLeaf64MaxG : kMaxG;
  if (G > max_g) {
    set_error("panel of %d rows exceeds the leaf exchange (%d workgroups of %d rows)", m, max_g,
              rows);
    return kErrUnsupported;
  }
  const int SW = slot_words<T>();
  size_t need = 256 + sizeof(u64) * 2 * (size_t)(G + 1) * SW;
  void* base = nullptr;
  bool fresh = h->ws.bytes[kWsPanelSync] < need;
  EAMD_CHECK(h->ws.get(kWsPanelSync, need, &base));
  if (fresh || h->panel_epoch > (1u << 31)) {
    EAMD_HIP(hipMemsetAsync(base, 0, h->ws.bytes[kWsPanelSync], h->stream));
    h->panel_epoch = 0;
  }
  unsigned epoch_base = h->panel_epoch;
  h->panel_epoch += (unsigned)w + 1u;
  char* b = static_cast<char*>(base);
  // polls an exchange may take before the leaf gives up (the call then
  // reports a time-out); EAMD_LEAF_SPIN sets another limit
  static const int spin_limit = env_int("EAMD_LEAF_SPIN", kLeafSpin);
#define EAMD_LEAF(K, NT)                                                                      \
  hipLaunchKernelGGL((K), dim3(G), dim3(NT), 0, h->stream, P, ldp, m, w, G, piv, lperm_n, lpos, \
                     lsrc, pperm_n, ppos, psrc, row0, pnb, zero_col,                          \
                     reinterpret_cast<u64*>(b + 256), reinterpret_cast<int*>(b), epoch_base,  \
                     piv_offset, fz_global, spin_limit)
  if constexpr (k64) {
    if (m > 512) EAMD_LEAF((leaf64_kernel<1024, 1>), 1024);
    else EAMD_LEAF((leaf64_kernel<512, 1>), 512);
  } else {
    EAMD_LEAF((leaf_lu_kernel<T, BLOCK>), BLOCK);
  }
#undef EAMD_LEAF
  EAMD_HIP(hipGetLastError());
  return kOk;
}

// ---------------------------------------------------------------------------
// Tournament pivoting (CALU: Grigori, Demmel, Xiang, "CALU: a communication
// optimal LU factorization algorithm", SIAM J. Matrix Anal. Appl. 32, 2011)
// for the FP32 panel of the mixed-precision solver, whose result is judged
// by the backward error after refinement rather than by Eigen's pivot
// sequence.  A leaf of m rows costs a few short launches instead of one
// exchange round trip per column:
//   1. a workgroup per 256, 512 or 1024 rows (see leaf_lu_tournament) runs
//      partial pivoting on them, in registers, and records the rows it picked
//      (up to 32 candidates);
//   2. while more groups remain than one workgroup's rows hold, a workgroup
//      per 16 groups (8 with the wide rounds off) runs partial pivoting on the
//      original values of their candidates and keeps 32 of them;
//   3. one workgroup does the same over the last groups: the rows it picks, in
//      order, are the leaf's pivots, and each is a row of the factored top
//      block L11\U11 as it is picked, written in place; a wave without rows
//      keeps the books: it saves the original rows 0..w-1, derives the
//      transpositions, replays them into the permutation lists and lists where
//      the displaced rows go;
//   4. every other row is solved against U11 (l = a U11^-1) in parallel.
namespace {

// Shape of a round's workgroup over CAP rows (or candidates): a row per thread
// up to 512 (a wave per SIMD, then two), two rows per thread for 1024.  The
// final round's bookkeeping wave comes on top.  What bounds it: the columns
// follow each other, and a column is some 60 instructions of search, exchange
// and scaling per wave beside its FMAs, so a lone wave of each SIMD with four
// rows per lane issued one every six cycles and waited on LDS in between
// (1024 rows in four waves: 2000 cycles a column; 512 in two: 1650; 256 in
// one: 1350; now about 1600, 1300 and 1100).  16384 rows: local and final
// round 30 + 51 us before (512-row groups, 1024 candidates), 34 + 30 now;
// 4096 rows 24 + 50 before, 18 + 30 now.  The registers stay within what one of the trailing update's
// workgroups gives back when it ends (272 per SIMD): a round that needed the
// room of two would wait until the update drains.
template <int CAP>
struct Tsl {
  static constexpr int R = CAP == 1024 ? 2 : 1;  // rows per thread
  static constexpr int NW = CAP / 64 / R;        // waves with rows
  static constexpr int KB = CAP == 256 ? 9 : (CAP == 512 ? 10 : 11);
  static_assert((1 << KB) == 2 * CAP, "slot code width");
};

// a[C + q] += (lane (C + q) % 16 of each row of sixteen of u) * l for q = Q0
// .. 7 (as fmac_bcast8, in FP32).
template <int C, int Q0>
__device__ __forceinline__ void fmac_bcast8f(float (&a)[LW], float u, float l) {
  constexpr int N0 = C & 15;
  static_assert(Q0 == 0 || C == 0, "part groups start the row");
#define EAMD_F(I, U, L, N)                                                                \
  "v_fmac_f32_dpp %" #I ", %" #U ", %" #L " row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t"
#define EAMD_FN(I, N)                                                                     \
  "v_fmac_f32_dpp %" #I ", %8, %9 row_newbcast:%" #N " row_mask:0xf bank_mask:0xf\n\t"
  if constexpr (Q0 == 0) {
    asm volatile("s_nop 1\n\t" EAMD_FN(0, 10) EAMD_FN(1, 11) EAMD_FN(2, 12) EAMD_FN(3, 13)
                     EAMD_FN(4, 14) EAMD_FN(5, 15) EAMD_FN(6, 16) EAMD_FN(7, 17)
                 : "+v"(a[C]), "+v"(a[C + 1]), "+v"(a[C + 2]), "+v"(a[C + 3]), "+v"(a[C + 4]),
                   "+v"(a[C + 5]), "+v"(a[C + 6]), "+v"(a[C + 7])
                 : "v"(u), "v"(l), "n"(N0), "n"(N0 + 1), "n"(N0 + 2), "n"(N0 + 3), "n"(N0 + 4),
                   "n"(N0 + 5), "n"(N0 + 6), "n"(N0 + 7));
  } else if constexpr (Q0 == 1) {
    asm volatile("s_nop 1\n\t" EAMD_F(0, 7, 8, 1) EAMD_F(1, 7, 8, 2) EAMD_F(2, 7, 8, 3)
                     EAMD_F(3, 7, 8, 4) EAMD_F(4, 7, 8, 5) EAMD_F(5, 7, 8, 6) EAMD_F(6, 7, 8, 7)
                 : "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]),
                   "+v"(a[7])
                 : "v"(u), "v"(l));
  } else if constexpr (Q0 == 2) {
    asm volatile("s_nop 1\n\t" EAMD_F(0, 6, 7, 2) EAMD_F(1, 6, 7, 3) EAMD_F(2, 6, 7, 4)
                     EAMD_F(3, 6, 7, 5) EAMD_F(4, 6, 7, 6) EAMD_F(5, 6, 7, 7)
                 : "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7])
                 : "v"(u), "v"(l));
  } else if constexpr (Q0 == 3) {
    asm volatile("s_nop 1\n\t" EAMD_F(0, 5, 6, 3) EAMD_F(1, 5, 6, 4) EAMD_F(2, 5, 6, 5)
                     EAMD_F(3, 5, 6, 6) EAMD_F(4, 5, 6, 7)
                 : "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7])
                 : "v"(u), "v"(l));
  } else if constexpr (Q0 == 4) {
    asm volatile("s_nop 1\n\t" EAMD_F(0, 4, 5, 4) EAMD_F(1, 4, 5, 5) EAMD_F(2, 4, 5, 6)
                     EAMD_F(3, 4, 5, 7)
                 : "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7])
                 : "v"(u), "v"(l));
  } else if constexpr (Q0 == 5) {
    asm volatile("s_nop 1\n\t" EAMD_F(0, 3, 4, 5) EAMD_F(1, 3, 4, 6) EAMD_F(2, 3, 4, 7)
                 : "+v"(a[5]), "+v"(a[6]), "+v"(a[7])
                 : "v"(u), "v"(l));
  } else if constexpr (Q0 == 6) {
    asm volatile("s_nop 1\n\t" EAMD_F(0, 2, 3, 6) EAMD_F(1, 2, 3, 7)
                 : "+v"(a[6]), "+v"(a[7])
                 : "v"(u), "v"(l));
  } else if constexpr (Q0 == 7) {
    asm volatile("s_nop 1\n\t" EAMD_F(0, 1, 2, 7) : "+v"(a[7]) : "v"(u), "v"(l));
  }
#undef EAMD_FN
#undef EAMD_F
}

template <int C>
__device__ __forceinline__ void fmac_bcast1f(float (&a)[LW], float u, float l) {
  asm volatile("s_nop 1\n\tv_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
               : "+v"(a[C])
               : "v"(u), "v"(l), "n"(C));
}

// The largest of NK (16 or 32) keys in LDS, on every lane.
template <int NK>
__device__ __forceinline__ unsigned keys_max(const unsigned* s_key, int lane) {
  unsigned k = s_key[lane & 15];
  if (NK == 32) k = max(k, s_key[16 + (lane & 15)]);
  return row_max_u32(k);
}

// MODE 0: local selection over rows blockIdx.x * CAP + [0, CAP), candidates
// to cand.  MODE 2: merge of the n_in candidates' CAP / 32 groups from
// blockIdx.x * CAP / 32 on into group blockIdx.x of cand.  MODE 1: the final
// round over all n_in candidates (at most CAP / 32 groups).  Every candidate
// group is full (w candidates) but the last.  A column's pivot is the maximum
// over the waves' own maxima, exchanged through LDS; the pivot row is read from
// LDS once, an element per lane, and the update takes it by the FMA's lane
// broadcast (see leaf64_kernel).
template <int MODE, int CAP>
__global__ __launch_bounds__(64 * (Tsl<CAP>::NW + (MODE == 1))) void tsl_kernel(
    float* __restrict__ P, int64_t ldp, int m, int w, const int* __restrict__ cand_in, int n_in,
    int* __restrict__ cand, float* __restrict__ saved, int* __restrict__ moved,
    int* __restrict__ piv, int* __restrict__ lperm_n, int* __restrict__ lpos,
    int* __restrict__ lsrc, int* __restrict__ pperm_n, int* __restrict__ ppos,
    int* __restrict__ psrc, int row0, int pnb, int* __restrict__ zero_col, int piv_offset,
    int* __restrict__ fz_global, int fuse, float* __restrict__ xtop) {
  // the panel is the factorization's critical path while the trailing
  // update's waves share its SIMDs: its waves take issue priority
  __builtin_amdgcn_s_setprio(3);
  constexpr int R = Tsl<CAP>::R, NW = Tsl<CAP>::NW, KB = Tsl<CAP>::KB;
  constexpr int NT = 64 * (NW + (MODE == 1)), WROWS = 64 * R;
  constexpr unsigned kSlotMask = (1u << KB) - 1u;
  __shared__ unsigned s_key[4 * NW];         // each sixteen lanes' largest key
  __shared__ __align__(16) float s_row[LW];  // the pivot row
  __shared__ __align__(16) float s_in[NW][64 * LW];  // rows on their way to their lanes
  __shared__ int s_orig[MODE == 1 ? CAP : 1];        // each slot's row
  // the bookkeeping wave's lists, for the final moves
  __shared__ int s_pos[64], s_src[64], s_ps[MODE == 1 ? 512 : 1], s_n;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s0 = MODE == 1 ? 0 : blockIdx.x * (MODE == 0 ? CAP : CAP / LW * w);
  const int nrows = min(MODE == 0 ? CAP : CAP / LW * w, (MODE == 0 ? m : n_in) - s0);
  const int steps = min(w, nrows);
  if (MODE != 1 || wave < NW) {
    // slot q = WROWS wave + 64 r + lane
    int orig[R];
    unsigned em[R], kq[R];
    int st[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int q = wave * WROWS + r * 64 + lane;
      const bool valid = q < nrows;
      // (groups of w candidates, LW apart)
      const int e = s0 + q;
      orig[r] = !valid ? 0
                       : (MODE == 0 ? e : cand_in[w == LW ? e : (e / w) * LW + e % w]);
      if (MODE == 1) s_orig[q] = orig[r];
      em[r] = valid ? ~0u : 0u;
      kq[r] = kSlotMask - (unsigned)q;
      st[r] = -1;
    }
    // An empty slot loads row 0 and a leaf narrower than 32 repeats its last
    // column: such values are never keyed, selected or stored.
    float v[R][LW];
    if (w == LW && ((uintptr_t)P & 15) == 0 && (ldp & 3) == 0) {
      // eight lanes per row, so that a load instruction asks for eight whole
      // 128-byte lines (a row per lane: 64 lines, eight times over), then
      // through LDS to the rows' lanes.  Word c of row i lies at c ^ (i % 8):
      // consecutive lanes' 16-byte reads fall on different banks.
      v4f t[R][8];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int row = __shfl(orig[r], 8 * k + (lane >> 3));
          t[r][k] = reinterpret_cast<const v4f*>(P + (int64_t)row * ldp)[lane & 7];
        }
      v4f* buf = reinterpret_cast<v4f*>(s_in[wave]);
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          buf[(8 * k + (lane >> 3)) * 8 + ((lane & 7) ^ (lane >> 3))] = t[r][k];
        asm volatile("" ::: "memory");  // a wave's LDS accesses execute in order
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const v4f x = buf[lane * 8 + (c ^ (lane & 7))];
          v[r][4 * c] = x.x;
          v[r][4 * c + 1] = x.y;
          v[r][4 * c + 2] = x.z;
          v[r][4 * c + 3] = x.w;
        }
        asm volatile("" ::: "memory");
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float* src = P + (int64_t)orig[r] * ldp;
#pragma unroll
        for (int c = 0; c < LW; ++c) v[r][c] = src[w == LW ? c : min(c, w - 1)];
      }
    }
    // every row read before the final round's first top row is stored
    if (MODE == 1) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < LW; ++c) asm volatile("" : "+v"(v[r][c])::"memory");
    }
    // Rows never move between lanes.  A slot holds a candidate row while em[r]
    // is all ones (valid and not yet selected); st[r] is the step that
    // selected it.  The pivot key of slot q is |a| with its KB low mantissa
    // bits replaced by 2^KB - 1 - q (zero for a slot that is out), so the
    // maximum names its slot, exact ties go to the lowest slot (the first row
    // in order for the local round) and scores within 2^(KB-23) relative count
    // as ties, which keeps every multiplier within 1 + 2^(KB-23).  Column j
    // of group g8 is register slot jj (see rotate8); slots [live, 32) hold
    // columns of earlier groups and are skipped by uniform branches on 8-slot
    // chunks, so the update does exactly the triangle.  The multipliers use
    // the reciprocal of the pivot.
    // the wave's key of the column in slot c
    auto post_key = [&](auto cc) __attribute__((always_inline)) {
      constexpr int c = decltype(cc)::value;
      unsigned key = 0;
#pragma unroll
      for (int r = 0; r < R; ++r)
        key = max(key, ((__float_as_uint(v[r][c]) & (0x7fffffffu & ~kSlotMask)) | kq[r]) & em[r]);
      key = row_max_u32(key);
      if ((lane & 15) == 0) s_key[tid >> 4] = key;
    };
    // A column: the keys are out at the first barrier; the slot of the largest
    // stores its row, out at the second; the next column's slot is
    // updated first, so that its keys are searched and out while the rest of
    // the update runs.  (With every wave storing its own best row instead, for
    // one barrier less, the single-lane stores alone were 500 cycles with four
    // waves and 1000 with eight.)  A valid unselected slot exists (j <
    // steps), so the winner does.
    auto column = [&](auto jjc, int j, int live) __attribute__((always_inline)) {
      constexpr int jj = decltype(jjc)::value;
      __syncthreads();
      const unsigned code = keys_max<4 * NW>(s_key, lane) & kSlotMask;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const bool sel = kq[r] == code;
        if (sel) {
          float4* dst = reinterpret_cast<float4*>(s_row);
#pragma unroll
          for (int c = 0; c < LW / 4; ++c)
            dst[c] = make_float4(v[r][4 * c], v[r][4 * c + 1], v[r][4 * c + 2], v[r][4 * c + 3]);
          asm volatile("" ::: "memory");
        }
        em[r] = sel ? 0u : em[r];
        st[r] = sel ? j : st[r];
      }
      __syncthreads();
      const float u0 = s_row[lane & 15], u1 = s_row[16 + (lane & 15)];
      const float pv = readlane_f(u0, jj);
      const float rinv = pv != 0.f ? __builtin_amdgcn_rcpf(pv) : 0.f;
      float nl[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float l = v[r][jj] * rinv;
        nl[r] = __uint_as_float((__float_as_uint(l) ^ 0x80000000u) & em[r]);
        v[r][jj] = em[r] ? l : v[r][jj];
      }
      if (jj < 7) {
#pragma unroll
        for (int r = 0; r < R; ++r) fmac_bcast1f<(jj + 1) % 8>(v[r], u0, nl[r]);
        if (j + 1 < steps) post_key(std::integral_constant<int, (jj + 1) % 8>{});
#pragma unroll
        for (int r = 0; r < R; ++r) fmac_bcast8f<0, jj + 2>(v[r], u0, nl[r]);
      }
      if (live > 8)
#pragma unroll
        for (int r = 0; r < R; ++r) fmac_bcast8f<8, 0>(v[r], u0, nl[r]);
      if (jj == 7 && j + 1 < steps) post_key(std::integral_constant<int, 8>{});
      if (live > 16)
#pragma unroll
        for (int r = 0; r < R; ++r) fmac_bcast8f<16, 0>(v[r], u1, nl[r]);
      if (live > 24)
#pragma unroll
        for (int r = 0; r < R; ++r) fmac_bcast8f<24, 0>(v[r], u1, nl[r]);
    };
    post_key(std::integral_constant<int, 0>{});
#pragma unroll 1
    for (int j0 = 0; j0 < steps; j0 += 8) {
      const int live = LW - j0;
#define EAMD_COL(JJ) \
  if (j0 + JJ < steps) column(std::integral_constant<int, JJ>{}, j0 + JJ, live);
      EAMD_COL(0) EAMD_COL(1) EAMD_COL(2) EAMD_COL(3) EAMD_COL(4) EAMD_COL(5) EAMD_COL(6)
      EAMD_COL(7)
#undef EAMD_COL
#pragma unroll
      for (int r = 0; r < R; ++r) rotate8(v[r]);
    }
    if (MODE != 1) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (st[r] >= 0) cand[blockIdx.x * LW + st[r]] = orig[r];
    }
  } else {
    // ---- the bookkeeping wave of the final round.  The original rows 0..w-1,
    // read before the top block overwrites them:
#pragma unroll
    for (int k = 0; k < LW * LW / 64; ++k) {
      const int e = lane + 64 * k, r = e / LW, c = e % LW;
      const float x = P[(int64_t)r * ldp + min(c, w - 1)];
      saved[e] = c < w ? x : 0.f;
    }
    // the incoming panel list (row0 == 0 starts it as the identity): lane l
    // keeps the appended rows l, l + 64, ..., LDS the sources
    const bool first = row0 == 0;
    const int pn0 = first ? pnb : *pperm_n;
    int app[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = 64 * q + lane;
      app[q] = !first && e < pn0 - pnb ? ppos[pnb + e] : -1;
    }
    for (int e = lane; e < 2 * pnb; e += 64) {
      s_ps[e] = !first && e < pn0 ? psrc[e] : e;
      if (first && e < pnb) {
        ppos[e] = e;
        psrc[e] = e;
      }
    }
    // complete before the lists and the top block are stored over
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    LeafPerm lp;
    lp.start(w, lane);
    // entry k's slot of the panel list (rows 0..pnb-1 are slots 0..pnb-1,
    // rows below them are appended slots), found as the entry appears
    int slot = row0 + lane, pn = pn0, first_zero = -1, my_piv = 0;
#pragma unroll 1
    for (int j = 0; j < steps; ++j) {
      __syncthreads();
      const unsigned code = keys_max<4 * NW>(s_key, lane) & kSlotMask;
      const int p = __builtin_amdgcn_readfirstlane(s_orig[(int)(kSlotMask - code)]);
      __syncthreads();
      // the row picked is row j of the top block (slot s of group g8 holds
      // column (s + 8 g8) % 32)
      const float x = s_row[lane & (LW - 1)];
      const int col = (lane + (j & ~7)) & (LW - 1);
      if (lane < LW && col < w) P[(int64_t)j * ldp + col] = x;
      if (readlane_f(x, j & 7) == 0.f && first_zero < 0) first_zero = j;
      bool fresh;
      const int k = lp.step<true>(j, p, lane, &fresh);
      if (lane == j) my_piv = k;
      if (fresh) {
        const int prow = row0 + p;
        int f = prow;
        if (prow >= pnb) {
          f = -1;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const u64 hit = __ballot(app[t] == prow);
            if (hit) f = pnb + 64 * t + __ffsll((long long)hit) - 1;
          }
          if (f < 0) f = pn++;
        }
        if (lane == k) slot = f;
      }
    }
    // ---- the leaf's lists: column c is swapped with entry k's position
    const int ln = lp.n;
    const int tp = __shfl(lp.pos, my_piv);
    if (lane < w) piv[lane] = tp + piv_offset;
    if (lane < ln) {
      lpos[lane] = lp.pos;
      lsrc[lane] = lp.src;
    }
    s_pos[lane] = lp.pos;
    s_src[lane] = __shfl(lp.pos, lp.src);
    // the panel's: a touched slot's new source is the old source of its
    // entry's source slot, and an appended slot's old source is itself
    const bool add = slot >= pn0;
    int old = slot;
    if (lane < ln && !add) old = s_ps[slot];
    const int src_old = __shfl(old, lp.src);
    if (lane < ln) {
      psrc[slot] = src_old;
      if (add) ppos[slot] = row0 + lp.pos;
    }
    // positions >= w now hold displaced original rows < w: list them
    const bool mv = lane < ln && lp.pos >= w;
    const u64 mb = __ballot(mv);
    const int idx = __popcll(mb & ((1ull << lane) - 1ull));
    if (mv) {
      moved[1 + 2 * idx] = lp.pos;
      moved[2 + 2 * idx] = lp.row;
    }
    if (lane == 0) {
      s_n = ln;
      moved[0] = __popcll(mb);
      *lperm_n = ln;
      *pperm_n = pn;
      *zero_col = first_zero;
      if (fz_global && first_zero >= 0 && *fz_global < 0) *fz_global = first_zero + piv_offset;
    }
  }
  if constexpr (MODE == 1) {
    if (!fuse) return;
    // (w == 32) The leaf's interchanges on the other columns of the panel
    // (row0 = j0 is the leaf's first panel column, pnb the panel width), 96
    // columns at a time, all loads before the stores; the top rows' values
    // right of the leaf go to xtop (LW x (pnb - j0 - LW)), from which the
    // apply kernel solves U12.  16-byte words: the host fuses only panels
    // whose rows start 16-byte aligned with pnb and ldp multiples of 4 (a word
    // never straddles the leaf, whose columns start at a multiple of 32).
    __syncthreads();
    constexpr int CW = 24, NM = (64 * CW + NT - 1) / NT;  // words per pass, and per thread
    const int ln = s_n, j0 = row0, nq = (pnb - LW) / 4, rest = pnb - j0 - LW;
    float* base = P - j0;  // panel column 0 of leaf row 0
    for (int q0 = 0; q0 < nq; q0 += CW) {
      v4f x[NM];
#pragma unroll
      for (int t = 0; t < NM; ++t) {
        const int e = tid + NT * t, k = e / CW, c = 4 * (q0 + e % CW);
        if (k < ln && c < 4 * nq)
          x[t] = *reinterpret_cast<const v4f*>(base + (int64_t)s_src[k] * ldp +
                                               (c < j0 ? c : c + LW));
      }
      // the loads of every wave are complete when its barrier is reached
#pragma unroll
      for (int t = 0; t < NM; ++t) asm volatile("" : "+v"(x[t])::"memory");
      __syncthreads();
#pragma unroll
      for (int t = 0; t < NM; ++t) {
        const int e = tid + NT * t, k = e / CW, c = 4 * (q0 + e % CW);
        if (k < ln && c < 4 * nq) {
          const int tpos = s_pos[k];
          float* d = tpos < LW && c >= j0 ? xtop + tpos * rest + (c - j0)
                                          : base + (int64_t)tpos * ldp + (c < j0 ? c : c + LW);
          *reinterpret_cast<v4f*>(d) = x[t];
        }
      }
    }
  }
}

// Rows w..m-1 of the leaf: l = a U11^-1, where a is the row's original
// value (its own row, or a saved row 0..w-1 for a position listed in moved).
// FULL: w == 32, without the column guards (which would multiply the code).
template <bool FULL>
__global__ __launch_bounds__(256) void tsl_apply_kernel(float* __restrict__ P, int64_t ldp, int m,
                                                        int w, const float* __restrict__ saved,
                                                        const int* __restrict__ moved) {
  __builtin_amdgcn_s_setprio(3);  // on the critical path (see tsl_kernel)
  if (FULL) w = LW;
  __shared__ float U[LW][LW + 1];
  __shared__ int mpos[LW], msrc[LW];
  __shared__ int s_nm;
  const int tid = threadIdx.x;
  for (int e = tid; e < LW * LW; e += 256) {
    const int r = e / LW, c = e - r * LW;
    U[r][c] = (r < w && c < w) ? P[(int64_t)r * ldp + c] : 0.f;
  }
  if (tid == 0) s_nm = moved[0];
  if (tid < LW) {
    mpos[tid] = moved[1 + 2 * tid];
    msrc[tid] = moved[2 + 2 * tid];
  }
  __syncthreads();
  const int i = w + blockIdx.x * 256 + tid;
  if (i >= m) return;
  int src = -1;
  for (int k = 0; k < s_nm; ++k)
    if (mpos[k] == i) src = msrc[k];
  float a[LW];
  // 16-byte words when the rows allow (saved rows always do)
  const bool vec = FULL && ((uintptr_t)P & 15) == 0 && (ldp & 3) == 0;
  if (FULL && (src >= 0 || vec)) {
    const v4f* ar = reinterpret_cast<const v4f*>(src >= 0 ? saved + src * LW
                                                          : P + (int64_t)i * ldp);
#pragma unroll
    for (int q = 0; q < LW / 4; ++q) {
      const v4f t = ar[q];
      a[4 * q] = t.x;
      a[4 * q + 1] = t.y;
      a[4 * q + 2] = t.z;
      a[4 * q + 3] = t.w;
    }
  } else {
    // one load path (a saved row or the row itself), word by word, every
    // load unconditional (columns past w re-read column w - 1 and are
    // masked): conditional loads of a narrow leaf's row keep `a` in scratch
    const float* row = src >= 0 ? saved + src * LW : P + (int64_t)i * ldp;
#pragma unroll
    for (int c = 0; c < LW; ++c) {
      const float v = row[FULL ? c : min(c, w - 1)];
      a[c] = (FULL || c < w) ? v : 0.f;
    }
  }
#pragma unroll
  for (int k = 0; k < LW; ++k) {
    const float d = U[k][k];
    const float x = d != 0.f ? a[k] / d : a[k];  // a zero pivot leaves its column unscaled
    a[k] = x;
#pragma unroll
    for (int c = k + 1; c < LW; ++c) a[c] -= x * U[k][c];
  }
  float* dst = P + (int64_t)i * ldp;
  if (vec) {
#pragma unroll
    for (int q = 0; q < LW / 4; ++q)
      reinterpret_cast<v4f*>(dst)[q] = v4f{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
  } else {
    // unconditional stores, last column first: columns past w land on
    // column w - 1, which its own value overwrites last (conditional stores
    // of a narrow leaf keep `a` in scratch memory)
#pragma unroll
    for (int c = LW - 1; c >= 0; --c) dst[FULL ? c : min(c, w - 1)] = a[c];
  }
}


// As tsl_apply_kernel (w == 32), and the row's `rest` panel columns right of
// the leaf (at most 96, a multiple of 4) take the update x -= l U12 (the rows'
// values already permuted).  64 rows per workgroup: wave 0 solves them, a row
// per lane, while waves 1 and 2 solve U12 = L11^-1 xtop (the permuted top rows
// right of the leaf), a column per lane; workgroup 0 also stores that as the
// top rows.  Then each wave updates 16 rows by FP32 matrix products, C
// requested at the start.  The solves' serial chains bound it (500 dependent
// steps, L11\U11 read from LDS four values at a time); with four threads a
// row, each solving it again and reading an LDS word per FMA, it took 23 us on
// average over the panels of n = 16384, and 15 now.
constexpr int kApplyRows = 64;
constexpr int kFuseRestMax = 96;  // panel columns right of a fused leaf (panels <= 128)
__global__ __launch_bounds__(256) void tsl_apply_rest_kernel(float* __restrict__ P, int64_t ldp,
                                                             int m, const float* __restrict__ saved,
                                                             const int* __restrict__ moved,
                                                             const float* __restrict__ xtop,
                                                             int rest) {
  __builtin_amdgcn_s_setprio(3);  // on the critical path (see tsl_kernel)
  // row strides whose fragment reads (16 rows x 4 k, 16 columns x 4 k) and row
  // reads (16 bytes a lane) fall on different banks
  constexpr int LS = LW + 4, US = kFuseRestMax + 16, NTJ = kFuseRestMax / 16;
  __shared__ __align__(16) float s_lu[LW][LW];          // L11\U11
  __shared__ __align__(16) float s_l[kApplyRows * LS];  // the rows, then l
  __shared__ float s_u12[LW * US];
  __shared__ int s_m[2 * LW + 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lk = lane >> 4;
  const int i0 = LW + blockIdx.x * kApplyRows;  // the workgroup's first row
  const int nr = min(kApplyRows, m - i0);
  // this lane's C: row i0 + 16 wave + l16, columns 16 t + 4 lk .. + 3 (past
  // the last row or column: the last one's, never stored)
  float* xrow = P + (int64_t)(i0 + min(16 * wave + l16, nr - 1)) * ldp + LW;
  v4f x[NTJ];
#pragma unroll
  for (int t = 0; t < NTJ; ++t)
    x[t] = *reinterpret_cast<const v4f*>(xrow + min(16 * t + 4 * lk, rest - 4));
  reinterpret_cast<v4f*>(&s_lu[0][0])[tid] =
      *reinterpret_cast<const v4f*>(P + (int64_t)(tid >> 3) * ldp + 4 * (tid & 7));
  const int nm = moved[0];
  if (tid < 2 * nm) s_m[tid] = moved[1 + tid];
  // the rows' 16-byte words, eight lanes a row
  v4f a2[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = 32 * h + (tid >> 3);
    a2[h] = *reinterpret_cast<const v4f*>(P + (int64_t)(i0 + min(r, nr - 1)) * ldp + 4 * (tid & 7));
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = 32 * h + (tid >> 3);
    int src = -1;
    for (int k = 0; k < nm; ++k)
      if (s_m[2 * k] == i0 + r) src = s_m[2 * k + 1];
    if (src >= 0) a2[h] = reinterpret_cast<const v4f*>(saved + src * LW)[tid & 7];
    *reinterpret_cast<v4f*>(&s_l[r * LS + 4 * (tid & 7)]) = a2[h];
  }
  __syncthreads();
  if (wave == 0) {
    float a[LW];
    v4f* row = reinterpret_cast<v4f*>(&s_l[lane * LS]);
#pragma unroll
    for (int c = 0; c < LW / 4; ++c) {
      const v4f t = row[c];
      a[4 * c] = t.x;
      a[4 * c + 1] = t.y;
      a[4 * c + 2] = t.z;
      a[4 * c + 3] = t.w;
    }
    // a zero pivot leaves its column unscaled
    const float d = s_lu[lane & (LW - 1)][lane & (LW - 1)];
    const float dinv = d != 0.f ? 1.0f / d : 1.0f;
#pragma unroll
    for (int k = 0; k < LW; ++k) {
      const float xk = a[k] * readlane_f(dinv, k);
      a[k] = xk;
#pragma unroll
      for (int q = (k + 1) / 4; q < LW / 4; ++q) {
        const v4f u = reinterpret_cast<const v4f*>(s_lu[k])[q];
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (4 * q + c > k) a[4 * q + c] -= xk * u[c];
      }
    }
#pragma unroll
    for (int c = 0; c < LW / 4; ++c)
      row[c] = v4f{a[4 * c], a[4 * c + 1], a[4 * c + 2], a[4 * c + 3]};
  } else if (wave < 3) {
    const int c = tid - 64;
    if (c < rest) {
      float u[LW];
#pragma unroll
      for (int i = 0; i < LW; ++i) u[i] = xtop[i * rest + c];
#pragma unroll
      for (int i = 0; i < LW; ++i) {
#pragma unroll
        for (int q = 0; q < (i + 3) / 4; ++q) {
          const v4f l = reinterpret_cast<const v4f*>(s_lu[i])[q];
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (4 * q + k < i) u[i] -= l[k] * u[4 * q + k];
        }
        s_u12[i * US + c] = u[i];
      }
      if (blockIdx.x == 0)
#pragma unroll
        for (int i = 0; i < LW; ++i) P[(int64_t)i * ldp + LW + c] = u[i];
    } else if (c < kFuseRestMax) {
#pragma unroll
      for (int i = 0; i < LW; ++i) s_u12[i * US + c] = 0.f;
    }
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = 32 * h + (tid >> 3);
    if (r < nr)
      *reinterpret_cast<v4f*>(P + (int64_t)(i0 + r) * ldp + 4 * (tid & 7)) =
          *reinterpret_cast<const v4f*>(&s_l[r * LS + 4 * (tid & 7)]);
  }
  // x^T -= U12^T l^T: a lane's four results are four columns of one row
  float lb[LW / 4];
#pragma unroll
  for (int k = 0; k < LW / 4; ++k) lb[k] = -s_l[(16 * wave + l16) * LS + 4 * k + lk];
#pragma unroll
  for (int t = 0; t < NTJ; ++t) {
    if (16 * t >= rest) break;
#pragma unroll
    for (int k = 0; k < LW / 4; ++k)
      x[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(s_u12[(4 * k + lk) * US + 16 * t + l16], lb[k],
                                                  x[t], 0, 0, 0);
    if (16 * wave + l16 < nr && 16 * t + 4 * lk < rest)
      *reinterpret_cast<v4f*>(xrow + 16 * t + 4 * lk) = x[t];
  }
}

}  // namespace

// Same outputs as leaf_lu; FP32 only.  Panels of up to 256 rows take the
// partial-pivoting leaf.  The local round's groups: 256 rows up to 4096, 512
// up to 8192, 1024 above, so that a final round over at most 512 candidates
// follows (over 256 candidates for up to 8 groups); past 16384 rows, groups
// are merged 16 at a time first.  With the wide rounds switched off every
// round takes 256 rows.
int leaf_lu_tournament(eamd_handle* h, float* P, int64_t ldp, int m, int w, int* piv,
                       int* lperm_n, int* lpos, int* lsrc, int* pperm_n, int* ppos, int* psrc,
                       int row0, int pnb, int* zero_col, int piv_offset, int* fz_global,
                       bool* fused) {
  static const bool wide = env_int("EAMD_TSL_WIDE", 1) != 0;
  const int cap = !wide || m <= 4096 ? 256 : (m <= 8192 ? 512 : 1024);
  const int G1 = ceil_div(m, cap);
  // the leaf's interchanges on the other panel columns, the U rows right of
  // it and their update are done here too when w == 32 (the caller skips
  // its own)
  const bool fuse = fused && w == LW && G1 > 1 && pnb - row0 - w <= kFuseRestMax &&
                    ((uintptr_t)(P - row0) & 15) == 0 && ldp % 4 == 0 && pnb % 4 == 0;
  if (fused) *fused = fuse;
  if (G1 <= 1)
    return leaf_lu<float>(h, P, ldp, m, w, piv, lperm_n, lpos, lsrc, pperm_n, ppos, psrc, row0,
                          pnb, zero_col, piv_offset, fz_global);
  if (w > LW || pnb > 256) {
    set_error("tournament leaf: %d rows x %d columns unsupported", m, w);
    return kErrUnsupported;
  }
  void* base = nullptr;
  // two candidate buffers (ping-pong between merge levels), moved list and the
  // saved rows
  const size_t need = sizeof(int) * (2 * (size_t)G1 * LW + 2 * LW + 8) +
                      sizeof(float) * LW * LW + sizeof(float) * LW * 256;
  EAMD_CHECK(h->ws.get(kWsTsl, need, &base));
  int* candA = static_cast<int*>(base);
  int* candB = candA + (size_t)G1 * LW;
  int* moved = candB + (size_t)G1 * LW;
  float* saved = reinterpret_cast<float*>(moved + 2 * LW + 8);
  float* xtop = saved + LW * LW;  // permuted top rows right of the leaf (fused)
  hipStream_t s = h->stream;
  int *cin = nullptr, *cout = candA, *spare = candB;
  int G = G1, n = 0;  // groups, and candidates in them
#define EAMD_TSL(MODE, CAP, BLOCKS)                                                           \
  hipLaunchKernelGGL((tsl_kernel<MODE, CAP>), dim3(BLOCKS),                                   \
                     dim3(64 * (Tsl<CAP>::NW + (MODE == 1))), 0, s, P, ldp, m, w, cin, n, cout, \
                     saved, moved, piv, lperm_n, lpos, lsrc, pperm_n, ppos, psrc, row0, pnb,  \
                     zero_col, piv_offset, fz_global, fuse ? 1 : 0, xtop)
  if (cap == 256) EAMD_TSL(0, 256, G);
  else if (cap == 512) EAMD_TSL(0, 512, G);
  else EAMD_TSL(0, 1024, G);
  n = (G - 1) * w + std::min(w, m - (G - 1) * cap);
  cin = cout;
  cout = spare;
  spare = cin;
  const int fan = wide ? 512 / LW : 256 / LW;
  while (G > fan) {
    const int Gn = ceil_div(G, fan);
    if (wide) EAMD_TSL(2, 512, Gn);
    else EAMD_TSL(2, 256, Gn);
    n = (Gn - 1) * w + std::min(w, n - (Gn - 1) * fan * w);
    G = Gn;
    cin = cout;
    cout = spare;
    spare = cin;
  }
  if (G > 256 / LW) EAMD_TSL(1, 512, 1);
  else EAMD_TSL(1, 256, 1);
#undef EAMD_TSL
  const int rest = pnb - row0 - w;
  if (fuse && rest > 0) {
    hipLaunchKernelGGL(tsl_apply_rest_kernel, dim3(ceil_div(m - w, kApplyRows)), dim3(256), 0, s,
                       P, ldp, m, saved, moved, xtop, rest);
  } else if (m > w) {
    if (w == LW)
      hipLaunchKernelGGL(tsl_apply_kernel<true>, dim3(ceil_div(m - w, 256)), dim3(256), 0, s, P,
                         ldp, m, w, saved, moved);
    else
      hipLaunchKernelGGL(tsl_apply_kernel<false>, dim3(ceil_div(m - w, 256)), dim3(256), 0, s, P,
                         ldp, m, w, saved, moved);
  }
  EAMD_HIP(hipGetLastError());
  return kOk;
}

template int leaf_lu<double>(eamd_handle*, double*, int64_t, int, int, int*, int*, int*, int*,
                             int*, int*, int*, int, int, int*, int, int*);
template int leaf_lu<float>(eamd_handle*, float*, int64_t, int, int, int*, int*, int*, int*,
                            int*, int*, int*, int, int, int*, int, int*);

}  // namespace eamd

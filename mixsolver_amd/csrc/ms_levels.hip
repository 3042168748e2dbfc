// ms_levels.hip -- level-scheduled natural-order factorizations and
// triangular sweeps (ILU(0) / IC(0), mod_uns_linsolver.f90:79-142, :328-399).
//
// A level holds the rows whose lower (forward) or upper (backward)
// neighbours all lie in earlier levels.  Levels wider than kNarrowRows take
// one launch each, a thread per row.  A run of narrower levels takes one
// workgroup that steps through it: on lexicographic meshes such a run is the
// whole sweep, a serial chain of hundreds of levels of a few hundred rows,
// so its time is the latency of one level times their number.
#include <type_traits>

#include "ms_linalg.hpp"
#include "ms_reduce.hpp"

namespace ms {
namespace {

constexpr double kTiny = 2.2250738585072014e-308;   // tiny(1.0_dp)

struct LMat {
  const long long *off;
  const int *rowlen, *col, *diagk;
};
LMat lmat(const SellPattern &p) { return LMat{p.d_off.p, p.d_rowlen.p, p.d_col.p, p.d_diagk.p}; }

// natural IC(0) of row i, its lower neighbours final (mod_uns_linsolver.f90:328-365)
template <class T>
__device__ void ic0_factor_row(int i, const LMat &A, T *F, int *flag) {
  const long long bi = A.off[i >> 6] + (i & 63);
  const int dpi = A.diagk[i];
  for (int kp = 0; kp < dpi; kp++) {
    const long long qkp = bi + (long long)kp * kSlice;
    const int k = A.col[qkp];
    const long long bk = A.off[k >> 6] + (k & 63);
    const int dpk = A.diagk[k];
    int p = 0, q = 0;
    T dsum = T(0);
    while (p <= kp - 1 && q <= dpk - 1) {
      const int cp = A.col[bi + (long long)p * kSlice], cq = A.col[bk + (long long)q * kSlice];
      if (cp < cq) p++;
      else if (cp > cq) q++;
      else {
        dsum = dsum + F[bi + (long long)p * kSlice] * F[bk + (long long)q * kSlice];
        p++;
        q++;
      }
    }
    const T s = F[qkp] - dsum;
    F[qkp] = s / F[bk + (long long)dpk * kSlice];
  }
  const long long qd = bi + (long long)dpi * kSlice;
  T s = F[qd];
  for (int kp = 0; kp < dpi; kp++) {
    const T v = F[bi + (long long)kp * kSlice];
    s = s - v * v;
  }
  if (s <= T(0)) {
    *flag = 2;
    return;
  }
  F[qd] = tsqrt(s);
}

// natural ILU(0) of row i, IKJ variant (mod_uns_linsolver.f90:79-115)
template <class T>
__device__ void ilu0_factor_row(int i, const LMat &A, T *F, int *flag) {
  const long long bi = A.off[i >> 6] + (i & 63);
  const int dpi = A.diagk[i], leni = A.rowlen[i];
  for (int kk = 0; kk < dpi; kk++) {
    const long long q = bi + (long long)kk * kSlice;
    const int k = A.col[q];
    const long long bk = A.off[k >> 6] + (k & 63);
    const int dpk = A.diagk[k], lenk = A.rowlen[k];
    const T piv = F[bk + (long long)dpk * kSlice];
    if (tabs(piv) < (T)kTiny) {
      *flag = 2;
      return;
    }
    const T aik = F[q] / piv;
    F[q] = aik;
    for (int jj = dpk; jj < lenk; jj++) {
      const int j = A.col[bk + (long long)jj * kSlice];
      if (j <= k) continue;
      for (int m = 0; m < leni; m++) {
        const long long qm = bi + (long long)m * kSlice;
        const int cm = A.col[qm];
        if (cm == j) {
          F[qm] = F[qm] - aik * F[bk + (long long)jj * kSlice];
          break;
        }
        if (cm > j) break;
      }
    }
  }
}

// one wide level: a thread per row
template <class T>
__global__ void k_factor_level(const int *rows, int nr, LMat A, T *F, int ic0, int *flag) {
  int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= nr) return;
  if (ic0) ic0_factor_row(rows[t], A, F, flag);
  else ilu0_factor_row(rows[t], A, F, flag);
}

// a run of narrow levels [l0, l1) in one workgroup: rows of a level are
// spread over the threads, a barrier orders the levels (the workgroup shares
// one L1, so rows of the next level see the values just stored).  Every
// thread reaches every barrier: the level loop is uniform, only the row loop
// inside a level depends on the thread.
template <class T>
__global__ __launch_bounds__(kSegThreads) void k_factor_seg(const int *lev_ptr, int l0, int l1, const int *rows,
                                                             LMat A, T *F, int ic0, int *flag) {
  for (int l = l0; l < l1; l++) {
    const int a = lev_ptr[l], b = lev_ptr[l + 1];
    for (int t = a + (int)threadIdx.x; t < b; t += kSegThreads) {
      if (ic0) ic0_factor_row(rows[t], A, F, flag);
      else ilu0_factor_row(rows[t], A, F, flag);
    }
    __syncthreads();
  }
}

// --------------------------------------------------------- unpacked sweeps
// Patterns that are not packed (sweep_packs): the same two launch forms, from
// the factor in the matrix's own layout.

// forward substitution of row i (unit lower for ILU(0), L of IC(0))
template <class T>
__device__ void lower_row(int i, const LMat &A, const T *F, const T *r, T *z, int ic0) {
  const long long bi = A.off[i >> 6] + (i & 63);
  const int dpi = A.diagk[i];
  T s = r[i];
  for (int k = 0; k < dpi; k++) {
    const long long q = bi + (long long)k * kSlice;
    s = s - F[q] * z[A.col[q]];
  }
  z[i] = ic0 ? s / F[bi + (long long)dpi * kSlice] : s;
}

// backward substitution of row i (U of ILU(0), L^T of IC(0) via tpos)
template <class T>
__device__ void upper_row(int i, const LMat &A, const long long *tpos, const T *F, T *z, int ic0) {
  const long long bi = A.off[i >> 6] + (i & 63);
  const int dpi = A.diagk[i], len = A.rowlen[i];
  T s = z[i];
  if (ic0) {
    for (int k = len - 1; k > dpi; k--) {
      const long long q = bi + (long long)k * kSlice;
      s = s - F[tpos[q]] * z[A.col[q]];
    }
  } else {
    for (int k = dpi + 1; k < len; k++) {
      const long long q = bi + (long long)k * kSlice;
      s = s - F[q] * z[A.col[q]];
    }
  }
  z[i] = s / F[bi + (long long)dpi * kSlice];
}

template <class T>
__global__ void k_lower_level(const int *rows, int nr, LMat A, const T *F, const T *r, T *z, int ic0,
                              const int *done) {
  if (*done) return;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t < nr) lower_row(rows[t], A, F, r, z, ic0);
}
template <class T>
__global__ void k_upper_level(const int *rows, int nr, LMat A, const long long *tpos, const T *F, T *z, int ic0,
                              const int *done) {
  if (*done) return;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t < nr) upper_row(rows[t], A, tpos, F, z, ic0);
}
template <class T>
__global__ __launch_bounds__(kSegThreads) void k_lower_seg(const int *lev_ptr, int l0, int l1, const int *rows,
                                                           LMat A, const T *F, const T *r, T *z, int ic0,
                                                           const int *done) {
  if (*done) return;
  for (int l = l0; l < l1; l++) {
    const int a = lev_ptr[l], b = lev_ptr[l + 1];
    for (int t = a + (int)threadIdx.x; t < b; t += kSegThreads) lower_row(rows[t], A, F, r, z, ic0);
    __syncthreads();
  }
}
template <class T>
__global__ __launch_bounds__(kSegThreads) void k_upper_seg(const int *lev_ptr, int l0, int l1, const int *rows,
                                                           LMat A, const long long *tpos, const T *F, T *z, int ic0,
                                                           const int *done) {
  if (*done) return;
  for (int l = l0; l < l1; l++) {
    const int a = lev_ptr[l], b = lev_ptr[l + 1];
    for (int t = a + (int)threadIdx.x; t < b; t += kSegThreads) upper_row(rows[t], A, tpos, F, z, ic0);
    __syncthreads();
  }
}

// ------------------------------------------------------------ packed sweeps
// One workgroup steps through a run of narrow levels.  A step is a level, or
// a part of at most kSegThreads rows of a wider one; a row's place in the
// level order is its position.
//
// What bounds it is the latency of one step times the number of steps, so
// everything that does not depend on the step before is taken off that
// chain: the factor's off-diagonal entries of each row are packed in step
// order (pcol: the neighbour's position, pval: the value; entry k of lane t
// at base + k * stride + t), so they load coalesced and without the SELL
// offsets, and they, the row ids and the right-hand side are fetched three
// steps ahead into registers.  The solution of the last kRing positions
// stays in LDS, so a step costs an LDS read per entry, the row's arithmetic,
// an LDS write and one barrier that waits for LDS only (the loads in flight
// and the stores to `out` go on across it).  A step that reads a position
// older than the ring takes it from `out` behind a full barrier, which
// orders this workgroup's stores.
// One FP64 sweep of a 40^3 hex grid (118 levels of up to 1200 rows) went
// from 541 us (lower) and 698 us (upper) to 84 us each, and of a 128^2
// cavity (255 levels of up to 128 rows) from 170 and 189 us to 62 and 64 us:
// 0.25 us a level where the level is its latency, about 45 GB/s where it is
// wide, which is what one compute unit draws.
constexpr int kRing = 16384;   // positions kept in LDS (128 KB in FP64)
constexpr int kOrderedBlock = 512;   // widest level (in whole wavefronts) from which vectors go in level order
constexpr int kAheadRows = 3, kAheadOrdered = 4;   // steps fetched ahead (vectors in row order / level order)

// LDS only: a release of the ring's writes, no wait for loads or stores in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <class T, int W>
struct Ahead {
  T rhs, dg, v[W], x[W];
  int c[W];
};

// W: entries per row fetched ahead; MORE: rows may have more than W
// ORDERED: in and out are in level order (rows is not read), else in row order
// DIV: divide by the factor's diagonal (U of ILU(0), L and L^T of IC(0))
// DESC: the entries in descending column order (L^T of IC(0)), as the
// reference's loops run
// FAC: the diagonal of a factorization instead of a sweep (factor_levels):
// 1 ILU(0), 2 IC(0); pval2 holds the transposed entries, flag a breakdown
template <class T, int W, bool MORE, bool ORDERED, bool DIV, bool DESC, int FAC = 0>
__global__ __launch_bounds__(kSegThreads) void k_sweep_seg(const SweepStep *__restrict__ steps, int nsteps, int seg0,
                                                           const int *__restrict__ rows,
                                                           const int *__restrict__ pcol,
                                                           const T *__restrict__ pval, const T *__restrict__ pdiag,
                                                           const T *in, T *out, const int *done,
                                                           const T *__restrict__ pval2 = nullptr,
                                                           int *flag = nullptr) {
  if (FAC == 0 && *done) return;
  constexpr T pad = FAC ? T(1) : T(0);   // the value padding reads
  __shared__ T ring[kRing + 1];
  const int t = threadIdx.x;
  if (t == 0) ring[kRing] = pad;
  __syncthreads();
  // constant address space: the steps come through scalar loads, which do
  // not queue behind the fetches
  typedef const __attribute__((address_space(4))) SweepStep *StepPtr;
  const StepPtr sp = (StepPtr)(unsigned long long)steps;
  auto desc = [&](int s) { return SweepStep{sp[s].t0, sp[s].n, sp[s].w, sp[s].near, sp[s].base, sp[s].stride}; };
  // the loads of lanes beyond a step's rows go to its last row: no branch
  // around them, so nothing waits for them before their step
  auto lane = [&](const SweepStep &d) { return (unsigned)min(t, max(d.n, 1) - 1); };
  // uniform pointers plus a 32-bit lane index: one vector instruction per
  // load, which matters as much as the latency does (16 wavefronts share
  // four SIMDs)
  auto fetch = [&](Ahead<T, W> &a, const SweepStep &d, int row) {
    const unsigned l = lane(d);
    const int stride = d.stride;
    const int *pc = pcol + d.base;
    const T *pv = pval + d.base;
    const T *pw = FAC == 1 ? pval2 + d.base : nullptr;
    if (FAC) a.rhs = (pdiag + d.t0)[l];
    else if (ORDERED) a.rhs = (in + d.t0)[l];
    else a.rhs = in[row];
    if (DIV) a.dg = (pdiag + d.t0)[l];
#pragma unroll
    for (int k = 0; k < W; k++) {
      a.c[k] = pc[l];
      a.v[k] = pv[l];
      if (FAC == 1) a.x[k] = pw[l];
      pc += stride;
      pv += stride;
      if (FAC == 1) pw += stride;
    }
  };
  // one entry's share of the row's sum; z: the neighbour's value
  auto term = [&](T &sum, T v, T x, T z) {
    if constexpr (FAC == 0) {
      sum = sum - v * z;   // padding: 0 * 0, which leaves the sum as it is
    } else {
      if (FAC == 1 && tabs(z) < (T)kTiny) *flag = 2;
      const T f = v / z;   // padding: 0 / 1
      sum = sum - f * (FAC == 1 ? x : f);
    }
  };
  // U steps per turn of the loop, so that every register set has a fixed
  // name; in row order the row ids come two steps before what they address
  constexpr int NS = ORDERED ? kAheadOrdered : kAheadRows, U = ORDERED ? NS : 2 * NS, DN = ORDERED ? NS : NS + 2;
  SweepStep d[U];
  int row[U];
  Ahead<T, W> a[NS];
#pragma unroll
  for (int j = 0; j < DN; j++) d[j] = desc(j);
#pragma unroll
  for (int j = 0; j < DN; j++) row[j] = ORDERED ? 0 : (rows + d[j].t0)[lane(d[j])];
#pragma unroll
  for (int j = 0; j < NS; j++) fetch(a[j], d[j], row[j]);
  auto step = [&](auto jc, int s) {
    constexpr int j = decltype(jc)::value;
    Ahead<T, W> &p = a[j % NS];
    const SweepStep e = d[j], next = desc(s + DN);
    const int r = row[j];
    // A step whose neighbours are all in the ring has their ring slots in
    // pcol (the zero slot kRing for padding).  Any other step has positions
    // (-1: padding): those in [lo, e.t0) are in the ring, older ones in `out`
    // behind a barrier that orders this workgroup's stores, those before seg0
    // from earlier launches.
    const bool near = e.near != 0;
    const int lo = max(seg0, e.t0 + e.n - kRing);
    if (!near && lo > seg0) __syncthreads();
    auto solve = [&](auto get) {
      T sum = p.rhs;
      const int stride = e.stride;
      if (MORE && DESC)
        for (int k = e.w - 1; k >= W; k--) {
          const long long q = e.base + (long long)k * stride + t;
          term(sum, pval[q], T(0), get(pcol[q]));
        }
      T z[W];
#pragma unroll
      for (int k = 0; k < W; k++) z[k] = get(p.c[k]);
#pragma unroll
      for (int i = 0; i < W; i++) {
        const int k = DESC ? W - 1 - i : i;
        term(sum, p.v[k], p.x[k], z[k]);
      }
      if (MORE && !DESC)
        for (int k = W; k < e.w; k++) {
          const long long q = e.base + (long long)k * stride + t;
          term(sum, pval[q], FAC == 1 ? pval2[q] : T(0), get(pcol[q]));
        }
      if (DIV) sum = sum / p.dg;
      if (FAC == 2) {
        if (sum <= T(0)) *flag = 2;
        else sum = tsqrt(sum);
      }
      ring[(e.t0 + t) & (kRing - 1)] = sum;
      if (ORDERED) (out + e.t0)[(unsigned)t] = sum;
      else out[r] = sum;
    };
    // two bodies: one select between an LDS and a memory address would make
    // every read a flat load, which waits for the fetches in flight
    if (near) {
      if (t < e.n) solve([&](int c) { return ring[c]; });
    } else if (t < e.n) {
      solve([&](int c) {
        T v = c >= lo ? ring[c & (kRing - 1)] : (c < 0 ? pad : out[ORDERED ? c : rows[c]]);
        asm volatile("" : "+v"(v));   // waited for here, not where the two bodies' common code begins
        return v;
      });
    }
    lds_barrier();
    d[(j + DN) % U] = next;
    fetch(p, d[(j + NS) % U], row[(j + NS) % U]);
    if (!ORDERED) row[(j + DN) % U] = (rows + next.t0)[lane(next)];
  };
  auto turn = [&](auto self, auto jc, int s) {
    constexpr int j = decltype(jc)::value;
    if constexpr (j < U) {
      if (s + j < nsteps) {
        step(jc, s + j);
        self(self, std::integral_constant<int, j + 1>{}, s);
      }
    }
  };
  for (int s = 0; s < nsteps; s += U) turn(turn, std::integral_constant<int, 0>{}, s);
}

// A wide level: a thread per row, its entries packed as above with the
// neighbours' rows in pcol.  The row id, columns and values are independent
// loads (through the SELL offsets they were a chain of three), and only the
// neighbours' values follow them.  Averages over the levels of multicolour
// ILU(0) sweeps on prisms, four of 48,000 rows: 2.7 us, through the offsets
// 3.7; of 480,000 rows, which memory bounds: 7.8 and 8.9.
template <class T, int W, bool MORE, bool DIV, bool DESC>
__global__ __launch_bounds__(kBlock) void k_sweep_wide(SweepStep d, const int *__restrict__ rows,
                                                       const int *__restrict__ pcol, const T *__restrict__ pval,
                                                       const T *__restrict__ pdiag, const T *in, T *out,
                                                       const int *done) {
  const int dn = *done, t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= d.n) return;
  const int stride = d.stride;
  const int row = rows[d.t0 + t];
  int c[W];
  T v[W], z[W];
#pragma unroll
  for (int k = 0; k < W; k++) c[k] = pcol[d.base + (long long)k * stride + t];
#pragma unroll
  for (int k = 0; k < W; k++) v[k] = pval[d.base + (long long)k * stride + t];
  const T dg = DIV ? pdiag[d.t0 + t] : T(1);
  T sum = in[row];
  if (dn) return;
  auto extra = [&](int k) {
    const long long q = d.base + (long long)k * stride + t;
    const int ck = pcol[q];
    if (ck >= 0) sum = sum - pval[q] * out[ck];
  };
  if (MORE && DESC)
    for (int k = d.w - 1; k >= W; k--) extra(k);
#pragma unroll
  for (int k = 0; k < W; k++) z[k] = c[k] >= 0 ? out[c[k]] : T(0);
#pragma unroll
  for (int i = 0; i < W; i++) {
    const int k = DESC ? W - 1 - i : i;
    sum = c[k] >= 0 ? sum - v[k] * z[k] : sum;
  }
  if (MORE && !DESC)
    for (int k = W; k < d.w; k++) extra(k);
  out[row] = DIV ? sum / dg : sum;
}

// the same for a wide level of a factorization's diagonal
template <int FAC>
__global__ __launch_bounds__(kBlock) void k_diag_wide(SweepStep d, const int *rows, const int *pcol,
                                                      const double *pval, const double *pval2, const double *pdiag,
                                                      double *out, int *flag) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= d.n) return;
  const int stride = d.stride;
  double sum = pdiag[d.t0 + t];
  for (int k = 0; k < d.w; k++) {
    const long long q = d.base + (long long)k * stride + t;
    const int c = pcol[q];
    if (c < 0) continue;
    const double z = out[c];
    if (FAC == 1 && tabs(z) < kTiny) *flag = 2;
    const double f = pval[q] / z;
    sum = sum - f * (FAC == 1 ? pval2[q] : f);
  }
  if (FAC == 2) {
    if (sum <= 0.0) *flag = 2;
    else sum = sqrt(sum);
  }
  out[rows[d.t0 + t]] = sum;
}

// the factor in place of the matrix, given its diagonal d: entries below the
// diagonal divided by their column's
__global__ void k_diag_fill(int n, LMat A, const double *d, double *F) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const long long bi = A.off[i >> 6] + (i & 63);
  const int dk = A.diagk[i];
  for (int k = 0; k < dk; k++) {
    const long long q = bi + (long long)k * kSlice;
    F[q] = F[q] / d[A.col[q]];
  }
  F[bi + (long long)dk * kSlice] = d[i];
}

// *found = 1 when some row and a neighbour of it share a neighbour
__global__ void k_find_triangle(int n, LMat A, int *found) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n || *found) return;
  const long long bi = A.off[i >> 6] + (i & 63);
  const int li = A.rowlen[i];
  for (int a = 0; a < li; a++) {
    const int k = A.col[bi + (long long)a * kSlice];
    if (k >= i) break;
    const long long bk = A.off[k >> 6] + (k & 63);
    const int lk = A.rowlen[k];
    for (int p = 0, q = 0; p < li && q < lk;) {
      const int ci = A.col[bi + (long long)p * kSlice], ck = A.col[bk + (long long)q * kSlice];
      if (ci == ck && ci != i && ci != k) {
        *found = 1;
        return;
      }
      if (ci <= ck) p++;
      if (ck <= ci) q++;
    }
  }
}

__global__ void k_pack_cols_wide(SweepStep d, const int *rows, LMat A, int upper, int *pcol) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= d.n) return;
  const int stride = d.stride;
  const int r = rows[d.t0 + t], dk = A.diagk[r];
  const long long br = A.off[r >> 6] + (r & 63);
  const int k0 = upper ? dk + 1 : 0, m = upper ? A.rowlen[r] - dk - 1 : dk;
  for (int k = 0; k < d.w; k++)
    pcol[d.base + (long long)k * stride + t] = k < m ? A.col[br + (long long)(k0 + k) * kSlice] : -1;
}

// pcol of every step's rows (one workgroup per step of a run whose first
// position is seg0): ring slots where all neighbours will be in the ring,
// else positions; upper: the entries above the diagonal
__global__ void k_pack_cols(SweepStep *steps, int seg0, const int *rows, const int *pos, LMat A, int upper,
                            int *pcol) {
  const SweepStep d = steps[blockIdx.x];
  const int stride = d.stride;
  __shared__ int far;
  if (threadIdx.x == 0) far = 0;
  __syncthreads();
  for (int pass = 0; pass < 2; pass++) {
    const bool near = pass == 1 && !far;
    for (int t = threadIdx.x; t < d.n; t += kBlock) {
      const int r = rows[d.t0 + t], dk = A.diagk[r];
      const long long br = A.off[r >> 6] + (r & 63);
      const int k0 = upper ? dk + 1 : 0, m = upper ? A.rowlen[r] - dk - 1 : dk;
      for (int k = 0; k < d.w; k++) {
        const int c = k < m ? pos[A.col[br + (long long)(k0 + k) * kSlice]] : -1;
        if (pass == 0) {
          if (k < m && c < max(seg0, d.t0 + d.n - kRing)) far = 1;
        } else {
          pcol[d.base + (long long)k * stride + t] = !near ? c : (c < 0 ? kRing : c & (kRing - 1));
        }
      }
    }
    __syncthreads();
    if (near && threadIdx.x == 0) steps[blockIdx.x].near = 1;
  }
}

// the factor's entries and diagonal in step order (tpos: L^T of IC(0))
template <class T>
__global__ void k_pack_vals(const SweepStep *steps, const int *rows, LMat A, int upper, const long long *tpos,
                            const T *F, T *pval, T *pdiag) {
  const SweepStep d = steps[blockIdx.x];
  const int stride = d.stride;
  for (int t = blockIdx.y * kBlock + threadIdx.x; t < d.n; t += kBlock * gridDim.y) {
    const int r = rows[d.t0 + t], dk = A.diagk[r];
    const long long br = A.off[r >> 6] + (r & 63);
    const int k0 = upper ? dk + 1 : 0, m = upper ? A.rowlen[r] - dk - 1 : dk;
    for (int k = 0; k < m; k++) {
      const long long q = br + (long long)(k0 + k) * kSlice;
      pval[d.base + (long long)k * stride + t] = F[tpos ? tpos[q] : q];
    }
    for (int k = m; k < d.w; k++) pval[d.base + (long long)k * stride + t] = T(0);
    pdiag[d.t0 + t] = F[br + (long long)dk * kSlice];
  }
}

template <class T>
__global__ void k_gather(int n, const int *idx, const T *in, T *out, const int *done) {
  if (*done) return;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t < n) out[t] = in[idx[t]];
}
template <class T>
__global__ void k_scatter(int n, const int *idx, const T *in, T *out, const int *done) {
  if (*done) return;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t < n) out[idx[t]] = in[t];
}

}  // namespace

// The steps of every run of narrow levels, and their packed columns.
void plan_sweeps(SellPattern &P, const std::vector<int> &rows_f, const std::vector<int> &rows_b) {
  const SweepSteps F = sweep_steps(P.lev_ptr_f, P.seg_f, [&](int t) { return P.diagk[rows_f[t]]; });
  const SweepSteps B = sweep_steps(P.lev_ptr_b, P.seg_b, [&](int t) {
    return P.rowlen[rows_b[t]] - P.diagk[rows_b[t]] - 1;
  });
  P.sweep_packed = sweep_packs(F.nent + B.nent, P.nstore);
  P.triangle_free = P.sweep_ordered = false;
  if (!P.sweep_packed) return;
  auto plan = [&](bool upper, const SweepSteps &H, const std::vector<int> &rows, const std::vector<LevSeg> &segs,
                  SweepPlan &S, const DBuf<int> &d_rows) {
    S.width = H.width;
    S.more = H.more;
    S.nent = H.nent;
    S.nsteps = (int)H.st.size();
    if (!S.nsteps) return;
    std::vector<int> pos(P.n);
    for (int t = 0; t < P.n; t++) pos[rows[t]] = t;
    DBuf<int> d_pos;
    d_pos.upload(pos);
    S.steps.upload(H.st);
    S.col.alloc(std::max<long long>(S.nent, 1));
    for (const auto &g : segs)
      if (g.narrow)
        hipLaunchKernelGGL(k_pack_cols, dim3(g.s1 - g.s0), dim3(kBlock), 0, stream(), S.steps.p + g.s0, g.t0,
                           d_rows.p, d_pos.p, lmat(P), (int)upper, S.col.p);
      else
        hipLaunchKernelGGL(k_pack_cols_wide, dim3(nblocks(g.step.n)), dim3(kBlock), 0, stream(), g.step, d_rows.p,
                           lmat(P), (int)upper, S.col.p);
    MS_CHECK_LAUNCH();
    MS_HIP(hipStreamSynchronize(stream()));   // the host arrays above and d_pos go out of scope
  };
  plan(false, F, rows_f, P.seg_f, P.sweep_f, P.d_lev_rows_f);
  plan(true, B, rows_b, P.seg_b, P.sweep_b, P.d_lev_rows_b);
  // Vectors in level order: the rows of a level are far apart in row order
  // (a diagonal plane of a grid), so reading and writing them there costs
  // the one workgroup a cache line per row, 150 us per sweep against 84
  // on a 40^3 grid; three launches of 4 us that permute for the whole chip cost
  // less once levels are this wide.  On a 128^2 grid (levels of at most 128
  // rows) a step is its latency either way and the launches would be lost.
  DBuf<int> found(1);
  int h = 0;
  MS_HIP(hipMemsetAsync(found.p, 0, sizeof(int), stream()));
  hipLaunchKernelGGL(k_find_triangle, dim3(nblocks(P.n)), dim3(kBlock), 0, stream(), P.n, lmat(P), found.p);
  MS_CHECK_LAUNCH();
  found.download(&h, 1);
  MS_HIP(hipStreamSynchronize(stream()));
  P.triangle_free = h == 0;
  P.sweep_ordered = P.seg_f.size() == 1 && P.seg_b.size() == 1 && P.seg_f[0].narrow && P.seg_b[0].narrow &&
                    P.seg_f[0].block >= kOrderedBlock;
  if (P.sweep_ordered) {
    std::vector<int> pos_f(P.n), fb(P.n);
    for (int t = 0; t < P.n; t++) pos_f[rows_f[t]] = t;
    for (int t = 0; t < P.n; t++) fb[t] = pos_f[rows_b[t]];
    P.d_lev_fb.upload(fb);
    MS_HIP(hipStreamSynchronize(stream()));
  }
}

// the factor F (SELL layout) in the order of the packed sweeps
template <class T>
void LevelFactor<T>::pack(const SellPattern &P, const T *F, bool ic0) {
  if (!P.sweep_packed) return;
  auto one = [&](const SweepPlan &S, const DBuf<int> &rows, DBuf<T> &v, DBuf<T> &d, bool upper) {
    if (!S.nsteps) return;
    if (v.n < (size_t)S.nent) v.alloc(S.nent);
    if (d.n < (size_t)P.n) d.alloc(P.n);
    // enough workgroups per step for the widest level
    int widest = 1;
    for (const auto &g : upper ? P.seg_b : P.seg_f)
      if (!g.narrow) widest = std::max(widest, nblocks(g.step.n));
    hipLaunchKernelGGL(k_pack_vals<T>, dim3(S.nsteps, std::min(widest, 64)), dim3(kBlock), 0, stream(), S.steps.p, rows.p, lmat(P),
                       (int)upper, ic0 && upper ? P.d_tpos.p : nullptr, F, v.p, d.p);
  };
  one(P.sweep_f, P.d_lev_rows_f, vf, df, false);
  one(P.sweep_b, P.d_lev_rows_b, vb, db, true);
  MS_CHECK_LAUNCH();
}

template <class T, bool DIV, bool DESC>
static void sweep_run(const SweepPlan &S, const LevSeg &g, const int *rows, const T *v, const T *d,
                      const T *in, T *out, const int *done) {
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, dim3(1), dim3(g.block), 0, stream(), S.steps.p + g.s0, g.s1 - g.s0, g.t0, rows, S.col.p, v,
                       d, in, out, done, (const T *)nullptr, (int *)nullptr);
  };
  auto by_width = [&](auto ordered) {
    constexpr bool O = decltype(ordered)::value;
    if (S.more) go(k_sweep_seg<T, kPre, true, O, DIV, DESC>);
    else if (S.width == 4) go(k_sweep_seg<T, 4, false, O, DIV, DESC>);
    else if (S.width == 3) go(k_sweep_seg<T, 3, false, O, DIV, DESC>);
    else if (S.width == 2) go(k_sweep_seg<T, 2, false, O, DIV, DESC>);
    else go(k_sweep_seg<T, 1, false, O, DIV, DESC>);
  };
  if (rows) by_width(std::false_type{});
  else by_width(std::true_type{});
}

template <class T, bool DIV, bool DESC>
static void sweep_wide(const SweepPlan &S, const LevSeg &g, const int *rows, const T *v, const T *d,
                       const T *in, T *out, const int *done) {
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, dim3(nblocks(g.step.n)), dim3(kBlock), 0, stream(), g.step, rows, S.col.p, v, d, in, out,
                       done);
  };
  // by the level's own width: with colour classes it goes from none below the
  // first class to all of a row's neighbours below the last
  if (g.step.w > kPre) go(k_sweep_wide<T, kPre, true, DIV, DESC>);
  else if (g.step.w == 4) go(k_sweep_wide<T, 4, false, DIV, DESC>);
  else if (g.step.w == 3) go(k_sweep_wide<T, 3, false, DIV, DESC>);
  else if (g.step.w == 2) go(k_sweep_wide<T, 2, false, DIV, DESC>);
  else go(k_sweep_wide<T, 1, false, DIV, DESC>);
}

// out = (L U)^-1 in or (L L^T)^-1 in
template <class T>
void LevelFactor<T>::apply(const SellPattern &P, bool ic0, const T *F, const T *in, T *out, const int *done) {
  hipStream_t S = stream();
  const dim3 G(nblocks(P.n)), B(kBlock);
  if (!P.sweep_packed) {
    const LMat A = lmat(P);
    for (const auto &g : P.seg_f) {
      const int a = P.lev_ptr_f[g.l0], m = P.lev_ptr_f[g.l1] - a;
      if (g.narrow)
        hipLaunchKernelGGL(k_lower_seg<T>, dim3(1), dim3(kSegThreads), 0, S, P.d_lev_ptr_f.p, g.l0, g.l1,
                           P.d_lev_rows_f.p, A, F, in, out, (int)ic0, done);
      else
        hipLaunchKernelGGL(k_lower_level<T>, dim3(nblocks(m)), B, 0, S, P.d_lev_rows_f.p + a, m, A, F, in, out,
                           (int)ic0, done);
    }
    for (const auto &g : P.seg_b) {
      const int a = P.lev_ptr_b[g.l0], m = P.lev_ptr_b[g.l1] - a;
      if (g.narrow)
        hipLaunchKernelGGL(k_upper_seg<T>, dim3(1), dim3(kSegThreads), 0, S, P.d_lev_ptr_b.p, g.l0, g.l1,
                           P.d_lev_rows_b.p, A, P.d_tpos.p, F, out, (int)ic0, done);
      else
        hipLaunchKernelGGL(k_upper_level<T>, dim3(nblocks(m)), B, 0, S, P.d_lev_rows_b.p + a, m, A, P.d_tpos.p, F,
                           out, (int)ic0, done);
    }
    MS_CHECK_LAUNCH();
    return;
  }
  auto fwd = [&](const LevSeg &g, const int *rows, const T *x, T *y) {
    if (ic0) sweep_run<T, true, false>(P.sweep_f, g, rows, vf.p, df.p, x, y, done);
    else sweep_run<T, false, false>(P.sweep_f, g, rows, vf.p, df.p, x, y, done);
  };
  auto bwd = [&](const LevSeg &g, const int *rows, const T *x, T *y) {
    if (ic0) sweep_run<T, true, true>(P.sweep_b, g, rows, vb.p, db.p, x, y, done);
    else sweep_run<T, true, false>(P.sweep_b, g, rows, vb.p, db.p, x, y, done);
  };
  if (P.sweep_ordered) {
    if (xf.n < (size_t)P.n) xf.alloc(P.n);
    if (xb.n < (size_t)P.n) xb.alloc(P.n);
    hipLaunchKernelGGL(k_gather<T>, G, B, 0, S, P.n, P.d_lev_rows_f.p, in, xf.p, done);
    fwd(P.seg_f[0], nullptr, xf.p, xf.p);
    hipLaunchKernelGGL(k_gather<T>, G, B, 0, S, P.n, P.d_lev_fb.p, xf.p, xb.p, done);
    bwd(P.seg_b[0], nullptr, xb.p, xb.p);
    hipLaunchKernelGGL(k_scatter<T>, G, B, 0, S, P.n, P.d_lev_rows_b.p, xb.p, out, done);
    MS_CHECK_LAUNCH();
    return;
  }
  for (const auto &g : P.seg_f) {
    if (g.narrow) {
      fwd(g, P.d_lev_rows_f.p, in, out);
      continue;
    }
    if (ic0) sweep_wide<T, true, false>(P.sweep_f, g, P.d_lev_rows_f.p, vf.p, df.p, in, out, done);
    else sweep_wide<T, false, false>(P.sweep_f, g, P.d_lev_rows_f.p, vf.p, df.p, in, out, done);
  }
  for (const auto &g : P.seg_b) {
    if (g.narrow) {
      bwd(g, P.d_lev_rows_b.p, out, out);
      continue;
    }
    if (ic0) sweep_wide<T, true, true>(P.sweep_b, g, P.d_lev_rows_b.p, vb.p, db.p, out, out, done);
    else sweep_wide<T, true, false>(P.sweep_b, g, P.d_lev_rows_b.p, vb.p, db.p, out, out, done);
  }
  MS_CHECK_LAUNCH();
}

// F (holding the matrix) becomes its ILU(0) / IC(0) factor; *flag = 2 on a
// breakdown.  Where no two neighbours share a neighbour (structured and most
// prismatic meshes) no entry of the factor receives fill from another, so
// only the diagonal is a recurrence,
//   ILU(0): d_i = a_ii - sum_k (a_ik / d_k) a_ki,
//   IC(0):  d_i = sqrt(a_ii - sum_k (a_ik / d_k)^2),
// in the order and with the operations of the general elimination: it runs
// as a sweep, and the entries below the diagonal follow in one launch.  The
// general kernels' merges of two rows' columns took 1.64 ms for a 128^2
// cavity (255 levels), this 0.12 ms.
void factor_levels(const SellPattern &P, double *F, bool ic0, int *flag, DiagFactor &D) {
  const LMat A = lmat(P);
  hipStream_t S = stream();
  if (P.symmetric && P.triangle_free) {
    const SweepPlan &W = P.sweep_f;
    if (D.lo.n < (size_t)W.nent) D.lo.alloc(W.nent);
    if (!ic0 && D.up.n < (size_t)W.nent) D.up.alloc(W.nent);
    if (D.dg.n < (size_t)P.n) D.dg.alloc(P.n);
    if (D.d.n < (size_t)P.n) D.d.alloc(P.n);
    int widest = 1;
    for (const auto &g : P.seg_f)
      if (!g.narrow) widest = std::max(widest, nblocks(g.step.n));
    const dim3 G(W.nsteps, std::min(widest, 64)), B(kBlock);
    const int *rows = P.d_lev_rows_f.p;
    hipLaunchKernelGGL(k_pack_vals<double>, G, B, 0, S, W.steps.p, rows, A, 0, (const long long *)nullptr, F, D.lo.p,
                       D.dg.p);
    if (!ic0)
      hipLaunchKernelGGL(k_pack_vals<double>, G, B, 0, S, W.steps.p, rows, A, 0, P.d_tpos.p, F, D.up.p, D.dg.p);
    for (const auto &g : P.seg_f) {
      auto seg = [&](auto k) {
        hipLaunchKernelGGL(k, dim3(1), dim3(g.block), 0, S, W.steps.p + g.s0, g.s1 - g.s0, g.t0, rows, W.col.p, D.lo.p,
                           D.dg.p, (const double *)nullptr, D.d.p, (const int *)nullptr, D.up.p, flag);
      };
      if (!g.narrow) {
        if (ic0)
          hipLaunchKernelGGL(k_diag_wide<2>, dim3(nblocks(g.step.n)), B, 0, S, g.step, rows, W.col.p, D.lo.p, D.up.p,
                             D.dg.p, D.d.p, flag);
        else
          hipLaunchKernelGGL(k_diag_wide<1>, dim3(nblocks(g.step.n)), B, 0, S, g.step, rows, W.col.p, D.lo.p, D.up.p,
                             D.dg.p, D.d.p, flag);
      } else if (W.more) {
        if (ic0) seg(k_sweep_seg<double, kPre, true, false, false, false, 2>);
        else seg(k_sweep_seg<double, kPre, true, false, false, false, 1>);
      } else if (W.width > 2) {
        if (ic0) seg(W.width == 4 ? k_sweep_seg<double, 4, false, false, false, false, 2>
                                  : k_sweep_seg<double, 3, false, false, false, false, 2>);
        else seg(W.width == 4 ? k_sweep_seg<double, 4, false, false, false, false, 1>
                              : k_sweep_seg<double, 3, false, false, false, false, 1>);
      } else {
        if (ic0) seg(W.width == 2 ? k_sweep_seg<double, 2, false, false, false, false, 2>
                                  : k_sweep_seg<double, 1, false, false, false, false, 2>);
        else seg(W.width == 2 ? k_sweep_seg<double, 2, false, false, false, false, 1>
                              : k_sweep_seg<double, 1, false, false, false, false, 1>);
      }
    }
    hipLaunchKernelGGL(k_diag_fill, dim3(nblocks(P.n)), B, 0, S, P.n, A, D.d.p, F);
    MS_CHECK_LAUNCH();
    return;
  }
  for (const auto &g : P.seg_f) {
    if (g.narrow) {
      hipLaunchKernelGGL(k_factor_seg<double>, dim3(1), dim3(kSegThreads), 0, stream(), P.d_lev_ptr_f.p, g.l0, g.l1,
                         P.d_lev_rows_f.p, A, F, (int)ic0, flag);
      continue;
    }
    const int a = P.lev_ptr_f[g.l0], b = P.lev_ptr_f[g.l1];
    hipLaunchKernelGGL(k_factor_level<double>, dim3(nblocks(b - a)), dim3(kBlock), 0, stream(), P.d_lev_rows_f.p + a,
                       b - a, A, F, (int)ic0, flag);
  }
  MS_CHECK_LAUNCH();
}

template struct LevelFactor<double>;
template struct LevelFactor<float>;

}  // namespace ms

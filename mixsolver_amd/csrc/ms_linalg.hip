// ms_linalg.hip -- SELL-64 sparse kernels and device-resident Krylov solvers
// for gfx950.
//
// Recurrences follow the reference solvers at one partition
// (mod_uns_linsolver_mpi.f90: bicgstab_ilu0_mpi :155-229, cg_jacobi_mpi
// :235-300, cg_ic0_mpi :306-363; factorizations mod_uns_linsolver.f90:79-142
// and :328-399).  Scalars (alpha, beta, rho, omega, residuals, iteration
// count, breakdown flags) live in device memory; every workgroup of the
// launch that needs a reduced value sums the partials of the launch before in
// a fixed order, and one of them keeps the state, so an iteration needs no
// host round trip.  The host enqueues iterations in chunks and reads the
// state once per chunk; every iteration kernel returns at once when the
// state says done.
//
// Launches per PCG iteration:
//   no coarse space, Jacobi: [p = z + beta p, q = A p, p.q] [x,r update, r.r, r.z]
//   (one launch a solve on small FP64 systems, k_cg_small), and otherwise with
//   the sweeps and r.z between the two;
//   coarse space: [q = A p, p.q] (two launches matrix-free) [x,r update, r.r,
//   r.(r/d), Z^T r] [sweeps of DILU, with nu = E^-1 Z^T r riding the first;
//   Jacobi: nu in a launch of its own] [p = z + nu + beta p].
// Vectors are templated on the value type: double for the FP64 path, float
// for the inner iterations of mixed precision (FP32 products and FP32
// accumulation of dot-product partials; scalar recurrences in double).
#include <atomic>
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include <hip/hip_ext.h>

#include "ms_kernels.hpp"
#include "ms_linalg.hpp"

namespace ms {
namespace {

// ------------------------------------------------------------------- PCG
// p = z (+ nu of the row's aggregate); partial r.z of the one-level part
template <class T>
__global__ void k_pcg_start(Rows R, const T *r, const T *z, const T *dg, int jac, T *p, const double *nu,
                            const KS *st, T *part) {
  if (st->done) return;
  int i, a;
  T v[1] = {T(0)};
  if (R.get(i, a)) {
    T zi = jac ? r[i] / dg[i] : z[i];
    p[i] = nu ? zi + (T)nu[a] : zi;
    v[0] = r[i] * zi;
  }
  block_partials<OpSum, 1>(v, part);
}

// partials (0, 0, sum r) per row set: Z^T r of the initial residual
template <class T>
__global__ void k_rsum(Rows R, const T *r, const KS *st, T *part) {
  if (st->done == 1) return;
  int i, a;
  T v[3] = {T(0), T(0), T(0)};
  if (R.get(i, a)) v[2] = r[i];
  block_partials<OpSum, 3>(v, part);
}

template <class T, int C16 = -1>
__global__ void k_pcg_spmv(int n, Mat A, const T *val, const T *p, T *q, const KS *st, T *part) {
  if (st->done) return;
  int i = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  T v[1] = {T(0)};
  if (i < n) {
    const T pi = p[i];   // read before the store to q, which may alias p for the compiler
    const T qi = row_apply<T, C16>(i, A, val, p);
    q[i] = qi;
    v[0] = pi * qi;
  }
  block_partials<OpSum, 1>(v, part);
}

// Matrix-free S p (MatFree): with g_k = sum_j (-a_kj / a_kk) x_j over the
// colour-1 neighbours of colour-0 row k, (S x)_i = sum_k (-a_ik) (x_i - g_k)
// + rowsum_i x_i.  Stage 1 forms, per colour-0 row, h_k = x_ref - g_k =
// sum_j w_kj (x_ref - x_j) + rho_k x_ref with x_ref the row's first
// colour-1 neighbour and rho_k = rowsum_k / a_kk; stage 2 forms
// sum_k (-a_ik) ((x_i - x_ref_k) + h_k) + rowsum_i x_i.  Every term is a
// difference or a row-sum term, as in row_apply's difference form, so a
// constant vector gives the row sums' product exactly.  The slot loop runs
// the slice width of A (diagonal and padding slots have col = row).
// The pending p update of the PCG with a coarse space (p = r/d + nu[agg] +
// beta p, as k_cx_p) can ride along the product (PU): stage 1 forms the
// updated p of each neighbour it reads, stage 2 that of its own row and
// stores it (stage 1 has finished reading the old p by then).  The values are
// those k_cx_p would store, bit for bit.
template <bool PU>
__device__ __forceinline__ float pu_val(int j, const float *p, const PUp &u, float beta, bool up) {
  if constexpr (PU) {
    if (up) {
      const float zj = u.r[j] / u.dg[j] + (float)u.nu[u.agg1[j]];
      return zj + beta * p[j];
    }
  }
  return p[j];
}

// 16-bit columns of the product (k_mf_cols).  Its two stages at 2M cells took 10.4
// and 11.9 us with 32-bit columns and a load per slot, 10.2 and 10.8 so: 52
// bytes a row instead of 64, but the chain offset - column - gather in the two
// rounds of workgroups now takes most of it.
struct MfCols {
  const unsigned short *c16;
  const int *win;
};
// column of slot code o: w holds window v of the row's slice in lane v + at;
// every lane of the wavefront takes part
__device__ __forceinline__ int mf_col(unsigned o, int w, int at, int r) {
  const int b = __shfl(w, (int)(o >> 12) + at, 64);
  return o == 0xFFFFu ? r : b + (int)(o & 4095u);
}

// x_ref (slot 1's column, the row's first colour-1 neighbour) is taken from
// the columns already loaded, so its gather is issued with the others.
// The diagonal comes first in a colour-0 row: its column is the row's own.
template <int W, bool PU>
__device__ __forceinline__ float mf1_row(int k, const unsigned short *c16, int win, const float *w, int n0,
                                         const float *x, float &xr, const PUp &u, float beta, bool up) {
  unsigned o[W];
  float a[W], xv[W];
  mf_load<W>(c16, k & 63, o);
  mf_load<W>(w, k & 63, a);
  int c[W];
#pragma unroll
  for (int j = 0; j < W; j++) c[j] = j == 0 ? k : mf_col(o[j], win, 0, k);
#pragma unroll
  for (int j = 0; j < W; j++) xv[j] = j == 0 || c[j] < n0 ? 0.f : pu_val<PU>(c[j] - n0, x, u, beta, up);
  xr = c[1] >= n0 ? xv[1] : 0.f;
  float acc = 0.f;
#pragma unroll
  for (int j = 0; j < W; j++) acc = acc + a[j] * (j == 0 || c[j] < n0 ? xr : xr - xv[j]);
  return acc;
}

template <bool PU>
__global__ void k_mf_stage1(int n0, Mat A, MfCols m, const float *w, const float *x, float2 *hx, KS *st, PUp u) {
  if (st->done) return;
  float beta = 0.f;
  bool up = false;
  if constexpr (PU) {   // the same for every workgroup: both change between products only
    up = st->pup != 0;
    beta = (float)st->beta;
  }
  // rows beyond the last repeat it without storing: all lanes pass on windows
  const int k1 = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x, k = min(k1, n0 - 1);
  const int s = __builtin_amdgcn_readfirstlane(k >> 6);   // the slice is the wavefront's: scalar loads
  const long long o0 = A.off[s];
  const int wd = (int)((A.off[s + 1] - o0) >> 6);
  const long long base = o0 + (k & 63);
  const int win = m.win[16 * s + (threadIdx.x & 15)];
  const bool near16 = m.win[16 * s + 15] != 0;
  const unsigned short *c16 = m.c16 + o0;
  const float *ws = w + o0;
  // slot 0 is the diagonal (colour-1 columns are above every colour-0 row)
  float xr = 0.f, acc;
  if (wd == 7 && near16) acc = mf1_row<7, PU>(k, c16, win, ws, n0, x, xr, u, beta, up);
  else if (wd == 6 && near16) acc = mf1_row<6, PU>(k, c16, win, ws, n0, x, xr, u, beta, up);
  else if (wd == 5 && near16) acc = mf1_row<5, PU>(k, c16, win, ws, n0, x, xr, u, beta, up);
  else {
    const int c1 = wd > 1 ? A.col[base + kSlice] : k;
    xr = c1 >= n0 ? pu_val<PU>(c1 - n0, x, u, beta, up) : 0.f;
    acc = 0.f;
    for (int j = 0; j < wd; j++) {
      const int c = A.col[base + (long long)j * kSlice];
      acc = acc + ws[mf_pos(wd, j, k & 63)] * (c < n0 ? xr : xr - pu_val<PU>(c - n0, x, u, beta, up));
    }
  }
  if (k1 < n0) hx[k] = make_float2(acc, xr);
}

// the last slot is the diagonal of a colour-1 row, or padding
template <int W>
__device__ __forceinline__ float mf2_row(int r, const unsigned short *c16, int win, int at, const float *w, int n0,
                                         const float2 *hx, float xi) {
  unsigned o[W];
  float a[W];
  mf_load<W>(c16, r & 63, o);
  mf_load<W>(w, r & 63, a);
  int c[W];
#pragma unroll
  for (int j = 0; j < W; j++) c[j] = j + 1 == W ? r : mf_col(o[j], win, at, r);
  float2 h[W];
#pragma unroll
  for (int j = 0; j < W; j++) h[j] = c[j] < n0 ? hx[c[j]] : make_float2(0.f, 0.f);
  float acc = 0.f;
#pragma unroll
  for (int j = 0; j < W; j++) acc = acc + a[j] * (c[j] < n0 ? (xi - h[j].y) + h[j].x : xi);
  return acc;
}

template <bool PU>
__global__ void k_mf_stage2(int n0, int n1, Mat A, MfCols m, const float *w, float *x, const float2 *hx, float *q,
                            KS *st, float *part, PUp u) {
  if (st->done) return;
  float beta = 0.f;
  bool up = false;
  if constexpr (PU) {
    up = st->pup != 0;
    beta = (float)st->beta;
  }
  const int i1 = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x, i = min(i1, n1 - 1);
  float v[1] = {0.f};
  // the rows of a wavefront lie in one slice or two (n0 is not a multiple of
  // 64): both slices' data come by scalar loads, a row selects its own; the
  // windows of the second are in lanes 16..31
  const int r = n0 + i, s0 = __builtin_amdgcn_readfirstlane(r >> 6);
  const bool first = (r >> 6) == s0;
  const int s1 = __all(first) ? s0 : s0 + 1;
  const long long oa = A.off[s0], ob = A.off[s1];
  const int wa = (int)((A.off[s0 + 1] - oa) >> 6), wb = (int)((A.off[s1 + 1] - ob) >> 6);
  const int win = m.win[16 * ((threadIdx.x & 16) ? s1 : s0) + (threadIdx.x & 15)], at = first ? 0 : 16;
  const bool near16 = m.win[16 * s0 + 15] != 0 && m.win[16 * s1 + 15] != 0;
  const int wd = wa == wb ? wa : 0;
  const float xi = pu_val<PU>(i, x, u, beta, up);
  float acc;
  const long long o0 = first ? oa : ob;
  const unsigned short *c16 = m.c16 + o0;
  const float *ws = w + o0;
  if (wd == 7 && near16) acc = mf2_row<7>(r, c16, win, at, ws, n0, hx, xi);
  else if (wd == 6 && near16) acc = mf2_row<6>(r, c16, win, at, ws, n0, hx, xi);
  else if (wd == 5 && near16) acc = mf2_row<5>(r, c16, win, at, ws, n0, hx, xi);
  else {
    acc = 0.f;
    const int wl = first ? wa : wb;
    for (int j = 0; j < wl; j++) {
      const int c = A.col[o0 + (long long)j * kSlice + (r & 63)];
      const float a = ws[mf_pos(wl, j, r & 63)];
      if (c < n0) {
        const float2 h = hx[c];
        acc = acc + a * ((xi - h.y) + h.x);
      } else {
        acc = acc + a * xi;
      }
    }
  }
  if (i1 < n1) {
    if (up) x[i] = xi;
    q[i] = acc;
    v[0] = xi * acc;
  }
  block_partials<OpSum, 1>(v, part);
}

// x += alpha p; r -= alpha q; partials r.r, (Jacobi) r.(r/d) and sum r
// (Z^T r when the rows are aggregate chunks).
// mode 0 plain, 1 Jacobi, 2 DILU: z = r/d on the first colour block [0,c0end)
template <class T, class X>
__global__ void k_pcg_update(Rows R, const T *p, const T *q, X *x, T *r, T *z, const T *dg, int mode, int c0end,
                             const KS *st, T *part) {
  if (st->done) return;
  int i, a;
  T v[3] = {T(0), T(0), T(0)};
  if (R.get(i, a)) {
    // every load before the first store: the compiler cannot tell the
    // pointers apart, and loads after a store would wait for it
    const T alpha = (T)st->alpha;
    const T pi = p[i], qi = q[i], r0 = r[i];
    const X xi = x[i];
    const T di = (mode == 1 || (mode == 2 && i < c0end)) ? dg[i] : T(1);
    x[i] = xi + (X)(alpha * pi);
    const T ri = r0 - alpha * qi;
    r[i] = ri;
    v[0] = ri * ri;
    v[2] = ri;
    if (mode == 1) v[1] = ri * (ri / di);
    else if (mode == 2 && i < c0end) z[i] = ri / di;
  }
  block_partials<OpSum, 3>(v, part);
}

// p = z (+ nu of the row's aggregate) + beta p
template <class T>
__global__ void k_pcg_p(Rows R, const T *r, const T *z, const T *dg, int jac, T *p, const double *nu,
                        const KS *st) {
  if (st->done) return;
  int i, a;
  if (R.get(i, a)) {
    T zi = jac ? r[i] / dg[i] : z[i];
    if (nu) zi = zi + (T)nu[a];
    p[i] = zi + (T)st->beta * p[i];
  }
}

// ------------------------------------------------------- two-launch PCG
// PCG without a coarse space.  An iteration is the launch-bound end of a
// solve: at 16,000 rows its five kernels (product, alpha, update, beta, p)
// took 15.5 us for 3 us of memory traffic.  Here the scalar recurrences have no
// kernels of their own: every workgroup reduces the partials of the launch
// before it, in the same fixed order, so all hold the same alpha or beta,
// and workgroup 0 keeps the solver state; and the p update rides along the
// product, which forms each neighbour's p = z + beta p_old from the two
// vectors (p is double-buffered, so nobody reads what this launch writes).
//   k_cg_ps: [r.r, r.z -> stop?, beta]  p = z + beta p_old, q = A p; p.q
//   k_cg_xr: [p.q -> alpha]             x += alpha p, r -= alpha q; r.r
//            and with Jacobi z = r/d; r.z
// Preconditioners with sweeps run between the two and leave their own r.z
// partials.  The grid is capped so that the partials every workgroup reads
// stay few; a workgroup takes a contiguous range of row blocks.
// Kernel time per iteration, five launches before, two now: 13.4 -> 7.4 us at
// 1,728 rows in FP64 (a size that k_cg_small takes since), 15.5 -> 7.3 at
// 16,384, 21 -> 13.2 at 216,000; 20.5 -> 16.3 at 432,000 rows in FP32.  Every
// size takes this form: whole PISO steps with FP64 DILU-PCG p' solves, before
// and now, 92 -> 84 ms at 480,000 cells, 199 -> 179 at 1M, 353 -> 338 at 2M
// and 2541 -> 2449 at 8.2M (k_fold_parts from 1M on).
// The parity of the iteration comes from the device's own count: st->it
// changes in k_cg_xr only, st->par in k_cg_ps only.
constexpr int kCgGrid = 2048;
constexpr int kCgPre = 8;   // entries of the first row loaded before the partials arrive

struct RowRange {
  int b0, b1;
};
__device__ __forceinline__ RowRange cg_range(int n) {
  const int nb = (n + kBlock - 1) / kBlock, G = gridDim.x, b = xcd_block(blockIdx.x, G);
  return RowRange{(int)((long long)b * nb / G), (int)((long long)(b + 1) * nb / G)};
}

// sum of up to two partial arrays by a whole workgroup, in a fixed order
template <class T>
__device__ __forceinline__ void cg_sums(int n1, const T *p1, int n2, const T *p2, T (&a)[2]) {
  __shared__ T lds[2 * (kBlock / 64)];
  a[0] = a[1] = T(0);
  int b = threadIdx.x;
  const int nmax = max(n1, n2);
  for (; b < nmax; b += 4 * kBlock) {
    T u[4], v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int i = b + j * kBlock;
      u[j] = i < n1 ? p1[i] : T(0);
      v[j] = i < n2 ? p2[i] : T(0);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      a[0] = a[0] + u[j];
      a[1] = a[1] + v[j];
    }
  }
  block_reduce<OpSum, 2, T, kBlock>(a, lds);
}

// Partials too many for every workgroup of the next launch to add up, to
// kFoldParts (two arrays with grid.y = 2): a launch of 4.6 us against reads
// that every workgroup repeats at some 15 TB/s out of the L2s, so worth it
// above kFoldBytes.  DILU sweeps over 2M rows leave 7,813 for the 2,048
// workgroups of k_cg_ps: 47.8 us after folding, 54.9 without, and an iteration
// takes 114 us of kernels (118 in the seven launches of a finisher each).
constexpr int kFoldParts = 64;
constexpr long long kFoldBytes = 64LL << 20;
template <class T>
__global__ __launch_bounds__(kBlock) void k_fold_parts(int n, const T *a, const T *b, T *out, const KS *st) {
  if (st->done) return;
  const T *src = blockIdx.y ? b : a;
  const int i0 = (int)((long long)blockIdx.x * n / kFoldParts), i1 = (int)((long long)(blockIdx.x + 1) * n / kFoldParts);
  T v[1] = {T(0)};
  for (int i = i0 + threadIdx.x; i < i1; i += kBlock) v[0] = v[0] + src[i];
  block_partials<OpSum, 1>(v, out, blockIdx.y * kFoldParts + blockIdx.x);
}

struct CgParts {   // r.r and r.z partials of the last update / preconditioner
  int nrr, nrz;
};

// The residual test and beta of the next iteration from the partials (all
// threads call it; the result is thread 0's).  Returns 0 go on, 1 converged,
// 2 breakdown.  writer: keep the solver state.
// mixed: the FP32 iteration on r / sigma, as FinUpdateRU.
template <class T, bool MIXED>
__device__ __forceinline__ int cg_test(KS *st, int first, T rr, double rzn, int par, bool writer, double &beta) {
  const double old = st->rz2[par ^ 1];
  beta = 0.0;
  if (!first) {
    if constexpr (MIXED) {
      const double rn = sqrt((double)rr), res = rn * st->sigma / st->bnrm;
      const bool test = !st->trig;
      if (writer) {
        st->res = res;
        if (test && (res <= st->tol || rn < st->delta * st->rmax)) st->ru = 1;
        if (!test) st->ru = 0;
      }
      if (test && res <= st->tol) {
        if (writer) st->done = 2;
        return 1;
      }
      if (writer && rn > st->rmax) st->rmax = rn;
    } else {
      const double res = sqrt((double)rr) / st->bnrm;
      if (writer) {
        st->rr = rr;
        st->res = res;
      }
      if (res <= st->tol) {
        if (writer) st->done = 1;
        return 1;
      }
    }
    if (fabs(old) < kTiny) {
      if (writer) {
        st->ierr = 2;
        st->done = 1;
      }
      return 2;
    }
    beta = rzn / old;
  }
  return 0;
}

template <class T, bool MIXED, int C16>
__global__ __launch_bounds__(kBlock) void k_cg_ps(int n, Mat A, const T *val, const T *z, T *p0, T *p1, T *q, KS *st,
                                                  CgParts np, const T *rrp, const T *rzp, T *pqp) {
  if (st->done) return;
  const int first = st->it == 0, par = st->it & 1;
  const T *po = par ? p0 : p1;
  T *pn = par ? p1 : p0;
  const RowRange R = cg_range(n);
  __shared__ double beta_s;
  __shared__ int stop_s;
  // the first row's matrix entries and vector values are loaded before the
  // partials are waited for
  int i = R.b0 * kBlock + threadIdx.x, w = 0;
  long long base = 0;
  int c[kCgPre];
  T a[kCgPre], zc[kCgPre], pc[kCgPre], zi = T(0), pi = T(0);
  auto load = [&]() {
    const int s = i >> 6;
    const long long o0 = A.off[s];
    w = (int)((A.off[s + 1] - o0) >> 6);
    base = o0 + (i & 63);
    zi = z[i];
    pi = first ? T(0) : po[i];
#pragma unroll
    for (int k = 0; k < kCgPre; k++) c[k] = k < w ? col_at<C16>(A, base + (long long)k * kSlice, i, s) : i;
#pragma unroll
    for (int k = 0; k < kCgPre; k++) a[k] = k < w ? val[base + (long long)k * kSlice] : T(0);
#pragma unroll
    for (int k = 0; k < kCgPre; k++) zc[k] = k < w ? z[c[k]] : T(0);
#pragma unroll
    for (int k = 0; k < kCgPre; k++) pc[k] = (k < w && !first) ? po[c[k]] : T(0);
  };
  if (R.b0 < R.b1 && i < n) load();
  T sums[2];
  cg_sums<T>(np.nrr, rrp, np.nrz, rzp, sums);
  if (threadIdx.x == 0) {
    double beta;
    stop_s = cg_test<T, MIXED>(st, first, sums[0], (double)sums[1], par, blockIdx.x == 0, beta);
    beta_s = beta;
    if (blockIdx.x == 0 && !stop_s) {
      st->beta = beta;
      st->rz2[par] = (double)sums[1];
      st->par = par;
    }
  }
  __syncthreads();
  if (stop_s) return;
  const T beta = (T)beta_s;
  T v[1] = {T(0)};
  for (int b = R.b0; b < R.b1; b++) {
    i = b * kBlock + threadIdx.x;
    if (i < n) {
      if (b > R.b0) load();
      const T xi = zi + beta * pi;
      T acc = T(0);
#pragma unroll
      for (int k = 0; k < kCgPre; k++)
        if (k < w) {
          const T xk = zc[k] + beta * pc[k];
          if constexpr (sizeof(T) == 4) acc = acc + a[k] * (c[k] == i ? xi : xk - xi);
          else acc = acc + a[k] * xk;
        }
      for (int k = kCgPre; k < w; k++) {
        const long long e = base + (long long)k * kSlice;
        const int ck = col_at<C16>(A, e, i, i >> 6);
        const T xk = z[ck] + beta * (first ? T(0) : po[ck]);
        if constexpr (sizeof(T) == 4) acc = acc + val[e] * (ck == i ? xi : xk - xi);
        else acc = acc + val[e] * xk;
      }
      pn[i] = xi;
      q[i] = acc;
      v[0] = v[0] + xi * acc;
    }
  }
  block_partials<OpSum, 1>(v, pqp);
}

// mode 1 Jacobi (z = r/d, r.z), 2 DILU (z = r/d on the first colour block),
// 0 neither
template <class T, class X>
__global__ __launch_bounds__(kBlock) void k_cg_xr(int n, const T *p0, const T *p1, const T *q, X *x, T *r, T *z,
                                                  const T *dg, int mode, int c0end, KS *st, int npq, const T *pqp,
                                                  T *rrp, T *rzp) {
  if (st->done) return;
  const int par = st->par;
  const T *p = par ? p1 : p0;
  const RowRange R = cg_range(n);
  __shared__ double alpha_s;
  __shared__ int bad_s;
  int i = R.b0 * kBlock + threadIdx.x;
  T pi = T(0), qi = T(0), ri = T(0), di = T(1);
  X xi = X(0);
  auto load = [&]() {
    pi = p[i];
    qi = q[i];
    ri = r[i];
    xi = x[i];
    if (mode == 1 || (mode == 2 && i < c0end)) di = dg[i];
  };
  if (R.b0 < R.b1 && i < n) load();
  T sums[2];
  cg_sums<T>(npq, pqp, 0, pqp, sums);
  if (threadIdx.x == 0) {
    const double pap = (double)sums[0];
    const int bad = fabs(pap) < kTiny;
    bad_s = bad;
    alpha_s = bad ? 0.0 : st->rz2[par] / pap;
    if (blockIdx.x == 0) {
      st->it = st->it + 1;
      st->pap = pap;
      st->trig = 0;
      if (bad) {
        st->ierr = 2;
        st->done = 1;
      } else {
        st->alpha = alpha_s;
      }
    }
  }
  __syncthreads();
  if (bad_s) return;
  const T alpha = (T)alpha_s;
  T v[2] = {T(0), T(0)};
  for (int b = R.b0; b < R.b1; b++) {
    i = b * kBlock + threadIdx.x;
    if (i < n) {
      if (b > R.b0) load();
      x[i] = xi + (X)(alpha * pi);
      const T rn = ri - alpha * qi;
      r[i] = rn;
      v[0] = v[0] + rn * rn;
      if (mode == 1 || (mode == 2 && i < c0end)) {
        const T zn = rn / di;
        z[i] = zn;
        if (mode == 1) v[1] = v[1] + rn * zn;
      }
    }
  }
  __shared__ T lds[2 * (kBlock / 64)];
  block_reduce<OpSum, 2, T>(v, lds);
  if (threadIdx.x == 0) {
    rrp[blockIdx.x] = v[0];
    if (mode == 1) rzp[blockIdx.x] = v[1];
  }
}

// the tests after the last update of a chunk, for the host to read (the next
// k_cg_ps comes to the same answer; BiCGSTAB tests its rho at the next
// iteration's start)
template <class T, bool MIXED, bool PCG = true>
__global__ __launch_bounds__(kBlock) void k_cg_peek(KS *st, int nrr, const T *rrp) {
  if (st->done || st->it == 0) return;
  T sums[2];
  cg_sums<T>(nrr, rrp, 0, rrp, sums);
  if (threadIdx.x != 0) return;
  const double rn = sqrt((double)sums[0]);
  if constexpr (MIXED) {
    st->res = rn * st->sigma / st->bnrm;
    if (!st->trig && (st->res <= st->tol || rn < st->delta * st->rmax)) st->ru = 1;
    if (!st->trig && st->res <= st->tol) st->done = 2;
  } else {
    st->rr = (double)sums[0];
    st->res = rn / st->bnrm;
    if (st->res <= st->tol) st->done = 1;
  }
  if (PCG && !st->done && fabs(st->rz2[st->par]) < kTiny) {
    st->ierr = 2;
    st->done = 1;
  }
}

// after a reliable update: r32 = r64 / sigma, the p the next k_cg_ps reads as
// the old one moved to the new scale, r.r and z, r.z as k_cg_xr
__global__ __launch_bounds__(kBlock) void k_cg_rescale(int n, const double *r64, float *r32, float *p0, float *p1,
                                                       float *z, const float *dg, int mode, int c0end, const KS *st,
                                                       float *rrp, float *rzp) {
  if (st->done || st->ru != 2) return;
  const RowRange R = cg_range(n);
  float *p = (st->it & 1) ? p0 : p1;
  float v[2] = {0.0f, 0.0f};
  for (int b = R.b0; b < R.b1; b++) {
    const int i = b * kBlock + threadIdx.x;
    if (i < n) {
      const float ri = (float)(r64[i] / st->sigma);
      r32[i] = ri;
      p[i] = p[i] * (float)st->scale;
      v[0] = v[0] + ri * ri;
      if (mode == 1 || (mode == 2 && i < c0end)) {
        const float zi = ri / dg[i];
        z[i] = zi;
        if (mode == 1) v[1] = v[1] + ri * zi;
      }
    }
  }
  __shared__ float lds[2 * (kBlock / 64)];
  block_reduce<OpSum, 2, float>(v, lds);
  if (threadIdx.x == 0) {
    rrp[blockIdx.x] = v[0];
    if (mode == 1) rzp[blockIdx.x] = v[1];
  }
}

// -------------------------------------------------- PCG with a coarse space
// The same idea where the coarse solve needs Z^T r of the whole update before
// p can be formed, so p keeps a launch of its own:
//   product with p.q partials
//   k_cx_update: [p.q -> alpha]  x, r; r.r, (Jacobi) r.z, chunk sums of r,
//                (DILU) z on the first colour
//   Jacobi: k_cx_coarse, nu = E^-1 Z^T r;  DILU: the sweeps, the first of
//                which carries the coarse solve
//   k_cx_p:      [r.r, r.z + c.nu -> stop?, beta]  p = z + nu + beta p
// A wavefront takes a chunk (at most 256 rows of one aggregate, four per
// lane): its loads are all in flight at once and issued before the partials
// are waited for, its chunk sum needs shuffles only, and four chunks share
// the reduction of the partials, which every workgroup repeats.  With one
// workgroup per chunk (3,907 at 1M rows) those repeats read 61 MB through the
// L2s, twice the data of the update itself.
// Per iteration of the reduced p' solve at 2M cells, in us: update 11.9 ->
// 8.3, coarse solve 8.0 -> 6.0; the p update stays at 6.0.
constexpr int kCxGrid = 1024;
constexpr int kCxRows = kBlock / kSlice;   // rows per lane

struct Chunks {
  const int *ptr, *agg, *pos;
  int n;
};
__device__ __forceinline__ RowRange cx_range(const Chunks &C) {
  const int G = gridDim.x, b = xcd_block(blockIdx.x, G);
  return RowRange{(int)((long long)b * C.n / G), (int)((long long)(b + 1) * C.n / G)};
}

// sum over the wavefront, on every lane, in a fixed order
template <class T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = v + __shfl_xor(v, o, 64);
  return v;
}

template <class T, class X>
__global__ __launch_bounds__(kBlock) void k_cx_update(Chunks C, int npq, const T *pqp, const T *p, const T *q, X *x,
                                                      T *r, T *z, const T *dg, int mode, int c0end, KS *st, T *rrp,
                                                      T *rzp, T *csum) {
  const int done = st->done;
  const RowRange R = cx_range(C);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int ch = R.b0 + wv, r0 = 0, r1 = 0, pos = 0;
  T pi[kCxRows], qi[kCxRows], ri[kCxRows], di[kCxRows];
  X xi[kCxRows];
  auto load = [&]() {
    r0 = C.ptr[ch] + lane;
    r1 = C.ptr[ch + 1];
    pos = C.pos[ch];
#pragma unroll
    for (int u = 0; u < kCxRows; u++) {
      const int i = min(r0 + u * kSlice, r1 - 1);   // lanes beyond the chunk repeat its last row
      pi[u] = p[i];
      qi[u] = q[i];
      ri[u] = r[i];
      xi[u] = x[i];
      di[u] = dg[i];
    }
  };
  if (ch < R.b1) load();
  if (done) return;
  __shared__ double alpha_s;
  __shared__ int bad_s;
  T sums[2];
  cg_sums<T>(npq, pqp, 0, pqp, sums);
  if (threadIdx.x == 0) {
    const double pap = (double)sums[0];
    const int bad = fabs(pap) < kTiny;
    bad_s = bad;
    alpha_s = bad ? 0.0 : st->rz2[st->par] / pap;
    if (blockIdx.x == 0) {
      st->it = st->it + 1;
      st->pap = pap;
      st->trig = 0;
      st->pup = 0;   // the product before this launch applied a pending p update
      if (bad) {
        st->ierr = 2;
        st->done = 1;
      } else {
        st->alpha = alpha_s;
      }
    }
  }
  __syncthreads();
  if (bad_s) return;
  const T alpha = (T)alpha_s;
  T v[2] = {T(0), T(0)};
  for (; ch < R.b1; ch += kBlock / kSlice) {
    if (ch >= R.b0 + kBlock / kSlice) load();
    T cs = T(0);
#pragma unroll
    for (int u = 0; u < kCxRows; u++) {
      const int i = r0 + u * kSlice;
      if (i < r1) {
        x[i] = xi[u] + (X)(alpha * pi[u]);
        const T rn = ri[u] - alpha * qi[u];
        r[i] = rn;
        v[0] = v[0] + rn * rn;
        cs = cs + rn;
        if (mode == 1) v[1] = v[1] + rn * (rn / di[u]);
        else if (i < c0end) z[i] = rn / di[u];
      }
    }
    cs = wave_sum(cs);
    if (lane == 0) csum[pos] = cs;
  }
  __shared__ T lds[2 * (kBlock / 64)];
  block_reduce<OpSum, 2, T>(v, lds);
  if (threadIdx.x == 0) {
    rrp[blockIdx.x] = v[0];
    if (mode == 1) rzp[blockIdx.x] = v[1];
  }
}

// The sums of an r that no update made: the initial residual (r64 null), or
// after a reliable update r = r64 / sigma with p moved to the new scale.
template <class T>
__global__ __launch_bounds__(kBlock) void k_cx_start(Chunks C, const double *r64, T *r, T *p, T *z, const T *dg,
                                                     int mode, int c0end, const KS *st, T *rrp, T *rzp, T *csum) {
  if (st->done || (r64 && st->ru != 2)) return;
  const RowRange R = cx_range(C);
  const int lane = threadIdx.x & 63;
  T v[2] = {T(0), T(0)};
  for (int ch = R.b0 + (threadIdx.x >> 6); ch < R.b1; ch += kBlock / kSlice) {
    const int r1 = C.ptr[ch + 1];
    T cs = T(0);
    for (int i = C.ptr[ch] + lane; i < r1; i += kSlice) {
      T ri;
      if (r64) {
        ri = (T)(r64[i] / st->sigma);
        r[i] = ri;
        p[i] = p[i] * (T)st->scale;
      } else {
        ri = r[i];
      }
      v[0] = v[0] + ri * ri;
      cs = cs + ri;
      if (mode == 1) v[1] = v[1] + ri * (ri / dg[i]);
      else if (i < c0end) z[i] = ri / dg[i];
    }
    cs = wave_sum(cs);
    if (lane == 0) csum[C.pos[ch]] = cs;
  }
  __shared__ T lds[2 * (kBlock / 64)];
  block_reduce<OpSum, 2, T>(v, lds);
  if (threadIdx.x == 0) {
    rrp[blockIdx.x] = v[0];
    if (mode == 1) rzp[blockIdx.x] = v[1];
  }
}

// nu = E^-1 c, c = Z^T r from the chunk sums: workgroup g recomputes c and
// forms rows [kSplitRows g, kSplitRows (g + 1)) of nu, a wavefront per row,
// and the c.nu sum of its rows.  It is a chain of far loads in few
// workgroups: E^-1, which no load waits for, is fetched first, and an
// aggregate's chunk sums lie side by side.
constexpr int kCoPre = 4;   // 64-column pieces of an E^-1 row fetched ahead (k <= 256)
template <class T>
__global__ __launch_bounds__(kFinThreads) void k_cx_coarse(int k, const int *cptr, const float *Einv, const T *csum,
                                                           double *nu, double *cnu_part, const KS *st) {
  const int done = st->done;
  __shared__ double c[kMaxAgg], partq[kFinThreads], pr[kSplitRows];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, a = blockIdx.x * kSplitRows + w;
  float e[kCoPre];
#pragma unroll
  for (int j = 0; j < kCoPre; j++) {
    const int b = lane + 64 * j;
    e[j] = a < k && b < k ? Einv[(size_t)a * k + b] : 0.0f;
  }
  // Q threads per aggregate, each every Q-th of its chunks
  const int Q = k <= kFinThreads / 4 ? 4 : (k <= kFinThreads / 2 ? 2 : 1), span = kFinThreads / Q;
  const int g = threadIdx.x % span, qq = threadIdx.x / span;
  if (g < k) {
    double s = 0.0;
    int j = cptr[g] + qq;
    const int je = cptr[g + 1];
    for (; j + 3 * Q < je; j += 4 * Q) {
      const T v0 = csum[j], v1 = csum[j + Q], v2 = csum[j + 2 * Q], v3 = csum[j + 3 * Q];
      s = s + (double)v0;
      s = s + (double)v1;
      s = s + (double)v2;
      s = s + (double)v3;
    }
    for (; j < je; j += Q) s = s + (double)csum[j];
    partq[qq * span + g] = s;
  }
  if (done) return;
  __syncthreads();
  if (qq == 0 && g < k) {
    double s = partq[g];
    for (int i = 1; i < Q; i++) s = s + partq[i * span + g];
    c[g] = s;
  }
  __syncthreads();
  double prod = 0.0;
  if (a < k) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < kCoPre; j++) {
      const int b = lane + 64 * j;
      if (b < k) s = s + (double)e[j] * c[b];
    }
    for (int b = lane + 64 * kCoPre; b < k; b += 64) s = s + (double)Einv[(size_t)a * k + b] * c[b];
    s = wave_sum(s);
    if (lane == 0) {
      nu[a] = s;
      prod = s * c[a];
    }
  }
  if (lane == 0) pr[w] = prod;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int j = 0; j < kSplitRows; j++) t = t + pr[j];
    cnu_part[blockIdx.x] = t;
  }
}

// p = z + nu + beta p (z = r/d with Jacobi); ncn coarse parts of r.z.
// what: kCxAll; kCxTest (one workgroup, C.n = 0): the test and beta only, and
// the update is left pending for the product; kCxPending: a pending update
// only.
enum { kCxAll = 0, kCxTest = 1, kCxPending = 2 };
template <class T, bool MIXED>
__global__ __launch_bounds__(kBlock) void k_cx_p(Chunks C, const T *r, const T *z, const T *dg, int mode, T *p,
                                                 const double *nu, KS *st, CgParts np, const T *rrp, const T *rzp,
                                                 int ncn, const double *cnu_part, int what) {
  const int done = st->done;
  if (what == kCxPending && !st->pup) return;
  const RowRange R = cx_range(C);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int ch = R.b0 + wv, r0 = 0, r1 = 0;
  T zi[kCxRows], di[kCxRows], pi[kCxRows], nua = T(0);
  auto load = [&]() {
    r0 = C.ptr[ch] + lane;
    r1 = C.ptr[ch + 1];
    nua = (T)nu[C.agg[ch]];
#pragma unroll
    for (int u = 0; u < kCxRows; u++) {
      const int i = min(r0 + u * kSlice, r1 - 1);
      zi[u] = mode == 1 ? r[i] : z[i];
      di[u] = mode == 1 ? dg[i] : T(1);
      pi[u] = p[i];
    }
  };
  if (ch < R.b1) load();
  double cn = wv == 0 && lane < ncn ? cnu_part[lane] : 0.0;
  if (done) return;
  const int first = st->it == 0, par = st->it & 1;
  T sums[2];
  cg_sums<T>(np.nrr, rrp, np.nrz, rzp, sums);
  cn = wave_sum(cn);
  __shared__ double beta_s;
  __shared__ int stop_s;
  if (threadIdx.x == 0) {
    const double rzn = (double)sums[1] + cn;
    double beta = st->beta;
    stop_s = what == kCxPending ? 0 : cg_test<T, MIXED>(st, first, sums[0], rzn, par, blockIdx.x == 0, beta);
    beta_s = beta;
    if (what != kCxPending && blockIdx.x == 0 && !stop_s) {
      st->beta = beta;
      st->rz2[par] = rzn;
      st->par = par;
      st->pup = what == kCxTest;
    }
  }
  __syncthreads();
  if (stop_s) return;
  const T beta = (T)beta_s;
  for (; ch < R.b1; ch += kBlock / kSlice) {
    if (ch >= R.b0 + kBlock / kSlice) load();
#pragma unroll
    for (int u = 0; u < kCxRows; u++) {
      const int i = r0 + u * kSlice;
      if (i < r1) {
        const T zn = (mode == 1 ? zi[u] / di[u] : zi[u]) + nua;
        p[i] = first ? zn : zn + beta * pi[u];
      }
    }
  }
}

// -------------------------------------------------------- PCG of one workgroup
// A system whose matrix fits one workgroup's registers: FP64, Jacobi, at most
// kSmallRows rows and kSmallWidth entries per row.  The direction is in LDS,
// everything else in registers, two rows per thread at most, and an iteration
// is three barriers instead of two launches, whose latency is all that the
// two-launch form spends on such a system: 7.4 us an iteration at 1,728 rows,
// here 2.5.  A launch runs at most kSmallIters iterations, so that it ends
// whatever maxit is; p and r.z are kept for the next.
constexpr int kSmallRows = 2048, kSmallWidth = 8, kSmallThreads = 1024, kSmallIters = 4096;

template <int NV>
__device__ __forceinline__ void small_sums(double (&v)[NV], double *lds) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int j = 0; j < NV; j++) v[j] = wave_sum(v[j]);
  if (lane == 0)
#pragma unroll
    for (int j = 0; j < NV; j++) lds[w * NV + j] = v[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NV; j++) {
    double s = lds[j];
    for (int q = 1; q < nw; q++) s = s + lds[q * NV + j];
    v[j] = s;
  }
}

template <int R>   // rows per thread
__global__ __launch_bounds__(kSmallThreads) void k_cg_small(int n, Mat A, const double *val, const double *dg,
                                                            double *x, double *r, double *p, KS *st, int iters) {
  if (st->done) return;
  __shared__ double ps[kSmallRows], l1[kSmallThreads / 64], l2[2 * (kSmallThreads / 64)];
  const int t = threadIdx.x, nt = blockDim.x;
  const double bnrm = st->bnrm, tol = st->tol;
  int it = st->it, c[R][kSmallWidth];
  const bool first = it == 0;
  double rz = st->rz2[0];
  double a[R][kSmallWidth], xi[R], ri[R], di[R], pi[R];
#pragma unroll
  for (int u = 0; u < R; u++) {
    const int i = t + u * nt;
    const bool in = i < n;
    const long long o0 = in ? A.off[i >> 6] : 0;
    const int w = in ? (int)((A.off[(i >> 6) + 1] - o0) >> 6) : 0;
#pragma unroll
    for (int k = 0; k < kSmallWidth; k++) {
      const long long q = o0 + (i & 63) + (long long)k * kSlice;
      c[u][k] = k < w ? A.col[q] : (in ? i : 0);
      a[u][k] = k < w ? val[q] : 0.0;
    }
    xi[u] = in ? x[i] : 0.0;
    ri[u] = in ? r[i] : 0.0;
    di[u] = in ? dg[i] : 1.0;
    pi[u] = in && !first ? p[i] : 0.0;
  }
  if (first) {
    double v[1] = {0.0};
#pragma unroll
    for (int u = 0; u < R; u++) {
      pi[u] = ri[u] / di[u];
      v[0] = v[0] + ri[u] * pi[u];
    }
    small_sums<1>(v, l1);
    rz = v[0];
  }
  int ierr = 0, done = 0;
  double res = st->res;
  for (int e = 0; e < iters; e++) {
#pragma unroll
    for (int u = 0; u < R; u++)
      if (t + u * nt < n) ps[t + u * nt] = pi[u];
    __syncthreads();
    double qi[R], v1[1] = {0.0};
#pragma unroll
    for (int u = 0; u < R; u++) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < kSmallWidth; k++) s = s + a[u][k] * ps[c[u][k]];
      qi[u] = s;
      v1[0] = v1[0] + pi[u] * s;
    }
    small_sums<1>(v1, l1);   // its barrier also ends the reads of ps
    it++;
    if (fabs(v1[0]) < kTiny) {
      ierr = 2;
      done = 1;
      break;
    }
    const double alpha = rz / v1[0];
    double v2[2] = {0.0, 0.0}, zi[R];
#pragma unroll
    for (int u = 0; u < R; u++) {
      xi[u] = xi[u] + alpha * pi[u];
      ri[u] = ri[u] - alpha * qi[u];
      zi[u] = ri[u] / di[u];
      v2[0] = v2[0] + ri[u] * ri[u];
      v2[1] = v2[1] + ri[u] * zi[u];
    }
    small_sums<2>(v2, l2);
    res = sqrt(v2[0]) / bnrm;
    if (res <= tol) {
      done = 1;
      break;
    }
    if (fabs(rz) < kTiny) {
      ierr = 2;
      done = 1;
      break;
    }
    const double beta = v2[1] / rz;
    rz = v2[1];
#pragma unroll
    for (int u = 0; u < R; u++) pi[u] = zi[u] + beta * pi[u];
  }
#pragma unroll
  for (int u = 0; u < R; u++) {
    const int i = t + u * nt;
    if (i < n) {
      x[i] = xi[u];
      r[i] = ri[u];
      p[i] = pi[u];
    }
  }
  __syncthreads();   // every thread has read the state
  if (t == 0) {
    st->it = it;
    st->rz2[0] = rz;
    st->res = res;
    st->ierr = ierr;
    st->done = done;
  }
}

__global__ void k_clear_pup(KS *st) {
  if (threadIdx.x == 0) st->pup = 0;
}

template <class T>
__global__ void k_dot(int n, const T *a, const T *b, const KS *st, T *part) {
  if (st->done) return;
  int i = blockIdx.x * kBlock + threadIdx.x;
  T v[1] = {i < n ? a[i] * b[i] : T(0)};
  block_partials<OpSum, 1>(v, part);
}

// z of the initial residual: r/d and r.z (mode 1), r/d on the first colour
// block (mode 2)
template <class T>
__global__ __launch_bounds__(kBlock) void k_cg_z(int n, const T *r, const T *dg, T *z, int mode, int c0end,
                                                 const KS *st, T *rzp) {
  if (st->done) return;
  const RowRange R = cg_range(n);
  T v[1] = {T(0)};
  for (int b = R.b0; b < R.b1; b++) {
    const int i = b * kBlock + threadIdx.x;
    if (i < (mode == 2 ? c0end : n)) {
      const T ri = r[i], zi = ri / dg[i];
      z[i] = zi;
      v[0] = v[0] + ri * zi;
    }
  }
  if (mode == 1) block_partials<OpSum, 1>(v, rzp);
}

// ------------------------------------------------------- reliable updates
// x64 += sigma * y; y = 0   (only when a reliable update is pending)
__global__ void k_fold(int n, float *y, double *x, const KS *st) {
  if (st->done == 1 || st->ru != 1) return;
  int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) {
    x[i] = x[i] + st->sigma * (double)y[i];
    y[i] = 0.0f;
  }
}
// r64 = b - A64 x and r64.r64 (FP64)
__global__ void k_true_res(int n, Mat A, const double *val, const double *b, const double *x, double *r64,
                           const KS *st, double *part) {
  if (st->done == 1 || st->ru != 1) return;
  int i = blockIdx.x * kBlock + threadIdx.x;
  double v[1] = {0.0};
  if (i < n) {
    double ri = b[i] - row_dot(i, A, val, x);
    r64[i] = ri;
    v[0] = ri * ri;
  }
  block_partials<OpSum, 1>(v, part);
}
// r32 = r64 / sigma; p *= scale (after FinRU moved to the new scale), with
// the partials and colour-0 DILU values of k_pcg_update for the new r
__global__ void k_ru_rescale(Rows R, const double *r64, float *r32, float *p, float *z, const float *dg, int mode,
                             int c0end, const KS *st, float *part) {
  if (st->done || st->ru != 2) return;
  int i, a;
  float v[3] = {0.0f, 0.0f, 0.0f};
  if (R.get(i, a)) {
    const float ri = (float)(r64[i] / st->sigma);
    r32[i] = ri;
    p[i] = p[i] * (float)st->scale;
    v[0] = ri * ri;
    v[2] = ri;
    if (mode == 1) v[1] = ri * (ri / dg[i]);
    else if (mode == 2 && i < c0end) z[i] = ri / dg[i];
  }
  block_partials<OpSum, 3>(v, part);
}
// initial scaled residual r32 = r64 / sigma
__global__ void k_scale_down(int n, const double *r64, float *r32, const KS *st) {
  int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) r32[i] = (float)(r64[i] / st->sigma);
}
__global__ void k_set_sigma(KS *st) {
  if (threadIdx.x == 0) {
    st->sigma = sqrt(st->rr);
    st->rmax = 1.0;
  }
}

// -------------------------------------------------------------- BiCGSTAB
// Additive coarse correction of a BiCGSTAB preconditioner application,
// out += Z E^-1 Z^T in (the p' matrix and so E are symmetric): chunk sums of
// in come from the launch that formed it (FP64), nu = E^-1 c from k_cx_coarse,
// then nu of each row's aggregate is added to out.
template <class T>
__global__ void k_co_prolong(Rows RW, const double *nu, T *out, const int *done) {
  if (*done) return;
  int i, a;
  if (RW.get(i, a)) out[i] = out[i] + (T)nu[a];
}

// An iteration, with the scalar recurrences in the prologues of the launches
// that need them, as the PCG above (it took fourteen launches beside the
// preconditioner's, most of them a few microseconds of latency each):
//   k_bi_p:  [r.r -> stop?, rho = r.r0 -> beta]  p = r + beta (p - omega v)
//            and the preconditioner's first stage; chunk sums of p
//   (preconditioner)   ph = M^-1 p
//   k_bi_spmv_dot:     v = A ph; v.r0
//   k_bi_s:  [v.r0 -> alpha]  s = r - alpha v, first stage; s.s
//   k_finish (FinBiS): |s| small enough?  (x + alpha ph then ends the solve)
//   (preconditioner)   sh = M^-1 s
//   k_bi_spmv_omega:   t = A sh; t.t, t.s
//   k_bi_xr: [t.t, t.s -> omega]  x += alpha ph + omega sh, r = s - omega t;
//            r.r, r.r0
// First stage: Jacobi's ph = p/d (mode 1), DILU's p/d on the first colour
// (mode 2).  Rows go by chunks of at most 256, a wavefront each: aggregate
// chunks with a coarse space, else plain blocks (C.ptr null).
__device__ __forceinline__ void chunk_rows(const Chunks &C, int n, int ch, int &r0, int &r1) {
  if (C.ptr) {
    r0 = C.ptr[ch];
    r1 = C.ptr[ch + 1];
  } else {
    r0 = ch * kBlock;
    r1 = min(n, r0 + kBlock);
  }
}

// r0 = r and the r.r, r.r0 partials of the initial residual
template <class T>
__global__ __launch_bounds__(kBlock) void k_bi_init(int n, const T *r, T *r0, T *rrp, T *rhop) {
  T v[1] = {T(0)};
  const RowRange R = cg_range(n);
  for (int b = R.b0; b < R.b1; b++) {
    const int i = b * kBlock + threadIdx.x;
    if (i < n) {
      const T ri = r[i];
      r0[i] = ri;
      v[0] = v[0] + ri * ri;
    }
  }
  __shared__ T lds[kBlock / 64];
  block_reduce<OpSum, 1, T>(v, lds);
  if (threadIdx.x == 0) {
    rrp[blockIdx.x] = v[0];
    rhop[blockIdx.x] = v[0];
  }
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_bi_p(Chunks C, int n, const T *r, const T *v, T *p, T *ph, const T *dg,
                                                 int mode, int c0end, KS *st, int np, const T *rrp, const T *rhop,
                                                 double *csum) {
  const int done = st->done;
  const RowRange R = cx_range(C);
  const int lane = threadIdx.x & 63;
  int ch = R.b0 + (int)(threadIdx.x >> 6), r0 = 0, r1 = 0;
  T ri[kCxRows], pi[kCxRows], vi[kCxRows];
  auto load = [&]() {
    chunk_rows(C, n, ch, r0, r1);
    r0 += lane;
#pragma unroll
    for (int u = 0; u < kCxRows; u++) {
      const int i = min(r0 + u * kSlice, r1 - 1);
      ri[u] = r[i];
      pi[u] = p[i];
      vi[u] = v[i];
    }
  };
  if (ch < R.b1) load();
  if (done) return;
  const int first = st->it == 0, par = st->it & 1;
  T sums[2];
  cg_sums<T>(np, rrp, np, rhop, sums);
  __shared__ double beta_s;
  __shared__ int stop_s;
  if (threadIdx.x == 0) {
    const bool w = blockIdx.x == 0;
    const double res = sqrt((double)sums[0]) / st->bnrm, rho = (double)sums[1];
    double beta = 0.0;
    int stop = 0;
    if (!first && res <= st->tol) {
      stop = 1;
      if (w) {
        st->rr = (double)sums[0];
        st->res = res;
        st->done = 1;
      }
    } else if (fabs(rho) < kTiny) {
      stop = 1;
      if (w) {
        st->it = st->it + 1;
        st->rho = rho;
        st->ierr = 2;
        st->done = 1;
      }
    } else {
      beta = first ? rho : (rho / st->rz2[par ^ 1]) * (st->alpha / st->omega);
      if (w) {
        if (!first) {
          st->rr = (double)sums[0];
          st->res = res;
        }
        st->rho = rho;
        st->beta = beta;
        st->rz2[par] = rho;
        st->par = par;
      }
    }
    beta_s = beta;
    stop_s = stop;
  }
  __syncthreads();
  if (stop_s) return;
  const T beta = (T)beta_s, omega = first ? T(1) : (T)st->omega;
  for (; ch < R.b1; ch += kBlock / kSlice) {
    if (ch >= R.b0 + kBlock / kSlice) load();
    double cs = 0.0;
#pragma unroll
    for (int u = 0; u < kCxRows; u++) {
      const int i = r0 + u * kSlice;
      if (i < r1) {
        const T pn = first ? ri[u] : ri[u] + beta * (pi[u] - omega * vi[u]);
        p[i] = pn;
        cs = cs + (double)pn;
        if (mode == 1 || (mode == 2 && i < c0end)) ph[i] = pn / dg[i];
      }
    }
    if (csum) {
      cs = wave_sum(cs);
      if (lane == 0) csum[C.pos[ch]] = cs;
    }
  }
}

template <class T, int C16 = -1>
__global__ void k_bi_spmv_dot(int n, Mat A, const T *val, const T *ph, const T *r0, T *v, const KS *st, T *part) {
  if (st->done) return;
  int i = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  T w[1] = {T(0)};
  if (i < n) {
    const T r0i = r0[i];
    const T vi = row_apply<T, C16>(i, A, val, ph);
    v[i] = vi;
    w[0] = r0i * vi;
  }
  block_partials<OpSum, 1>(w, part);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_bi_s(Chunks C, int n, const T *r, const T *v, T *s, T *sh, const T *dg,
                                                 int mode, int c0end, KS *st, int nvp, const T *vp, T *ssp,
                                                 double *csum) {
  const int done = st->done;
  const RowRange R = cx_range(C);
  const int lane = threadIdx.x & 63;
  int ch = R.b0 + (int)(threadIdx.x >> 6), r0 = 0, r1 = 0;
  T ri[kCxRows], vi[kCxRows];
  auto load = [&]() {
    chunk_rows(C, n, ch, r0, r1);
    r0 += lane;
#pragma unroll
    for (int u = 0; u < kCxRows; u++) {
      const int i = min(r0 + u * kSlice, r1 - 1);
      ri[u] = r[i];
      vi[u] = v[i];
    }
  };
  if (ch < R.b1) load();
  if (done) return;
  T sums[2];
  cg_sums<T>(nvp, vp, 0, vp, sums);
  __shared__ double alpha_s;
  if (threadIdx.x == 0) {
    alpha_s = st->rz2[st->par] / (double)sums[0];
    if (blockIdx.x == 0) st->alpha = alpha_s;
  }
  __syncthreads();
  const T alpha = (T)alpha_s;
  T w[1] = {T(0)};
  for (; ch < R.b1; ch += kBlock / kSlice) {
    if (ch >= R.b0 + kBlock / kSlice) load();
    double cs = 0.0;
#pragma unroll
    for (int u = 0; u < kCxRows; u++) {
      const int i = r0 + u * kSlice;
      if (i < r1) {
        const T si = ri[u] - alpha * vi[u];
        s[i] = si;
        w[0] = w[0] + si * si;
        cs = cs + (double)si;
        if (mode == 1 || (mode == 2 && i < c0end)) sh[i] = si / dg[i];
      }
    }
    if (csum) {
      cs = wave_sum(cs);
      if (lane == 0) csum[C.pos[ch]] = cs;
    }
  }
  block_partials<OpSum, 1>(w, ssp);
}

// x + alpha ph of a solve that ended on |s| (done = 2)
template <class T>
__global__ void k_bi_early(int n, const T *ph, T *x, const KS *st) {
  if (st->done != 2) return;
  int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] = x[i] + (T)st->alpha * ph[i];
}

template <class T, int C16 = -1>
__global__ void k_bi_spmv_omega(int n, Mat A, const T *val, const T *sh, const T *s, T *t, const KS *st, T *ttp,
                                T *tsp) {
  if (st->done) return;
  int i = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  T w[2] = {T(0), T(0)};
  if (i < n) {
    const T si = s[i];
    const T ti = row_apply<T, C16>(i, A, val, sh);
    t[i] = ti;
    w[0] = ti * ti;
    w[1] = ti * si;
  }
  __shared__ T lds[2 * (kBlock / 64)];
  block_reduce<OpSum, 2, T>(w, lds);
  if (threadIdx.x == 0) {
    ttp[blockIdx.x] = w[0];
    tsp[blockIdx.x] = w[1];
  }
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_bi_xr(Chunks C, int n, const T *ph, const T *sh, const T *s, const T *t,
                                                  const T *r0v, T *x, T *r, KS *st, int np, const T *ttp,
                                                  const T *tsp, T *rrp, T *rhop) {
  const int done = st->done;
  const RowRange R = cx_range(C);
  const int lane = threadIdx.x & 63;
  int ch = R.b0 + (int)(threadIdx.x >> 6), r0 = 0, r1 = 0;
  T pi[kCxRows], hi[kCxRows], si[kCxRows], ti[kCxRows], xi[kCxRows], oi[kCxRows];
  auto load = [&]() {
    chunk_rows(C, n, ch, r0, r1);
    r0 += lane;
#pragma unroll
    for (int u = 0; u < kCxRows; u++) {
      const int i = min(r0 + u * kSlice, r1 - 1);
      pi[u] = ph[i];
      hi[u] = sh[i];
      si[u] = s[i];
      ti[u] = t[i];
      xi[u] = x[i];
      oi[u] = r0v[i];
    }
  };
  if (ch < R.b1) load();
  if (done) return;
  T sums[2];
  cg_sums<T>(np, ttp, np, tsp, sums);
  __shared__ double omega_s;
  __shared__ int stop_s;
  if (threadIdx.x == 0) {
    const double tt = (double)sums[0], omega = (double)sums[1] / tt;
    stop_s = tt < kTiny || fabs(omega) < kTiny;
    omega_s = omega;
    if (blockIdx.x == 0) {
      st->tt = tt;
      if (!(tt < kTiny)) st->omega = omega;
      if (stop_s) {
        st->ierr = 2;
        st->done = 1;
      }
    }
  }
  __syncthreads();
  if (stop_s) return;
  const T alpha = (T)st->alpha, omega = (T)omega_s;
  T w[2] = {T(0), T(0)};
  for (; ch < R.b1; ch += kBlock / kSlice) {
    if (ch >= R.b0 + kBlock / kSlice) load();
#pragma unroll
    for (int u = 0; u < kCxRows; u++) {
      const int i = r0 + u * kSlice;
      if (i < r1) {
        x[i] = xi[u] + alpha * pi[u] + omega * hi[u];
        const T rn = si[u] - omega * ti[u];
        r[i] = rn;
        w[0] = w[0] + rn * rn;
        w[1] = w[1] + rn * oi[u];
      }
    }
  }
  __shared__ T lds[2 * (kBlock / 64)];
  block_reduce<OpSum, 2, T>(w, lds);
  if (threadIdx.x == 0) {
    rrp[blockIdx.x] = w[0];
    rhop[blockIdx.x] = w[1];
  }
}

// ------------------------------------------------ preconditioner kernels
template <class T>
__global__ void k_jacobi(int n, const T *in, const T *dg, T *out, const int *done) {
  if (*done) return;
  int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) out[i] = in[i] / dg[i];
}

template <class T>
__global__ void k_dilu_first(int r0, int r1, const T *dg, const T *r, T *z, const int *done) {
  if (*done) return;
  int i = r0 + blockIdx.x * kBlock + threadIdx.x;
  if (i < r1) z[i] = r[i] / dg[i];
}

// forward sweep of one colour [r0, r1) over nbr row blocks; the first
// cw.nwg blocks carry the coarse solve when a coarse space rides along (they
// start first and overlap the sweep)
template <class T, int C16 = -1>
__global__ void k_dilu_fwd(int r0, int r1, int nbr, Mat A, const T *val, const T *dg, const T *r, T *z, int last,
                           const int *done, T *part, CoWork<T> cw) {
  if (*done) return;
  if ((int)blockIdx.x < cw.nwg) {
    coarse_ride<T>(cw, blockIdx.x);
    return;
  }
  const int rb = blockIdx.x - cw.nwg;
  int i = r0 + xcd_block(rb, nbr) * kBlock + threadIdx.x;
  T v[1] = {T(0)};
  if (i < r1) {
    const long long bi = A.off[i >> 6] + (i & 63);
    const int dpi = A.diagk[i];
    const T ri = r[i];   // kept: a load after the store to z would wait for it
    T s = ri;
    for (int k = 0; k < dpi; k++) {
      const long long q = bi + (long long)k * kSlice;
      const int c = sizeof(T) == 4 ? col_at<C16>(A, q, i, i >> 6) : A.col[q];
      s = s - val[q] * z[c];
    }
    const T zi = s / dg[i];
    z[i] = zi;
    if (last) v[0] = ri * zi;
  }
  if (part) block_partials<OpSum, 1>(v, part, rb);
}

template <class T, int C16 = -1>
__global__ void k_dilu_bwd(int r0, int r1, Mat A, const T *val, const T *dg, const T *r, T *z, const int *done,
                           T *part) {
  if (*done) return;
  int i = r0 + xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  T v[1] = {T(0)};
  if (i < r1) {
    const long long bi = A.off[i >> 6] + (i & 63);
    const int dpi = A.diagk[i], len = A.rowlen[i];
    const T ri = r[i];   // loaded before the store to z
    T s = T(0);
    for (int k = dpi + 1; k < len; k++) {
      const long long q = bi + (long long)k * kSlice;
      const int c = sizeof(T) == 4 ? col_at<C16>(A, q, i, i >> 6) : A.col[q];
      s = s + val[q] * z[c];
    }
    const T zi = z[i] - s / dg[i];
    z[i] = zi;
    v[0] = ri * zi;
  }
  if (part) block_partials<OpSum, 1>(v, part);
}

// --------------------------------------------------- mixed precision glue
__global__ void k_mp_scale_down(int n, const double *r, const KS *st, float *r32, float *x32, KS *s32,
                                double inner_tol, int inner_max) {
  int i = blockIdx.x * kBlock + threadIdx.x;
  const double inv = 1.0 / sqrt(st->rr);
  if (i < n) {
    r32[i] = (float)(r[i] * inv);
    x32[i] = 0.0f;
  }
  if (i == 0) {
    s32->it = 0;
    s32->ierr = 0;
    s32->done = 0;
    s32->bnrm = 1.0;
    s32->tol = inner_tol;
    s32->maxit = inner_max;
  }
}

__global__ void k_mp_correct(int n, const float *x32, const KS *st, double *x) {
  int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] = x[i] + sqrt(st->rr) * (double)x32[i];
}

// streaming copy (calibration of traffic counters and achievable bandwidth)
__global__ void k_copy4(long long n4, const float4 *a, float4 *b) {
  const long long base = (long long)blockIdx.x * kBlock * 4 + threadIdx.x;
  float4 v[4];
#pragma unroll
  for (int u = 0; u < 4; u++)
    if (base + u * kBlock < n4) v[u] = a[base + u * kBlock];
#pragma unroll
  for (int u = 0; u < 4; u++)
    if (base + u * kBlock < n4) b[base + u * kBlock] = v[u];
}

// streaming read of a zero-filled buffer: evicts the last-level cache before
// a cold-cache timing (reads only, so no dirty lines drain during the timed
// kernel); the store never happens for zeros but keeps the loads alive
__global__ void k_touch(long long n4, const float4 *a, float *sink) {
  float acc = 0.0f;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n4; i += (long long)gridDim.x * kBlock) {
    const float4 v = a[i];
    acc += v.x + v.y + v.z + v.w;
  }
  if (acc == 1.0f) sink[0] = acc;
}

// copy with non-temporal stores (the destination bypasses the caches)
typedef float f4v __attribute__((ext_vector_type(4)));
__global__ void k_copy4_nt(long long n4, const float4 *a, float4 *b) {
  const long long base = (long long)blockIdx.x * kBlock * 4 + threadIdx.x;
  f4v v[4];
#pragma unroll
  for (int u = 0; u < 4; u++)
    if (base + u * kBlock < n4) v[u] = *(const f4v *)&a[base + u * kBlock];
#pragma unroll
  for (int u = 0; u < 4; u++)
    if (base + u * kBlock < n4) __builtin_nontemporal_store(v[u], (f4v *)&b[base + u * kBlock]);
}

}  // namespace

// Average duration of a streaming kernel over `bytes`: kind 0 = k_copy4,
// 1 = copy with non-temporal stores, 2 = read only (k_touch, 8192 blocks).
double time_stream(long long bytes, int kind, int reps) {
  const long long n4 = bytes / 16;
  DBuf<float4> a(n4), b(kind == 2 ? 1 : n4);
  DBuf<float> sink(1);
  MS_HIP(hipMemsetAsync(a.p, 0, n4 * 16, stream()));
  const int grid = (int)((n4 + 4 * kBlock - 1) / (4 * kBlock));
  auto go = [&]() {
    if (kind == 0) hipLaunchKernelGGL(k_copy4, dim3(grid), dim3(kBlock), 0, stream(), n4, a.p, b.p);
    else if (kind == 1) hipLaunchKernelGGL(k_copy4_nt, dim3(grid), dim3(kBlock), 0, stream(), n4, a.p, b.p);
    else hipLaunchKernelGGL(k_touch, dim3(8192), dim3(kBlock), 0, stream(), n4, a.p, sink.p);
  };
  for (int i = 0; i < 2; i++) go();
  hipEvent_t e0, e1;
  MS_HIP(hipEventCreate(&e0));
  MS_HIP(hipEventCreate(&e1));
  MS_HIP(hipEventRecord(e0, stream()));
  for (int i = 0; i < reps; i++) go();
  MS_HIP(hipEventRecord(e1, stream()));
  MS_HIP(hipEventSynchronize(e1));
  float ms = 0.0f;
  MS_HIP(hipEventElapsedTime(&ms, e0, e1));
  MS_HIP(hipEventDestroy(e0));
  MS_HIP(hipEventDestroy(e1));
  MS_CHECK_LAUNCH();
  return (double)ms / reps;
}

double time_copy(long long bytes, int reps) {
  const long long n4 = bytes / 16;
  DBuf<float4> a(n4), b(n4);
  MS_HIP(hipMemsetAsync(a.p, 0, n4 * 16, stream()));
  const int grid = (int)((n4 + 4 * kBlock - 1) / (4 * kBlock));
  for (int i = 0; i < 2; i++) hipLaunchKernelGGL(k_copy4, dim3(grid), dim3(kBlock), 0, stream(), n4, a.p, b.p);
  hipEvent_t e0, e1;
  MS_HIP(hipEventCreate(&e0));
  MS_HIP(hipEventCreate(&e1));
  MS_HIP(hipEventRecord(e0, stream()));
  for (int i = 0; i < reps; i++) hipLaunchKernelGGL(k_copy4, dim3(grid), dim3(kBlock), 0, stream(), n4, a.p, b.p);
  MS_HIP(hipEventRecord(e1, stream()));
  MS_HIP(hipEventSynchronize(e1));
  float ms = 0.0f;
  MS_HIP(hipEventElapsedTime(&ms, e0, e1));
  MS_HIP(hipEventDestroy(e0));
  MS_HIP(hipEventDestroy(e1));
  MS_CHECK_LAUNCH();
  return (double)ms / reps;
}

// ============================================================ host side

template <class Op, int NV, class T, class Fin>
static void finish(int nparts, const T *part, Fin fin) {
  hipLaunchKernelGGL((k_finish<Op, NV, T, Fin>), dim3(1), dim3(kFinThreads), 0, stream(), nparts, part, fin);
}

Krylov::Krylov(const SellPattern *pat_) : pat(pat_), n(pat_->n) {
  nblk_ = nblocks(n);
  for (DBuf<double> *b : {&r_, &r0_, &p_, &q_, &z_, &s_, &t_, &ph_, &sh_, &dg_}) b->alloc(n);
  part_.alloc(4 * ((size_t)std::max(nblk_, pat_->coarse.nchunks) + 64) * 2);
  prz_.alloc(2 * ((size_t)nblk_ + 64) + kMaxAgg);
  st_.alloc(1);
  flag_.alloc(1);
  host_ = borrow_host_state();
  hpin_ = host_.pin;
  for (int i = 0; i < 2; i++) state_ev_[i] = host_.ev[i];
}

Krylov::~Krylov() {
  if (chunk_exec_) {
    std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
    (void)hipGraphExecDestroy(chunk_exec_);
  }
  give_back_host_state(host_);
}

// Pinned page and events of a solver, kept for the next one: allocating and
// freeing the page alone takes 75 us, and every solver call on a caller's
// matrix has a solver of its own.  At most kIdleHostStates are kept.
namespace {
constexpr size_t kIdleHostStates = 32;
std::mutex g_host_mu;
std::vector<Krylov::HostState> g_host_idle;
}  // namespace
Krylov::HostState Krylov::borrow_host_state() {
  int dev = 0;
  MS_HIP(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> g(g_host_mu);
    for (size_t i = 0; i < g_host_idle.size(); i++)
      if (g_host_idle[i].dev == dev) {
        const HostState h = g_host_idle[i];
        g_host_idle.erase(g_host_idle.begin() + i);
        return h;
      }
  }
  HostState h;
  h.dev = dev;
  std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
  MS_HIP(hipHostMalloc(&h.pin, 4096, hipHostMallocDefault));
  for (auto &e : h.ev) MS_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  return h;
}
void Krylov::give_back_host_state(const HostState &h) {
  if (!h.pin) return;
  // nothing of this solver may still write the page; waiting on a stream that
  // another thread (a server's) is capturing would end that capture
  const auto lk = library_stream_lock();
  const bool ok = hipStreamSynchronize(stream()) == hipSuccess;
  if (ok) {
    std::lock_guard<std::mutex> g(g_host_mu);
    if (g_host_idle.size() < kIdleHostStates) {
      g_host_idle.push_back(h);
      return;
    }
  }
  std::lock_guard<std::recursive_mutex> alk(device_alloc_mutex());
  for (const auto &e : h.ev)
    if (e) (void)hipEventDestroy(e);
  (void)hipHostFree(h.pin);
}

void Krylov::ensure32() {
  if (have32_) return;
  for (DBuf<float> *v : {&r32_, &r032_, &p32_, &q32_, &z32_, &s32_, &t32_, &ph32_, &sh32_, &x32_, &dg32_}) v->alloc(n);
  part32_.alloc(4 * ((size_t)std::max(nblk_, pat->coarse.nchunks) + 64) * 2);
  prz32_.alloc(2 * ((size_t)nblk_ + 64) + kMaxAgg);
  st32_.alloc(1);
  have32_ = true;
}

template <class T>
KS Krylov::read_state(KS *d) {
  MS_HIP(hipMemcpyAsync(hpin_, d, sizeof(KS), hipMemcpyDeviceToHost, stream()));
  MS_HIP(hipStreamSynchronize(stream()));
  KS h;
  std::memcpy(&h, hpin_, sizeof(KS));
  return h;
}

void Krylov::spmv(const double *val, const double *x, double *y) {
  hipLaunchKernelGGL(k_spmv<double>, dim3(nblk_), dim3(kBlock), 0, stream(), n, matof(pat), val, x, y);
  MS_CHECK_LAUNCH();
}

void Krylov::spmv32(const double *val64, const float *v32, float *p, float *q, KS *st, float *part,
                    hipEvent_t e0, hipEvent_t e1, const PUp *pu) {
  (void)val64;
  const dim3 G(nblk_), B(kBlock);
  hipStream_t S = stream();
  if (matfree_on()) {
    const MatFree &M = *mf_;
    const Mat AM = matof(M.A);
    const MfCols mc{M.c16, M.win};
    const dim3 G0(nblocks(M.n0));
    const PUp u = pu ? *pu : PUp{};
    // stage 1 then stage 2; the start event on the first launch, the stop
    // event on the second
    auto launch = [&](auto k1, auto k2) {
      if (e0) hipExtLaunchKernelGGL(k1, G0, B, 0, S, e0, nullptr, 0, M.n0, AM, mc, M.w, p, M.hx, st, u);
      else hipLaunchKernelGGL(k1, G0, B, 0, S, M.n0, AM, mc, M.w, p, M.hx, st, u);
      if (e1) hipExtLaunchKernelGGL(k2, G, B, 0, S, nullptr, e1, 0, M.n0, M.n1, AM, mc, M.w, p, M.hx, q, st, part, u);
      else hipLaunchKernelGGL(k2, G, B, 0, S, M.n0, M.n1, AM, mc, M.w, p, M.hx, q, st, part, u);
    };
    if (pu) launch(k_mf_stage1<true>, k_mf_stage2<true>);
    else launch(k_mf_stage1<false>, k_mf_stage2<false>);
    return;
  }
  const Mat A = matof(pat);
  if (e0 || e1) {
    if (pat->has16)
      hipExtLaunchKernelGGL((k_pcg_spmv<float, 1>), G, B, 0, S, e0, e1, 0, n, A, v32, p, q, st, part);
    else
      hipExtLaunchKernelGGL((k_pcg_spmv<float, 0>), G, B, 0, S, e0, e1, 0, n, A, v32, p, q, st, part);
  } else if (pat->has16) {
    hipLaunchKernelGGL((k_pcg_spmv<float, 1>), G, B, 0, S, n, A, v32, p, q, st, part);
  } else {
    hipLaunchKernelGGL((k_pcg_spmv<float, 0>), G, B, 0, S, n, A, v32, p, q, st, part);
  }
}

double Krylov::time_spmv(const double *val, bool fp32, int reps, bool cold) {
  Mat A = matof(pat);
  const dim3 G(nblk_), B(kBlock);
  hipStream_t S = stream();
  KS h{};
  MS_HIP(hipMemcpyAsync(st_.p, &h, sizeof(h), hipMemcpyHostToDevice, S));
  if (fp32) {
    last_ = SetupKey{};
    ensure32();
    if (val32_.n < (size_t)pat->nstore) val32_.alloc(pat->nstore);
    hipLaunchKernelGGL(k_mat32_diff, G, B, 0, S, n, A, val, val32_.p);
    MS_HIP(hipMemsetAsync(p32_.p, 0, n * sizeof(float), S));
  } else {
    MS_HIP(hipMemsetAsync(p_.p, 0, n * sizeof(double), S));
  }
  auto launch = [&]() {
    if (fp32)
      spmv32(val, val32_.p, p32_.p, q32_.p, st_.p, part32_.p, nullptr, nullptr);
    else
      hipLaunchKernelGGL(k_pcg_spmv<double>, G, B, 0, S, n, A, val, p_.p, q_.p, st_.p, part_.p);
  };
  for (int i = 0; i < 3; i++) launch();
  if (cold) {
    // each launch timed alone after a 512 MiB read (twice the 256 MB
    // last-level cache), so its matrix and vectors come from HBM
    const long long n4 = (512LL << 20) / 16;
    DBuf<float4> flush(n4);
    DBuf<float> sink(1);
    MS_HIP(hipMemsetAsync(flush.p, 0, n4 * 16, S));
    std::vector<hipEvent_t> ev(2 * (size_t)reps);
    for (auto &e : ev) MS_HIP(hipEventCreate(&e));
    for (int i = 0; i < reps; i++) {
      hipLaunchKernelGGL(k_touch, dim3(8192), B, 0, S, n4, flush.p, sink.p);
      MS_HIP(hipEventRecord(ev[2 * i], S));
      launch();
      MS_HIP(hipEventRecord(ev[2 * i + 1], S));
    }
    MS_HIP(hipEventSynchronize(ev.back()));
    double tot = 0.0;
    for (int i = 0; i < reps; i++) {
      float ms = 0.0f;
      MS_HIP(hipEventElapsedTime(&ms, ev[2 * i], ev[2 * i + 1]));
      tot += ms;
    }
    for (auto &e : ev) MS_HIP(hipEventDestroy(e));
    MS_CHECK_LAUNCH();
    return tot / reps;
  }
  hipEvent_t e0, e1;
  MS_HIP(hipEventCreate(&e0));
  MS_HIP(hipEventCreate(&e1));
  MS_HIP(hipEventRecord(e0, S));
  for (int i = 0; i < reps; i++) launch();
  MS_HIP(hipEventRecord(e1, S));
  MS_HIP(hipEventSynchronize(e1));
  float ms = 0.0f;
  MS_HIP(hipEventElapsedTime(&ms, e0, e1));
  MS_HIP(hipEventDestroy(e0));
  MS_HIP(hipEventDestroy(e1));
  MS_CHECK_LAUNCH();
  return (double)ms / reps;
}

int Krylov::setup_pc64(PcKind pc, const double *val) {
  Mat A = matof(pat);
  if ((pc == PC_DILU || pc == PC_NATURAL_IC0) && !pat->symmetric)
    fail(MS_EINVAL, "IC0 / DILU need a structurally symmetric pattern");
  if (pc == PC_JACOBI) {
    hipLaunchKernelGGL(k_extract_diag<double>, dim3(nblk_), dim3(kBlock), 0, stream(), n, A, val, dg_.p);
    MS_CHECK_LAUNCH();
    return 0;
  }
  if (pc == PC_DILU) {
    for (size_t c = 0; c + 1 < pat->color_ptr.size(); c++) {
      int r0 = pat->color_ptr[c], r1 = pat->color_ptr[c + 1];
      if (r1 > r0)
        hipLaunchKernelGGL(k_dilu_setup<double>, dim3(nblocks(r1 - r0)), dim3(kBlock), 0, stream(), r0, r1, A,
                           pat->d_tpos.p, val, dg_.p);
    }
    MS_CHECK_LAUNCH();
    return 0;
  }
  if (!pat->has_levels) fail(MS_EINVAL, "natural-order factorization needs level schedules");
  if (fac_.n < (size_t)pat->nstore) fac_.alloc(pat->nstore);
  MS_HIP(hipMemcpyAsync(fac_.p, val, pat->nstore * sizeof(double), hipMemcpyDeviceToDevice, stream()));
  MS_HIP(hipMemsetAsync(flag_.p, 0, sizeof(int), stream()));
  const bool ic0 = pc == PC_NATURAL_IC0;
  factor_levels(*pat, fac_.p, ic0, flag_.p, diag_);
  lev_.pack(*pat, fac_.p, ic0);
  int h = 0;
  MS_HIP(hipMemcpyAsync(hpin_, flag_.p, sizeof(int), hipMemcpyDeviceToHost, stream()));
  MS_HIP(hipStreamSynchronize(stream()));
  std::memcpy(&h, hpin_, sizeof(int));
  return h;
}

void Krylov::setup_pc32(PcKind pc, const double *val) {
  Mat A = matof(pat);
  ensure32();
  if (pc == PC_JACOBI || pc == PC_DILU) {
    // the diagonal slot of val32 holds row sums: take d from the FP64 matrix
    setup_pc64(pc, val);
    hipLaunchKernelGGL(k_to_float, dim3(nblk_), dim3(kBlock), 0, stream(), (long long)n, dg_.p, dg32_.p);
  } else {
    int e = setup_pc64(pc, val);
    if (e) fail(MS_EINVAL, "factorization failed in mixed-precision setup");
    if (fac32_.n < (size_t)pat->nstore) fac32_.alloc(pat->nstore);
    hipLaunchKernelGGL(k_to_float, dim3(nblocks(pat->nstore)), dim3(kBlock), 0, stream(), pat->nstore, fac_.p,
                       fac32_.p);
    lev32_.pack(*pat, fac32_.p, pc == PC_NATURAL_IC0);
  }
  MS_CHECK_LAUNCH();
}

// the column format of a SELL pattern as a template argument of the FP32
// kernels (the FP64 kernels always read 32-bit columns)
template <class T>
static int c16_of(const SellPattern *pat) {
  return sizeof(T) == 4 && pat->has16 ? 1 : 0;
}

template <class T>
void Krylov::apply_pc(PcKind pc, const T *val, const T *fac, const T *dg, const T *in, T *out, const int *done,
                      bool staged) {
  Mat A = matof(pat);
  if (pc == PC_JACOBI) {
    if (!staged) hipLaunchKernelGGL(k_jacobi<T>, dim3(nblk_), dim3(kBlock), 0, stream(), n, in, dg, out, done);
  } else if (pc == PC_DILU) {
    const auto &cp = pat->color_ptr;
    const int nc = (int)cp.size() - 1;
    if (cp[1] > cp[0] && !staged)
      hipLaunchKernelGGL(k_dilu_first<T>, dim3(nblocks(cp[1] - cp[0])), dim3(kBlock), 0, stream(), cp[0], cp[1], dg,
                         in, out, done);
    for (int c = 1; c < nc; c++)
      if (cp[c + 1] > cp[c]) {
        const int gb = nblocks(cp[c + 1] - cp[c]);
        if (c16_of<T>(pat))
          hipLaunchKernelGGL((k_dilu_fwd<T, 1>), dim3(gb), dim3(kBlock), 0, stream(), cp[c], cp[c + 1], gb, A, val, dg,
                             in, out, (int)(c == nc - 1), done, (T *)nullptr, CoWork<T>{});
        else
          hipLaunchKernelGGL((k_dilu_fwd<T, 0>), dim3(gb), dim3(kBlock), 0, stream(), cp[c], cp[c + 1], gb, A, val, dg,
                             in, out, (int)(c == nc - 1), done, (T *)nullptr, CoWork<T>{});
      }
    for (int c = nc - 2; c >= 0; c--)
      if (cp[c + 1] > cp[c])
        if (c16_of<T>(pat))
          hipLaunchKernelGGL((k_dilu_bwd<T, 1>), dim3(nblocks(cp[c + 1] - cp[c])), dim3(kBlock), 0, stream(), cp[c],
                             cp[c + 1], A, val, dg, in, out, done, (T *)nullptr);
        else
          hipLaunchKernelGGL((k_dilu_bwd<T, 0>), dim3(nblocks(cp[c + 1] - cp[c])), dim3(kBlock), 0, stream(), cp[c],
                             cp[c + 1], A, val, dg, in, out, done, (T *)nullptr);
  } else {
    if constexpr (sizeof(T) == 8) lev_.apply(*pat, pc == PC_NATURAL_IC0, fac, in, out, done);
    else lev32_.apply(*pat, pc == PC_NATURAL_IC0, fac, in, out, done);
  }
  MS_CHECK_LAUNCH();
}

// DILU sweeps of colours 1.. with fused r.z partials (one section per launch);
// returns the number of partials written.  With cw.nwg > 0 the coarse solve
// rides along the first forward launch and its c.nu partials follow the
// sweep sections, so the sum of all partials is r.z of the two-level
// preconditioner.
template <class T>
static int dilu_sweeps(const SellPattern *pat, Mat A, const T *val, const T *dg, const T *r, T *z, const int *done,
                       T *part, CoWork<T> cw = CoWork<T>{}) {
  const auto &cp = pat->color_ptr;
  const int ncol = (int)cp.size() - 1;
  int total = 0;
  for (int c = 1; c < ncol; c++) total += nblocks(cp[c + 1] - cp[c]);
  for (int c = ncol - 2; c >= 0; c--) total += nblocks(cp[c + 1] - cp[c]);
  cw.cnu_part = part + total;
  T *sec = part;
  bool first = true;
  for (int c = 1; c < ncol; c++)
    if (cp[c + 1] > cp[c]) {
      const int gb = nblocks(cp[c + 1] - cp[c]);
      CoWork<T> cwl = cw;
      if (!first) cwl.nwg = 0;
      if (c16_of<T>(pat))
        hipLaunchKernelGGL((k_dilu_fwd<T, 1>), dim3(gb + cwl.nwg), dim3(kBlock), 0, stream(), cp[c], cp[c + 1], gb, A,
                           val, dg, r, z, (int)(c == ncol - 1), done, sec, cwl);
      else
        hipLaunchKernelGGL((k_dilu_fwd<T, 0>), dim3(gb + cwl.nwg), dim3(kBlock), 0, stream(), cp[c], cp[c + 1], gb, A,
                           val, dg, r, z, (int)(c == ncol - 1), done, sec, cwl);
      first = false;
      sec += gb;
    }
  for (int c = ncol - 2; c >= 0; c--)
    if (cp[c + 1] > cp[c]) {
      const int gb = nblocks(cp[c + 1] - cp[c]);
      if (c16_of<T>(pat))
        hipLaunchKernelGGL((k_dilu_bwd<T, 1>), dim3(gb), dim3(kBlock), 0, stream(), cp[c], cp[c + 1], A, val, dg, r, z,
                           done, sec);
      else
        hipLaunchKernelGGL((k_dilu_bwd<T, 0>), dim3(gb), dim3(kBlock), 0, stream(), cp[c], cp[c + 1], A, val, dg, r, z,
                           done, sec);
      sec += gb;
    }
  return total + (first ? 0 : cw.nwg);
}

// ---- PCG (FP64, reference recurrences) -------------------------------------
static Rows rows_of(const SellPattern *pat, bool coarse) {
  if (!coarse) return Rows{nullptr, nullptr, pat->n};
  return Rows{pat->coarse.d_chunk_ptr.p, pat->coarse.d_chunk_agg.p, pat->n};
}
static CoDev codev_of(const SellPattern *pat, const CoarseMat &cm, bool coarse, KS *st) {
  if (!coarse) return CoDev{0, nullptr, nullptr, nullptr, nullptr, st};
  const Coarse &C = pat->coarse;
  return CoDev{C.k, C.d_agg_cptr.p, C.d_agg_cidx.p, cm.Einv.p, cm.nu.p, st};
}
template <class T>
static CoWork<T> cowork_of(const SellPattern *pat, const CoarseMat &cm, bool fused, const T *csum) {
  CoWork<T> cw{};
  if (!fused) return cw;
  const Coarse &C = pat->coarse;
  cw.k = C.k;
  cw.nwg = (C.k + kBlock / 64 - 1) / (kBlock / 64);
  cw.agg_cptr = C.d_agg_cptr.p;
  cw.Einv = cm.Einv.p;
  cw.nu = cm.nu.p;
  cw.csum = csum;
  return cw;
}

template <int NV, class T, class Fin>
static void finish_co(int nparts, const T *part, Fin fin, const CoDev &co) {
  hipLaunchKernelGGL((k_finish_co<NV, T, Fin>), dim3(1), dim3(kFinThreads), 0, stream(), nparts, part, fin, co);
}

static bool coarse_inv32_enabled();
void Krylov::coarse_setup(const double *val) {
  const Coarse &C = pat->coarse;
  CoarseMat &M = cm_;
  M.ensure(C.k);
  const long long kk = (long long)C.k * C.k;
  const int nE = (int)C.e_key.size();
  hipLaunchKernelGGL(k_fill64, dim3(nblocks(kk)), dim3(kBlock), 0, stream(), kk, M.E.p, 0.0);
  if (M.Eparts.n < (size_t)nE * kEParts) M.Eparts.alloc((size_t)nE * kEParts);
  hipLaunchKernelGGL(k_coarse_E_parts, dim3(nblocks((long long)nE * kEParts, kBlock / 64)), dim3(kBlock), 0,
                     stream(), nE, C.d_e_ptr.p, C.d_e_slot.p, val, M.Eparts.p);
  hipLaunchKernelGGL(k_coarse_E_sum, dim3(nblocks(nE)), dim3(kBlock), 0, stream(), nE, C.d_e_key.p, M.Eparts.p,
                     M.E.p);
  if (C.k <= kInvRegMax && coarse_inv32_enabled()) {
    // one workgroup, E held in registers, Gauss-Jordan in FP32
    hipLaunchKernelGGL(k_coarse_inv, dim3(1), dim3(kInvThreads), 0, stream(), C.k, M.E.p, M.Einv.p);
    MS_CHECK_LAUNCH();
    return;
  }
  const int kb = (C.k + kGjBlock - 1) / kGjBlock;
  double *in = M.E.p, *out = M.W.p;
  for (int j = 0; j < kb; j++, std::swap(in, out))
    hipLaunchKernelGGL(k_gj_block, dim3(kb, kb), dim3(kBlock), 0, stream(), C.k, j, in, out,
                       j + 1 == kb ? M.Einv.p : nullptr);
  MS_CHECK_LAUNCH();
}

// out += Z E^-1 c, c the chunk sums a BiCGSTAB launch left in co_part_
template <class T>
void Krylov::coarse_apply(T *out, KS *st) {
  const Coarse &C = pat->coarse;
  const int ncn = (C.k + kSplitRows - 1) / kSplitRows;
  if (cnu_split_.n < (size_t)ncn) cnu_split_.alloc(ncn);
  hipLaunchKernelGGL(k_cx_coarse<double>, dim3(ncn), dim3(kFinThreads), 0, stream(), C.k, C.d_agg_cptr.p, cm_.Einv.p,
                     co_part_.p, cm_.nu.p, cnu_split_.p, st);
  hipLaunchKernelGGL((k_co_prolong<T>), dim3(C.nchunks), dim3(kBlock), 0, stream(), rows_of(pat, true), cm_.nu.p, out,
                     &st->done);
}

// buffers of the two-launch PCG: the vectors of the precision, p double
// buffered in the BiCGSTAB's ph, three partial arrays
template <class T>
Krylov::Cg2<T> Krylov::cg2(PcKind pc) {
  Cg2<T> c;
  c.pc = pc;
  c.mode = pc == PC_JACOBI ? 1 : (pc == PC_DILU ? 2 : 0);
  c.G = std::min(nblk_, kCgGrid);
  const size_t stride = (size_t)nblk_ + 64;
  T *part;
  if constexpr (sizeof(T) == 8) {
    c.r = r_.p, c.z = z_.p, c.p0 = p_.p, c.p1 = ph_.p, c.q = q_.p, c.dg = dg_.p;
    part = part_.p;
    c.swp = prz_.p;
  } else {
    c.r = r32_.p, c.z = z32_.p, c.p0 = p32_.p, c.p1 = ph32_.p, c.q = q32_.p, c.dg = dg32_.p;
    part = part32_.p;
    c.swp = prz32_.p;
  }
  c.rr = part;
  c.rz = part + stride;
  c.pq = part + 2 * stride;
  c.nrz = c.G;
  if (c.mode == 2) {   // the sweeps' partials: rows of colours 1.. forward, all but the last backward
    const auto &cp = pat->color_ptr;
    const int nc = (int)cp.size() - 1;
    c.nrz = 0;
    for (int k = 1; k < nc; k++) c.nrz += nblocks(cp[k + 1] - cp[k]);
    for (int k = nc - 2; k >= 0; k--) c.nrz += nblocks(cp[k + 1] - cp[k]);
    c.rz = c.swp;
  } else if (c.mode == 0) {
    c.nrz = nblk_;
    c.rz = c.swp;
  }
  return c;
}

// buffers of the PCG with a coarse space (Jacobi, or DILU with the coarse
// solve riding along the sweeps)
template <class T>
Krylov::Cx<T> Krylov::cx(PcKind pc) {
  const Coarse &C = pat->coarse;
  Cx<T> c;
  c.mode = pc == PC_JACOBI ? 1 : 2;
  c.G = std::min((C.nchunks + kBlock / kSlice - 1) / (kBlock / kSlice), kCxGrid);
  const size_t stride = (size_t)std::max(nblk_, C.nchunks) + 64;
  T *part, *sweep;
  if constexpr (sizeof(T) == 8) {
    c.r = r_.p, c.z = z_.p, c.p = p_.p, c.q = q_.p, c.dg = dg_.p;
    part = part_.p;
    sweep = prz_.p;
  } else {
    c.r = r32_.p, c.z = z32_.p, c.p = p32_.p, c.q = q32_.p, c.dg = dg32_.p;
    part = part32_.p;
    sweep = prz32_.p;
  }
  c.rr = part;
  c.rz = part + stride;
  c.csum = part + 2 * stride;
  c.pq = part + 3 * stride;
  c.nrz = c.G;
  if (c.mode == 1) {
    c.ncn = (C.k + kSplitRows - 1) / kSplitRows;
    if (cnu_split_.n < (size_t)c.ncn) cnu_split_.alloc(c.ncn);
  } else {
    c.rz = sweep;
    c.cw = (C.k + kBlock / 64 - 1) / (kBlock / 64);
    c.nrz = c.cw;
    const auto &cp = pat->color_ptr;
    const int nc = (int)cp.size() - 1;
    for (int k = 1; k < nc; k++) c.nrz += nblocks(cp[k + 1] - cp[k]);
    for (int k = nc - 2; k >= 0; k--) c.nrz += nblocks(cp[k + 1] - cp[k]);
  }
  return c;
}

static Chunks chunks_of(const SellPattern *pat) {
  const Coarse &C = pat->coarse;
  return Chunks{C.d_chunk_ptr.p, C.d_chunk_agg.p, C.d_chunk_pos.p, C.nchunks};
}

// the partials a (and b) for a launch of `readers` workgroups that all add them
// up: as they are, or folded
template <class T>
Krylov::Parts<T> Krylov::parts_for(int readers, int m, const T *a, const T *b, const KS *st) {
  if ((long long)m * readers * (long long)sizeof(T) * (b ? 2 : 1) <= kFoldBytes) return {m, a, b};
  // the end of the partials' buffer: the solvers use six of its eight parts at most
  T *out;
  if constexpr (sizeof(T) == 8) out = part_.p + part_.n - 2 * kFoldParts;
  else out = part32_.p + part32_.n - 2 * kFoldParts;
  hipLaunchKernelGGL(k_fold_parts<T>, dim3(kFoldParts, b ? 2 : 1), dim3(kBlock), 0, stream(), m, a, b, out, st);
  return {kFoldParts, out, out + kFoldParts};
}

// the preconditioner of the current r, and p
template <class T, bool MIXED>
void Krylov::cx_p(const Cx<T> &c, int what) {
  Chunks C = chunks_of(pat);
  if (what == kCxTest) C.n = 0;
  const int G = what == kCxTest ? 1 : c.G;
  const Parts<T> rz = parts_for<T>(G, c.nrz, c.rz, nullptr, st_.p);
  hipLaunchKernelGGL((k_cx_p<T, MIXED>), dim3(G), dim3(kBlock), 0, stream(), C, c.r, c.z, c.dg, c.mode, c.p, cm_.nu.p,
                     st_.p, CgParts{c.G, rz.n}, c.rr, rz.a, c.ncn, cnu_split_.p, what);
}

template <class T, bool MIXED>
void Krylov::cx_direction(const Cx<T> &c, const T *val, int what) {
  const Coarse &C = pat->coarse;
  hipStream_t S = stream();
  if (c.mode == 1) {
    hipLaunchKernelGGL(k_cx_coarse<T>, dim3(c.ncn), dim3(kFinThreads), 0, S, C.k, C.d_agg_cptr.p, cm_.Einv.p, c.csum,
                       cm_.nu.p, cnu_split_.p, st_.p);
  } else {
    dilu_sweeps<T>(pat, matof(pat), val, c.dg, c.r, c.z, &st_.p->done, c.rz, cowork_of<T>(pat, cm_, true, c.csum));
  }
  cx_p<T, MIXED>(c, what);
}

// sums and direction of a new r: the initial one (r64 null), or the one of a
// reliable update; direction = false: p is already that of the next iteration
template <class T, bool MIXED>
void Krylov::cx_restart(const Cx<T> &c, const T *val, const double *r64, bool direction) {
  hipLaunchKernelGGL(k_cx_start<T>, dim3(c.G), dim3(kBlock), 0, stream(), chunks_of(pat), r64, c.r, c.p, c.z, c.dg,
                     c.mode, pat->color_ptr[1], st_.p, c.rr, c.rz, c.csum);
  if (direction) cx_direction<T, MIXED>(c, val, kCxAll);
  MS_CHECK_LAUNCH();
}

// the part of an iteration after the product
template <class T, bool MIXED, class X>
void Krylov::cx_update(const Cx<T> &c, const T *val, X *x, bool ride) {
  const Parts<T> pq = parts_for<T>(c.G, nblk_, c.pq, nullptr, st_.p);
  hipLaunchKernelGGL((k_cx_update<T, X>), dim3(c.G), dim3(kBlock), 0, stream(), chunks_of(pat), pq.n, pq.a, c.p, c.q,
                     x, c.r, c.z, c.dg, c.mode, pat->color_ptr[1], st_.p, c.rr, c.rz, c.csum);
  cx_direction<T, MIXED>(c, val, ride ? kCxTest : kCxAll);
}

// z and the r.z partials of the current r
template <class T>
void Krylov::cg2_precond(const Cg2<T> &c, const T *val, const T *fac) {
  if (c.mode == 2) {
    dilu_sweeps<T>(pat, matof(pat), val, c.dg, c.r, c.z, &st_.p->done, c.swp);
  } else if (c.mode == 0) {
    apply_pc<T>(c.pc, val, fac, c.dg, c.r, c.z, &st_.p->done);
    hipLaunchKernelGGL(k_dot<T>, dim3(nblk_), dim3(kBlock), 0, stream(), n, c.r, c.z, st_.p, c.swp);
  }
}

template <class T>
void Krylov::cg2_start(const Cg2<T> &c, const T *val, const T *fac) {
  if (c.mode)
    hipLaunchKernelGGL(k_cg_z<T>, dim3(c.G), dim3(kBlock), 0, stream(), n, c.r, c.dg, c.z, c.mode, pat->color_ptr[1],
                       st_.p, c.rz);
  cg2_precond<T>(c, val, fac);
  MS_CHECK_LAUNCH();
}

template <class T, bool MIXED, class X>
void Krylov::cg2_iteration(const Cg2<T> &c, const T *val, const T *fac, X *x, hipEvent_t e0, hipEvent_t e1) {
  const Mat A = matof(pat);
  const dim3 G(c.G), B(kBlock);
  hipStream_t S = stream();
  const Parts<T> rz = parts_for<T>(c.G, c.nrz, c.rz, nullptr, st_.p);
  const CgParts np{c.G, rz.n};
  auto ps = [&](auto k) {
    if (e0) hipExtLaunchKernelGGL(k, G, B, 0, S, e0, e1, 0, n, A, val, c.z, c.p0, c.p1, c.q, st_.p, np, c.rr, rz.a, c.pq);
    else hipLaunchKernelGGL(k, G, B, 0, S, n, A, val, c.z, c.p0, c.p1, c.q, st_.p, np, c.rr, rz.a, c.pq);
  };
  if (sizeof(T) == 4 && pat->has16) ps(k_cg_ps<T, MIXED, 1>);
  else ps(k_cg_ps<T, MIXED, 0>);
  hipLaunchKernelGGL((k_cg_xr<T, X>), G, B, 0, S, n, c.p0, c.p1, c.q, x, c.r, c.z, c.dg, c.mode, pat->color_ptr[1],
                     st_.p, c.G, c.pq, c.rr, c.rz);
  cg2_precond<T>(c, val, fac);
}

// the whole matrix fits the registers of one workgroup (k_cg_small)
bool Krylov::small_system() const {
  if (n > kSmallRows) return false;
  for (int s = 0; s < pat->nslices; s++)
    if (pat->off[s + 1] - pat->off[s] > (long long)kSmallWidth * kSlice) return false;
  return true;
}

SolveResult Krylov::pcg(const double *val, const double *b, double *x, double tol, int maxit, PcKind pc,
                        bool coarse, bool reuse) {
  SolveResult R;
  Mat A = matof(pat);
  const dim3 G(nblk_), B(kBlock);
  hipStream_t S = stream();
  KS *st = st_.p;
  double *part = part_.p;
  coarse = coarse && pat->coarse.k > 0;
  // DILU with a coarse space: the coarse solve rides along the forward sweep
  const bool fused = coarse && pc == PC_DILU && pat->color_ptr.size() > 2;
  KS h{};
  h.tol = tol;
  h.maxit = maxit;
  h.coarse = coarse && !fused && pc != PC_JACOBI;
  MS_HIP(hipMemcpyAsync(st, &h, sizeof(h), hipMemcpyHostToDevice, S));
  hipLaunchKernelGGL(k_sumsq<double>, G, B, 0, S, n, b, part);
  finish<OpSum, 1>(nblk_, part, FinBnorm{st});
  MS_CHECK_LAUNCH();
  KS hs = read_state<double>(st);
  if (hs.bnrm == 0.0) {
    MS_HIP(hipMemsetAsync(x, 0, n * sizeof(double), S));
    return R;
  }
  const SetupKey key{val, (int)pc, 0, (int)coarse};
  if (!(reuse && last_ == key)) {
    last_ = SetupKey{};
    int fe = setup_pc64(pc, val);
    if (fe) {
      R.ierr = fe + 10;
      return R;
    }
    if (coarse) coarse_setup(val);
    last_ = key;
  }
  hipLaunchKernelGGL(k_residual<double>, G, B, 0, S, n, A, val, b, x, r_.p, part);
  finish<OpSum, 1>(nblk_, part, FinResidual{st});
  MS_CHECK_LAUNCH();
  hs = read_state<double>(st);
  R.res = hs.res;
  if (hs.done) return R;
  const int jac = pc == PC_JACOBI;
  const int *done = &st->done;
  if (!coarse && jac && small_system()) {
    const int rows = n <= kSmallThreads ? 1 : 2, nt = (n + 64 * rows - 1) / (64 * rows) * 64;
    for (int left = maxit; left > 0 && !hs.done; left -= kSmallIters) {
      const int m = std::min(left, kSmallIters);
      if (rows == 1)
        hipLaunchKernelGGL(k_cg_small<1>, dim3(1), dim3(nt), 0, S, n, A, val, dg_.p, x, r_.p, p_.p, st, m);
      else
        hipLaunchKernelGGL(k_cg_small<2>, dim3(1), dim3(nt), 0, S, n, A, val, dg_.p, x, r_.p, p_.p, st, m);
      MS_CHECK_LAUNCH();
      hs = read_state<double>(st);
    }
    R.it = hs.it;
    R.res = hs.res;
    R.ierr = hs.ierr;
    if (!hs.done) {        // DO-loop exhaustion: it = maxit + 1, ierr = 1
      R.it = maxit + 1;
      R.ierr = 1;
    }
    return R;
  }
  if (!coarse) {
    const Cg2<double> cg = cg2<double>(pc);
    cg2_start<double>(cg, val, fac_.p);
    for (int enq = 0, chunk = 8;;) {
      const int m = std::min(chunk, maxit - enq);
      for (int it = 0; it < m; it++) cg2_iteration<double, false>(cg, val, fac_.p, x, nullptr, nullptr);
      hipLaunchKernelGGL((k_cg_peek<double, false>), dim3(1), B, 0, S, st, cg.G, cg.rr);
      MS_CHECK_LAUNCH();
      enq += m;
      hs = read_state<double>(st);
      if (hs.done || enq >= maxit) break;
      chunk = std::min(chunk * 2, 128);
    }
    R.it = hs.it;
    R.res = hs.res;
    R.ierr = hs.ierr;
    if (!hs.done) {        // DO-loop exhaustion: it = maxit + 1, ierr = 1
      R.it = maxit + 1;
      R.ierr = 1;
    }
    return R;
  }
  if (jac || fused) {
    const Cx<double> c = cx<double>(pc);
    cx_restart<double, false>(c, val, nullptr, true);
    for (int enq = 0, chunk = 8;;) {
      const int m = std::min(chunk, maxit - enq);
      for (int it = 0; it < m; it++) {
        hipLaunchKernelGGL((k_pcg_spmv<double, 0>), G, B, 0, S, n, A, val, c.p, c.q, st, c.pq);
        cx_update<double, false>(c, val, x, false);
      }
      MS_CHECK_LAUNCH();
      enq += m;
      hs = read_state<double>(st);
      if (hs.done || enq >= maxit) break;
      chunk = std::min(chunk * 2, 128);
    }
    R.it = hs.it;
    R.res = hs.res;
    R.ierr = hs.ierr;
    if (!hs.done) {
      R.it = maxit + 1;
      R.ierr = 1;
    }
    return R;
  }
  // a coarse space beside a level-scheduled factorization
  const Rows RW = rows_of(pat, true);
  const dim3 GR(pat->coarse.nchunks);
  const CoDev co = codev_of(pat, cm_, true, st);
  const double *nu = cm_.nu.p;
  hipLaunchKernelGGL(k_rsum<double>, GR, B, 0, S, RW, r_.p, st, part);
  finish_co<3>((int)GR.x, part, FinNop{st}, co);
  apply_pc<double>(pc, val, fac_.p, dg_.p, r_.p, z_.p, done);
  hipLaunchKernelGGL(k_pcg_start<double>, GR, B, 0, S, RW, r_.p, z_.p, dg_.p, 0, p_.p, nu, st, part);
  finish<OpSum, 1>((int)GR.x, part, FinRz0{st});
  int enq = 0, chunk = 8;
  while (true) {
    int m = std::min(chunk, maxit - enq);
    for (int it = 0; it < m; it++) {
      hipLaunchKernelGGL(k_pcg_spmv<double>, G, B, 0, S, n, A, val, p_.p, q_.p, st, part);
      finish<OpSum, 1>(nblk_, part, FinPap{st});
      hipLaunchKernelGGL((k_pcg_update<double, double>), GR, B, 0, S, RW, p_.p, q_.p, x, r_.p, z_.p, dg_.p, 0, 0, st,
                         part);
      finish_co<3>((int)GR.x, part, FinUpdate{st}, co);
      apply_pc<double>(pc, val, fac_.p, dg_.p, r_.p, z_.p, done);
      hipLaunchKernelGGL(k_dot<double>, G, B, 0, S, n, r_.p, z_.p, st, part);
      finish<OpSum, 1>(nblk_, part, FinRz{st});
      hipLaunchKernelGGL(k_pcg_p<double>, GR, B, 0, S, RW, r_.p, z_.p, dg_.p, 0, p_.p, nu, st);
    }
    MS_CHECK_LAUNCH();
    enq += m;
    hs = read_state<double>(st);
    if (hs.done || enq >= maxit) break;
    chunk = std::min(chunk * 2, 128);
  }
  R.it = hs.it;
  R.res = hs.res;
  R.ierr = hs.ierr;
  if (!hs.done) {        // DO-loop exhaustion: it = maxit + 1, ierr = 1
    R.it = maxit + 1;
    R.ierr = 1;
  }
  return R;
}

// ---- BiCGSTAB -----------------------------------------------------------------
// partial arrays of a solve in its buffer: r.r, r.r0 | v.r0, s.s | t.t, t.s
template <class T>
static void bi_parts(const SellPattern *pat, T *part, T *(&a)[6]) {
  const size_t stride = (size_t)std::max(nblocks(pat->n), pat->coarse.nchunks) + 64;
  for (int i = 0; i < 6; i++) a[i] = part + i * stride;
}

template <class T>
void Krylov::bi_start(const Bi<T> &w) {
  T *pt[6];
  bi_parts(pat, w.part, pt);
  const int G = std::min((nblk_ + kBlock / kSlice - 1) / (kBlock / kSlice), kCxGrid);
  hipLaunchKernelGGL(k_bi_init<T>, dim3(G), dim3(kBlock), 0, stream(), n, w.r, w.r0, pt[0], pt[1]);
  MS_CHECK_LAUNCH();
}

template <class T>
void Krylov::bi_iteration(const Bi<T> &w, PcKind pc, const T *val, bool coarse) {
  T *pt[6];
  bi_parts(pat, w.part, pt);
  const Mat A = matof(pat);
  hipStream_t S = stream();
  const dim3 B(kBlock), GS(nblk_);
  const int *done = &w.st->done;
  const int mode = pc == PC_JACOBI ? 1 : (pc == PC_DILU ? 2 : 0), c0end = pat->color_ptr[1];
  const Chunks C = coarse ? chunks_of(pat) : Chunks{nullptr, nullptr, nullptr, nblk_};
  if (coarse && co_part_.n < (size_t)C.n) co_part_.alloc(C.n);
  double *csum = coarse ? co_part_.p : nullptr;
  // the grid of the vector launches; the first iteration's partials are k_bi_init's
  const int G0 = std::min((nblk_ + kBlock / kSlice - 1) / (kBlock / kSlice), kCxGrid);
  const dim3 G(G0);
  hipLaunchKernelGGL(k_bi_p<T>, G, B, 0, S, C, n, w.r, w.v, w.p, w.ph, w.dg, mode, c0end, w.st, G0, pt[0], pt[1],
                     csum);
  apply_pc<T>(pc, val, w.fac, w.dg, w.p, w.ph, done, true);
  if (coarse) coarse_apply<T>(w.ph, w.st);
  const bool c16 = c16_of<T>(pat);
  if (c16) hipLaunchKernelGGL((k_bi_spmv_dot<T, 1>), GS, B, 0, S, n, A, val, w.ph, w.r0, w.v, w.st, pt[2]);
  else hipLaunchKernelGGL((k_bi_spmv_dot<T, 0>), GS, B, 0, S, n, A, val, w.ph, w.r0, w.v, w.st, pt[2]);
  const Parts<T> vr = parts_for<T>(G0, nblk_, pt[2], nullptr, w.st);
  hipLaunchKernelGGL(k_bi_s<T>, G, B, 0, S, C, n, w.r, w.v, w.s, w.sh, w.dg, mode, c0end, w.st, vr.n, vr.a, pt[3],
                     csum);
  finish<OpSum, 1>(G0, pt[3], FinBiS{w.st});
  apply_pc<T>(pc, val, w.fac, w.dg, w.s, w.sh, done, true);
  if (coarse) coarse_apply<T>(w.sh, w.st);
  if (c16) hipLaunchKernelGGL((k_bi_spmv_omega<T, 1>), GS, B, 0, S, n, A, val, w.sh, w.s, w.t, w.st, pt[4], pt[5]);
  else hipLaunchKernelGGL((k_bi_spmv_omega<T, 0>), GS, B, 0, S, n, A, val, w.sh, w.s, w.t, w.st, pt[4], pt[5]);
  const Parts<T> tt = parts_for<T>(G0, nblk_, pt[4], pt[5], w.st);
  hipLaunchKernelGGL(k_bi_xr<T>, G, B, 0, S, C, n, w.ph, w.sh, w.s, w.t, w.r0, w.x, w.r, w.st, tt.n, tt.a, tt.b,
                     pt[0], pt[1]);
}

// the state after a chunk: the residual test of its last iteration, and x of a
// solve that ended on |s|
template <class T>
KS Krylov::bi_state(const Bi<T> &w) {
  T *pt[6];
  bi_parts(pat, w.part, pt);
  const int G0 = std::min((nblk_ + kBlock / kSlice - 1) / (kBlock / kSlice), kCxGrid);
  hipLaunchKernelGGL((k_cg_peek<T, false, false>), dim3(1), dim3(kBlock), 0, stream(), w.st, G0, pt[0]);
  MS_CHECK_LAUNCH();
  const KS hs = read_state<T>(w.st);
  if (hs.done == 2) {
    hipLaunchKernelGGL(k_bi_early<T>, dim3(nblk_), dim3(kBlock), 0, stream(), n, w.ph, w.x, w.st);
    MS_CHECK_LAUNCH();
  }
  return hs;
}

SolveResult Krylov::bicgstab(const double *val, const double *b, double *x, double tol, int maxit, PcKind pc,
                             bool coarse) {
  SolveResult R;
  Mat A = matof(pat);
  const dim3 G(nblk_), B(kBlock);
  hipStream_t S = stream();
  KS *st = st_.p;
  double *part = part_.p;
  KS h{};
  h.tol = tol;
  h.maxit = maxit;
  MS_HIP(hipMemcpyAsync(st, &h, sizeof(h), hipMemcpyHostToDevice, S));
  hipLaunchKernelGGL(k_sumsq<double>, G, B, 0, S, n, b, part);
  finish<OpSum, 1>(nblk_, part, FinBnorm{st});
  MS_CHECK_LAUNCH();
  KS hs = read_state<double>(st);
  if (hs.bnrm == 0.0) {
    MS_HIP(hipMemsetAsync(x, 0, n * sizeof(double), S));
    return R;
  }
  last_ = SetupKey{};
  int fe = setup_pc64(pc, val);
  if (fe) {
    R.ierr = fe + 10;
    return R;
  }
  coarse = coarse && pat->coarse.k > 0;
  if (coarse) coarse_setup(val);
  hipLaunchKernelGGL(k_residual<double>, G, B, 0, S, n, A, val, b, x, r_.p, part);
  finish<OpSum, 1>(nblk_, part, FinResidual{st});
  MS_CHECK_LAUNCH();
  hs = read_state<double>(st);
  R.res = hs.res;
  if (hs.done) return R;
  const Bi<double> w{r_.p, r0_.p, p_.p, q_.p, s_.p, t_.p, ph_.p, sh_.p, x, dg_.p, fac_.p, part, st};
  bi_start<double>(w);
  int enq = 0, chunk = 2;
  while (true) {
    int m = std::min(chunk, maxit - enq);
    for (int k = 0; k < m; k++) bi_iteration<double>(w, pc, val, coarse);
    enq += m;
    hs = bi_state<double>(w);
    if (hs.done || enq >= maxit) break;
    chunk = std::min(chunk * 2, 32);
  }
  R.it = hs.it;
  R.res = hs.res;
  R.ierr = hs.ierr;
  if (!hs.done) {        // exhaustion: ierr = 1, it = maxit (mod_uns_linsolver_mpi.f90:224-227)
    R.it = maxit;
    R.ierr = 1;
  }
  return R;
}

// FP32 BiCGSTAB on the scaled residual.  An inner solve whose recursive
// residual has not halved over `window` iterations ends early (the caller's
// refinement restarts it from the FP64 residual).
SolveResult Krylov::bicg32(PcKind pc, int maxit, int window, bool coarse) {
  SolveResult R;
  const Bi<float> w{r32_.p,  r032_.p, p32_.p, q32_.p,  s32_.p,  t32_.p, ph32_.p,
                    sh32_.p, x32_.p,  dg32_.p, fac32_.p, part32_.p, st32_.p};
  bi_start<float>(w);
  int enq = 0, chunk = 4;
  KS hs{};
  double best = HUGE_VAL;
  int it_best = 0;
  while (true) {
    int m = std::min(chunk, maxit - enq);
    for (int k = 0; k < m; k++) bi_iteration<float>(w, pc, val32_.p, coarse);
    enq += m;
    hs = bi_state<float>(w);
    if (hs.done || enq >= maxit) break;
    if (hs.res < 0.5 * best) {
      best = hs.res;
      it_best = enq;
    } else if (enq - it_best >= window) {
      R.stalled = 1;
      break;
    }
    chunk = std::min(chunk * 2, 32);
  }
  R.it = hs.it;
  R.ierr = hs.ierr;
  R.res = hs.res;
  return R;
}

// ---- in-loop SpMV timing ---------------------------------------------------------
// With the probe on, the mixed PCG launches the last FP32 SpMV of every
// 16-iteration chunk through hipExtLaunchKernelGGL with a start / stop event
// pair, which take the kernel's own dispatch timestamps (that iteration is
// enqueued behind the captured graph of the other 15, so it runs back to
// back with them); the pairs are read after each chunk (the host waits for
// the chunk's state anyway).
namespace {
struct SpmvProbe {
  bool on = false;
  std::vector<hipEvent_t> ev;   // a ring of start / stop pairs
  int next = 0;
  long long launches = 0, rows = 0;
  double ms = 0.0;
};
constexpr int kProbePairs = 32;
SpmvProbe g_probe;
void probe_harvest(int pair) {
  float t = 0.f;
  MS_HIP(hipEventSynchronize(g_probe.ev[2 * pair + 1]));
  MS_HIP(hipEventElapsedTime(&t, g_probe.ev[2 * pair], g_probe.ev[2 * pair + 1]));
  g_probe.ms += t;
  g_probe.launches++;
}
}  // namespace

void set_spmv_probe(bool on) {
  if (on && g_probe.ev.empty()) {
    g_probe.ev.resize(2 * kProbePairs);
    for (auto &e : g_probe.ev) MS_HIP(hipEventCreate(&e));
  }
  g_probe.on = on;
  g_probe.next = 0;
  g_probe.launches = g_probe.rows = 0;
  g_probe.ms = 0.0;
}
void read_spmv_probe(long long *launches, double *ms, long long *rows) {
  *launches = g_probe.launches;
  *ms = g_probe.ms;
  *rows = g_probe.rows;
}

// ---- mixed precision ------------------------------------------------------------
static std::atomic<int> g_schur_mf{-1};   // -1: not yet read from the environment
bool schur_matfree_enabled() {
  int v = g_schur_mf.load();
  if (v < 0) {
    const char *e = std::getenv("MIXSOLVER_SCHUR_MF");
    v = (e && e[0] == '0') ? 0 : 1;
    g_schur_mf.store(v);
  }
  return v != 0;
}
void set_schur_matfree(bool on) { g_schur_mf.store(on ? 1 : 0); }
// E^-1 of a coarse space of at most 256 aggregates by one workgroup in FP32
// (MIXSOLVER_COARSE_INV32=1) instead of k / 32 launches over the chip in FP64
// (k_gj_block); off by default: the one workgroup takes longer (21.99 against
// 22.90 PISO steps/s at 2M cells, 256 aggregates)
static bool coarse_inv32_enabled() {
  static const bool on = [] {
    const char *e = std::getenv("MIXSOLVER_COARSE_INV32");
    return e && e[0] == '1';
  }();
  return on;
}
static std::atomic<int> g_p_fused{-1};
bool p_fused_enabled() {
  int v = g_p_fused.load();
  if (v < 0) {
    const char *e = std::getenv("MIXSOLVER_P_FUSED");
    v = (e && e[0] == '1') ? 1 : 0;
    g_p_fused.store(v);
  }
  return v != 0;
}
void set_p_fused(bool on) { g_p_fused.store(on ? 1 : 0); }

static std::atomic<int> g_stall_window{1024};
void set_stall_window(int iters) { g_stall_window.store(iters > 0 ? iters : 1024); }
int stall_window() { return g_stall_window.load(); }

SolveResult Krylov::mixed(const double *val, const double *b, double *x, double tol, int maxit, PcKind pc,
                          int solver, double inner_tol, bool coarse, bool reuse) {
  // a system whose FP32 iteration stalled once is solved in FP64 from then on
  if (fp32_stalled_) {
    SolveResult F = solver == 0 ? pcg(val, b, x, tol, maxit, pc, coarse, reuse)
                                : bicgstab(val, b, x, tol, maxit, pc, coarse);
    F.stalled = 1;
    F.it64 = F.it;
    return F;
  }
  SolveResult R;
  Mat A = matof(pat);
  const dim3 G(nblk_), B(kBlock);
  hipStream_t S = stream();
  ensure32();
  if (val32_.n < (size_t)pat->nstore) val32_.alloc(pat->nstore);
  KS *st = st_.p;
  double *part = part_.p;
  KS h{};
  h.tol = tol;
  h.maxit = maxit;
  h.delta = inner_tol;
  MS_HIP(hipMemcpyAsync(st, &h, sizeof(h), hipMemcpyHostToDevice, S));
  hipLaunchKernelGGL(k_sumsq<double>, G, B, 0, S, n, b, part);
  finish<OpSum, 1>(nblk_, part, FinBnorm{st});
  MS_CHECK_LAUNCH();
  KS hs = read_state<double>(st);
  if (hs.bnrm == 0.0) {
    MS_HIP(hipMemsetAsync(x, 0, n * sizeof(double), S));
    return R;
  }
  coarse = coarse && pat->coarse.k > 0;
  const SetupKey key{val, (int)pc, 1, (int)coarse};
  const bool reused = reuse && last_ == key;
  if (!reused) {
    last_ = SetupKey{};
    hipLaunchKernelGGL(k_mat32_diff, G, B, 0, S, n, A, val, val32_.p);
    setup_pc32(pc, val);
    if (coarse && solver == 1) coarse_setup(val);
  }
  hipLaunchKernelGGL(k_residual<double>, G, B, 0, S, n, A, val, b, x, r_.p, part);
  finish<OpSum, 1>(nblk_, part, FinResidual{st});
  MS_CHECK_LAUNCH();
  hs = read_state<double>(st);
  R.res = hs.res;
  if (hs.done) return R;

  if (solver == 1) {
    // BiCGSTAB: FP32 inner solves inside FP64 iterative refinement.  An
    // inner solve ends at its tolerance or when its residual stops falling
    // (stall window); a refinement pass that does not halve the FP64
    // residual hands the system to FP64 BiCGSTAB (the remaining budget, from
    // the current x), and the system stays in FP64 from then on.
    int total = 0;
    double prev = R.res;
    while (true) {
      int imax = maxit - total;
      hipLaunchKernelGGL(k_mp_scale_down, G, B, 0, S, n, r_.p, st, r32_.p, x32_.p, st32_.p, kRefineTol, imax);
      SolveResult in = bicg32(pc, imax, stall_window(), coarse);
      total += std::max(in.it, 1);
      R.outer++;
      hipLaunchKernelGGL(k_mp_correct, G, B, 0, S, n, x32_.p, st, x);
      hipLaunchKernelGGL(k_residual<double>, G, B, 0, S, n, A, val, b, x, r_.p, part);
      finish<OpSum, 1>(nblk_, part, FinResidual{st});
      MS_CHECK_LAUNCH();
      hs = read_state<double>(st);
      R.res = hs.res;
      if (hs.done || total >= maxit || R.outer >= 200) break;
      if (in.ierr == 2 && in.it <= 1) {
        R.ierr = 2;
        break;
      }
      if (!(hs.res <= 0.5 * prev)) {
        fp32_stalled_ = true;
        const SolveResult F = bicgstab(val, b, x, tol, maxit - total, pc, coarse);
        R.it = total + F.it;
        R.it32 = total;
        R.it64 = F.it;
        R.res = F.res;
        R.ierr = F.ierr;
        R.stalled = 1;
        return R;
      }
      prev = hs.res;
    }
    R.it = total;
    R.it32 = total;
    if (R.ierr == 0 && !(R.res <= tol)) R.ierr = 1;
    return R;
  }

  // PCG with reliable updates: y accumulates alpha p in FP32 between updates.
  // The FP32 iteration pauses when its recursive residual meets the
  // tolerance; a drop below delta times its running maximum only flags an
  // update, which the host applies at the end of the chunk (after the
  // p update: r and p are rescaled, the recurrence continues).
  float *r = r32_.p, *z = z32_.p, *p = p32_.p, *q = q32_.p, *y = x32_.p;
  float *part32 = part32_.p;
  const float *v32 = val32_.p, *dg = dg32_.p, *fac = fac32_.p;
  const int *done = &st->done;
  const int jac = pc == PC_JACOBI;
  const int mode = jac ? 1 : (pc == PC_DILU ? 2 : 0);
  const int c0end = pat->color_ptr[1];
  // DILU with a coarse space: the coarse solve rides along the forward sweep
  const bool fused = coarse && pc == PC_DILU && pat->color_ptr.size() > 2;
  if (coarse) {
    h.coarse = fused ? 0 : 1;
    MS_HIP(hipMemcpyAsync(&st->coarse, &h.coarse, sizeof(int), hipMemcpyHostToDevice, S));
    if (!reused) coarse_setup(val);
  }
  last_ = key;
  const Rows RW = rows_of(pat, coarse);
  const dim3 GR(coarse ? pat->coarse.nchunks : nblk_);
  const CoDev co = codev_of(pat, cm_, coarse && !fused, st);
  const double *nu = coarse ? cm_.nu.p : nullptr;
  float *prz = prz32_.p;
  MS_HIP(hipMemsetAsync(y, 0, n * sizeof(float), S));
  hipLaunchKernelGGL(k_set_sigma, dim3(1), dim3(64), 0, S, st);
  hipLaunchKernelGGL(k_scale_down, G, B, 0, S, n, r_.p, r, st);
  // without a coarse space the two-launch iteration (the matrix-free product
  // has launches of its own)
  const bool two = !coarse && !matfree_on();
  const Cg2<float> cg = two ? cg2<float>(pc) : Cg2<float>{};
  // Jacobi or DILU with a coarse space; on request the p update rides along
  // the next matrix-free product
  const bool with_co = coarse && (fused || mode == 1);
  const bool pfused = with_co && mode == 1 && matfree_on() && mf_->agg1 && p_fused_enabled();
  const PUp pu{r, dg, mf_ ? mf_->agg1 : nullptr, nu};
  const Cx<float> cxf = with_co ? cx<float>(pc) : Cx<float>{};
  if (two) {
    cg2_start<float>(cg, v32, fac);
  } else if (with_co) {
    cx_restart<float, true>(cxf, v32, nullptr, true);
  } else {
    if (coarse) {
      hipLaunchKernelGGL(k_rsum<float>, GR, B, 0, S, RW, r, st, part32);
      finish_co<3>((int)GR.x, part32, FinNop{st}, co);
    }
    if (!jac) apply_pc<float>(pc, v32, fac, dg, r, z, done);
    hipLaunchKernelGGL(k_pcg_start<float>, GR, B, 0, S, RW, r, z, dg, jac, p, nu, st, part32);
    finish<OpSum, 1>((int)GR.x, part32, FinRz0{st});
  }
  // the part of an iteration after the update kernel: residual check,
  // preconditioner, r.z and p update (trigger: reliable-update checks active)
  auto tail = [&](int trigger) {
    finish_co<3>((int)GR.x, part32, FinUpdateRU{st, jac, trigger}, co);
    if (mode == 2) {
      int np = dilu_sweeps<float>(pat, A, v32, dg, r, z, done, prz);
      finish<OpSum, 1>(np, prz, FinRz{st});
    } else if (mode == 0) {
      apply_pc<float>(pc, v32, fac, dg, r, z, done);
      hipLaunchKernelGGL(k_dot<float>, G, B, 0, S, n, r, z, st, part32);
      finish<OpSum, 1>(nblk_, part32, FinRz{st});
    }
    hipLaunchKernelGGL(k_pcg_p<float>, GR, B, 0, S, RW, r, z, dg, jac, p, nu, st);
  };
  auto reliable_update = [&](bool paused) {
    if (two) {   // the p update of the last iteration is always pending here
      hipLaunchKernelGGL(k_fold, G, B, 0, S, n, y, x, st);
      hipLaunchKernelGGL(k_true_res, G, B, 0, S, n, A, val, b, x, r_.p, st, part);
      finish<OpSum, 1>(nblk_, part, FinRU{st});
      hipLaunchKernelGGL(k_cg_rescale, dim3(cg.G), B, 0, S, n, r_.p, r, cg.p0, cg.p1, z, dg, mode, c0end, st, cg.rr,
                         cg.rz);
      cg2_precond<float>(cg, v32, fac);
      MS_CHECK_LAUNCH();
      return;
    }
    if (with_co) {
      if (pfused) {   // apply a pending p update before r and p are rescaled
        cx_p<float, true>(cxf, kCxPending);
        hipLaunchKernelGGL(k_clear_pup, dim3(1), dim3(64), 0, S, st);
      }
      hipLaunchKernelGGL(k_fold, G, B, 0, S, n, y, x, st);
      hipLaunchKernelGGL(k_true_res, G, B, 0, S, n, A, val, b, x, r_.p, st, part);
      finish<OpSum, 1>(nblk_, part, FinRU{st});
      cx_restart<float, true>(cxf, v32, r_.p, paused);   // paused: complete the interrupted iteration on the new r
      return;
    }
    hipLaunchKernelGGL(k_fold, G, B, 0, S, n, y, x, st);
    hipLaunchKernelGGL(k_true_res, G, B, 0, S, n, A, val, b, x, r_.p, st, part);
    finish<OpSum, 1>(nblk_, part, FinRU{st});
    hipLaunchKernelGGL(k_ru_rescale, GR, B, 0, S, RW, r_.p, r, p, z, dg, mode, c0end, st, part32);
    if (paused) tail(0);   // complete the interrupted iteration on the new r
    MS_CHECK_LAUNCH();
  };
  constexpr int kChunk = 16;   // iterations between state reads
  const bool probe = g_probe.on;
  if (probe) g_probe.rows = n;
  int probe_pair = -1;   // the probe pair of the chunk last queued
  float *spart = with_co ? cxf.pq : part32;
  auto chunk = [&](int m, bool probe_last) {
    if (two) {
      for (int it = 0; it < m; it++) {
        hipEvent_t e0 = nullptr, e1 = nullptr;
        if (probe_last && it == m - 1) {
          probe_pair = g_probe.next;
          g_probe.next = (g_probe.next + 1) % kProbePairs;
          e0 = g_probe.ev[2 * probe_pair], e1 = g_probe.ev[2 * probe_pair + 1];
        }
        cg2_iteration<float, true>(cg, v32, fac, y, e0, e1);
      }
      hipLaunchKernelGGL((k_cg_peek<float, true>), dim3(1), B, 0, S, st, cg.G, cg.rr);
      return;
    }
    for (int it = 0; it < m; it++) {
      if (probe_last && it == m - 1) {
        probe_pair = g_probe.next;
        g_probe.next = (g_probe.next + 1) % kProbePairs;
        hipEvent_t e0 = g_probe.ev[2 * probe_pair], e1 = g_probe.ev[2 * probe_pair + 1];
        spmv32(val, v32, p, q, st, spart, e0, e1, pfused ? &pu : nullptr);
      } else {
        spmv32(val, v32, p, q, st, spart, nullptr, nullptr, pfused ? &pu : nullptr);
      }
      if (with_co) {
        cx_update<float, true>(cxf, v32, y, pfused);
        continue;
      }
      finish<OpSum, 1>(nblk_, part32, FinPap{st});
      hipLaunchKernelGGL((k_pcg_update<float, float>), GR, B, 0, S, RW, p, q, y, r, z, dg, mode, c0end, st, part32);
      tail(1);
    }
  };
  hs = read_state<double>(st);
  // Stall guard: when the FP32 recurrence cannot resolve the system (its
  // residual has not halved over kStall iterations), the iteration stops and
  // the FP64 PCG with the same preconditioner continues from the current x.
  // A solve that keeps converging never reaches it, so its result is
  // unchanged.
  const int kStall = stall_window();
  double best = hs.res;
  int it_best = hs.it;
  bool stalled = false;
  // Queue one chunk: the captured graph for a full chunk, else the
  // launches; then its state goes to pinned slot `slot` and an event marks it.
  auto queue_chunk = [&](int m, int slot) {
    probe_pair = -1;
    if (m == kChunk && graphs_enabled()) {
      // every argument of the chunk's launches is fixed by the key (device
      // state lives in st, the iteration count in st->it), so one captured
      // chunk replays for every full chunk of every solve with this set-up;
      // with the probe on, the chunk's last iteration runs after the graph
      const int glen = probe ? kChunk - 1 : kChunk;
      const ChunkKey ck{v32, fac, dg, nu, (int)pc, (int)coarse, (int)fused, glen, (int)matfree_on(), (int)pfused};
      if (!chunk_exec_ || !(chunk_key_ == ck)) {
        std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
        if (chunk_exec_) MS_HIP(hipGraphExecDestroy(chunk_exec_));
        chunk_exec_ = nullptr;
        hipGraph_t g = nullptr;
        MS_HIP(hipStreamBeginCapture(S, hipStreamCaptureModeRelaxed));
        try {
          chunk(glen, false);
        } catch (...) {
          (void)hipStreamEndCapture(S, &g);
          if (g) (void)hipGraphDestroy(g);
          throw;
        }
        MS_HIP(hipStreamEndCapture(S, &g));
        const hipError_t e = hipGraphInstantiate(&chunk_exec_, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) {
          chunk_exec_ = nullptr;
          fail(MS_EDEVICE, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
        }
        chunk_key_ = ck;
      }
      MS_HIP(hipGraphLaunch(chunk_exec_, S));
      if (probe) chunk(1, true);
    } else {
      chunk(m, probe);
    }
    MS_CHECK_LAUNCH();
    MS_HIP(hipMemcpyAsync(state_slot(slot), st, sizeof(KS), hipMemcpyDeviceToHost, S));
    MS_HIP(hipEventRecord(state_ev_[slot], S));
  };
  // Chunks run one ahead of the host: the next chunk is queued before the
  // state after the current one is read, so the device does not idle while
  // the host decides.  A solve that finished or paused makes the queued
  // chunk's kernels return at once; a reliable update flagged in a chunk is
  // applied after the chunk queued behind it (at most 2 x 16 iterations
  // late), as the state then read is the latest.
  struct Queued {
    int slot, m, pair;
  };
  Queued inq[2];
  int nq = 0, next_slot = 0, queued_it = hs.it;
  const bool ahead = pipeline_enabled();
  auto wait_front = [&]() {
    const Queued f = inq[0];
    inq[0] = inq[1];
    nq--;
    MS_HIP(hipEventSynchronize(state_ev_[f.slot]));
    KS h;
    std::memcpy(&h, state_slot(f.slot), sizeof(KS));
    if (f.pair >= 0) probe_harvest(f.pair);
    return h;
  };
  auto drain = [&]() {
    while (nq > 0) hs = wait_front();
  };
  while (true) {
    while (nq < (ahead ? 2 : 1) && queued_it < maxit) {
      const int m = std::min(kChunk, maxit - queued_it);
      queue_chunk(m, next_slot);
      inq[nq++] = Queued{next_slot, m, probe_pair};
      next_slot ^= 1;
      queued_it += m;
    }
    if (nq == 0) break;
    hs = wait_front();
    if (hs.done == 1) {
      drain();
      break;
    }
    if (hs.res < 0.5 * best) {
      best = hs.res;
      it_best = hs.it;
    } else if (hs.it - it_best >= kStall) {
      drain();
      if (hs.done != 1) stalled = true;
      break;
    }
    if (hs.ru == 1) {   // reliable update flagged, or the solve paused for one
      drain();
      if (hs.done == 1) break;
      if (hs.ru == 1) {
        reliable_update(hs.done == 2);
        hs = read_state<double>(st);
      }
      queued_it = hs.it;
      if (hs.done == 1) break;
    }
  }
  if (hs.done != 1) {    // exhaustion: fold y and report the true residual
    KS force = hs;
    force.ru = 1;
    force.done = 0;
    MS_HIP(hipMemcpyAsync(st, &force, sizeof(KS), hipMemcpyHostToDevice, S));
    hipLaunchKernelGGL(k_fold, G, B, 0, S, n, y, x, st);
    hipLaunchKernelGGL(k_true_res, G, B, 0, S, n, A, val, b, x, r_.p, st, part);
    finish<OpSum, 1>(nblk_, part, FinRU{st});
    MS_CHECK_LAUNCH();
    hs = read_state<double>(st);
  }
  R.it = hs.it;
  R.it32 = hs.it;
  R.res = hs.res;
  R.ierr = hs.ierr;
  R.outer = hs.nru;
  if (stalled && !(hs.res <= tol) && hs.it < maxit) {
    fp32_stalled_ = true;
    // the FP64 PCG gets the remaining budget; on exhaustion it reports its
    // budget + 1, so the total is maxit + 1 as for any exhausted CG
    const SolveResult F = pcg(val, b, x, tol, maxit - hs.it, pc, coarse, false);
    R.it += F.it;
    R.it64 = F.it;
    R.res = F.res;
    R.ierr = F.ierr;
    R.stalled = 1;
    return R;
  }
  if (hs.done != 1) {     // exhaustion: it = maxit + 1, as the FP64 CG (Fortran DO-loop count)
    if (R.ierr == 0) R.ierr = 1;
    R.it = maxit + 1;
  }
  return R;
}

}  // namespace ms

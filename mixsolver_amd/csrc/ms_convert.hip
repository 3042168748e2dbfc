// ms_convert.hip -- a caller's CSR matrix into the solvers' SELL-64 form, on
// the device.
//
// The solver entry points take a new matrix on every call, so the conversion
// is part of each solve: on one host thread it took 20 of the 29 ms of a
// PCG-Jacobi solve of 216,000 rows (1.5M entries).  The arrays are copied as
// the caller passes them (1-based), one thread per row checks its row and
// measures its slice, the host turns the slice widths into offsets, and a
// second kernel writes every stored slot: all memory-bound passes of a few
// microseconds behind the copies themselves.
#include <climits>

#include "ms_linalg.hpp"
#include "ms_reduce.hpp"

namespace ms {
namespace {

enum { CE_RANGE = 1, CE_ORDER = 2, CE_DIAG = 4 };   // err bits

// One wavefront per slice.  out: err, then width, lowest and highest
// off-diagonal column of every slice.  A row whose pointers leave [1, nnz + 1]
// is an error and is not read.
__global__ __launch_bounds__(kBlock) void k_csr_check(int n, int nslices, long long nnz, const int *rp, const int *ci,
                                                      int *rowlen, int *diagk, int *out) {
  const int r = blockIdx.x * kBlock + threadIdx.x;
  int len = 0, lo = INT_MAX, hi = -1, err = 0;
  if (r < n) {
    const long long a = (long long)rp[r] - 1, b = (long long)rp[r + 1] - 1;
    int dk = -1;
    if (a < 0 || b < a || b > nnz) {
      err |= CE_RANGE;
    } else {
      len = (int)(b - a);
      int prev = -1;
      for (int k = 0; k < len; k++) {
        const int c = ci[a + k] - 1;
        if (c < 0 || c >= n) err |= CE_RANGE;
        if (k > 0 && c <= prev) err |= CE_ORDER;
        if (c == r) {
          dk = k;
        } else {
          lo = min(lo, c);
          hi = max(hi, c);
        }
        prev = c;
      }
    }
    if (dk < 0) err |= CE_DIAG;
    rowlen[r] = len;
    diagk[r] = dk;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    len = max(len, __shfl_down(len, o, 64));
    lo = min(lo, __shfl_down(lo, o, 64));
    hi = max(hi, __shfl_down(hi, o, 64));
    err |= __shfl_down(err, o, 64);
  }
  const int s = r >> 6;
  if ((threadIdx.x & 63) == 0 && s < nslices) {
    out[1 + s] = len;
    out[1 + nslices + s] = lo;
    out[1 + 2 * nslices + s] = hi;
    if (err) atomicOr(out, err);
  }
}

// Every slot of every slice: column (the row itself for padding, 0 beyond the
// last row), value, 16-bit offset (has16) and transpose slot (tpos not null;
// out[0] = 1 when some entry has no transpose).
__global__ __launch_bounds__(kBlock) void k_csr_fill(int n, int nslices, const int *rp, const int *ci,
                                                     const double *cv, const long long *off, const int *cbase,
                                                     const int *diagk, int *col, double *val, unsigned short *col16,
                                                     long long *tpos, int *asym) {
  const int r = blockIdx.x * kBlock + threadIdx.x, s = r >> 6;
  if (s >= nslices) return;
  const long long o0 = off[s];
  const int w = (int)((off[s + 1] - o0) >> 6);
  const long long base = o0 + (r & 63);
  const long long a = r < n ? (long long)rp[r] - 1 : 0;
  const int len = r < n ? (int)((long long)rp[r + 1] - 1 - a) : 0;
  const int cb = cbase[s];
  for (int k = 0; k < w; k++) {
    const long long q = base + (long long)k * kSlice;
    const int c = k < len ? ci[a + k] - 1 : (r < n ? r : 0);
    col[q] = c;
    val[q] = k < len ? cv[a + k] : 0.0;
    if (col16) col16[q] = c == r || k >= len ? (unsigned short)0xFFFF : (unsigned short)(c - cb);
    if (tpos) {
      long long t = -1;
      if (k < len) {
        long long x = (long long)rp[c] - 1, y = (long long)rp[c + 1] - 1;
        const long long x0 = x, y0 = y;
        while (x < y) {   // first column >= r + 1 (1-based) of row c
          const long long m = (x + y) >> 1;
          if (ci[m] < r + 1) x = m + 1;
          else y = m;
        }
        if (x < y0 && ci[x] == r + 1) t = off[c >> 6] + (x - x0) * kSlice + (c & 63);
        else *asym = 1;
      }
      tpos[q] = t;
    }
  }
}

}  // namespace

// P gets the device arrays of the pattern (its host arrays stay empty but for
// off, cbase and the scalars), val the values in its layout.
void csr_to_device(SellPattern &P, int n, const int *row_ptr, const int *col_idx, const double *v, bool transpose,
                   DBuf<double> &val) {
  const long long nnz = (long long)row_ptr[n] - 1;
  if (nnz < 0) fail(MS_EINVAL, "row_ptr(n+1) must be at least 1");
  hipStream_t S = stream();
  const int ns = (n + kSlice - 1) / kSlice;
  P.n = n;
  P.nslices = ns;
  P.nnz = nnz;
  DBuf<int> rp((size_t)n + 1), ci((size_t)std::max(nnz, 1LL)), out(1 + 3 * (size_t)ns);
  DBuf<double> cv((size_t)std::max(nnz, 1LL));
  P.d_rowlen.alloc(n);
  P.d_diagk.alloc(n);
  rp.upload(row_ptr, (size_t)n + 1);
  ci.upload(col_idx, (size_t)nnz);
  cv.upload(v, (size_t)nnz);
  MS_HIP(hipMemsetAsync(out.p, 0, sizeof(int), S));
  const dim3 G(nblocks((long long)ns * kSlice)), B(kBlock);
  hipLaunchKernelGGL(k_csr_check, G, B, 0, S, n, ns, nnz, rp.p, ci.p, P.d_rowlen.p, P.d_diagk.p, out.p);
  MS_CHECK_LAUNCH();
  std::vector<int> h(1 + 3 * (size_t)ns);
  out.download(h.data(), h.size());
  MS_HIP(hipStreamSynchronize(S));
  if (h[0] & CE_RANGE) fail(MS_EINVAL, "column index out of range");
  if (h[0] & CE_ORDER) fail(MS_EINVAL, "CSR columns must be strictly ascending per row");
  if (h[0] & CE_DIAG) fail(MS_EINVAL, "matrix row without diagonal entry");
  P.off.assign((size_t)ns + 1, 0);
  P.cbase.assign(ns, 0);
  P.has16 = true;   // as csr_to_sell: every slice's off-diagonal columns within one 16-bit window
  for (int s = 0; s < ns; s++) {
    P.off[s + 1] = P.off[s] + (long long)h[1 + s] * kSlice;
    const int lo = h[1 + ns + s], hi = h[1 + 2 * ns + s];
    if (hi < 0) continue;
    P.cbase[s] = lo;
    if (hi - lo > 0xFFFD) P.has16 = false;
  }
  P.nstore = P.off[ns];
  P.nfar = 0;
  P.color_ptr = {0, n};
  P.d_off.upload(P.off);
  P.d_cbase.upload(P.cbase);
  P.d_col.alloc(P.nstore);
  if (P.has16) P.d_col16.alloc(P.nstore);
  if (transpose) P.d_tpos.alloc(P.nstore);
  val.alloc(P.nstore);
  MS_HIP(hipMemsetAsync(out.p, 0, sizeof(int), S));
  hipLaunchKernelGGL(k_csr_fill, G, B, 0, S, n, ns, rp.p, ci.p, cv.p, P.d_off.p, P.d_cbase.p, P.d_diagk.p, P.d_col.p,
                     val.p, P.has16 ? P.d_col16.p : nullptr, transpose ? P.d_tpos.p : nullptr, out.p);
  MS_CHECK_LAUNCH();
  P.symmetric = true;
  if (transpose) {
    out.download(h.data(), 1);
    MS_HIP(hipStreamSynchronize(S));
    P.symmetric = h[0] == 0;
  } else {
    MS_HIP(hipStreamSynchronize(S));   // the staging arrays are freed here
  }
}

}  // namespace ms

// ms_io.hip -- fields and matrices across the API boundary: the caller's
// natural order on one side, the device numbering on the other.
//
// The reordering runs on the device, in the order of the caller's array, and
// the copy goes straight between the caller's memory and a staging buffer.
// On the host it was one random access per value on one thread, beside a
// temporary copy: a 2M-cell velocity field took 15 ms to set and 20 ms to
// get, now 1.7 and 4.8 ms, of which the copy over PCIe is most.
//
// The staging buffer is the face coefficient array af, which every driver and
// per-call routine forms before it reads it, so it is free between calls and
// no device memory is held for this.
#include "ms_system.hpp"

namespace ms {
namespace {

__global__ void k_get_cells(long long m, long long e0, int w, const int *o2n, const double *src, double *dst) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (t >= m) return;
  const long long e = e0 + t, i = e / w;
  dst[t] = src[(long long)o2n[i] * w + (e - i * w)];
}
__global__ void k_set_cells(long long m, long long e0, int w, const int *o2n, const double *src, double *dst) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (t >= m) return;
  const long long e = e0 + t, i = e / w;
  dst[(long long)o2n[i] * w + (e - i * w)] = src[t];
}
// idx >= 0: device face; ~idx: the device face with the sign turned (shadows)
__global__ void k_get_faces(long long m, const int *idx, const double *src, double *dst) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (t >= m) return;
  const int f = idx[t];
  dst[t] = f >= 0 ? src[f] : -src[~f];
}
__global__ void k_set_faces(long long m, const int *idx, const double *src, double *dst) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (t < m) dst[idx[t]] = src[t];
}
__global__ void k_get_slots(long long m, const long long *slot, const double *src, double *dst) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (t < m) dst[t] = src[slot[t]];
}

// the caller's n values in pieces of the staging buffer's size
template <class Get>
void pieces_out(System &s, long long n, double *h, Get get) {
  const long long step = (long long)s.af.n;
  for (long long e0 = 0; e0 < n; e0 += step) {
    const long long m = std::min(step, n - e0);
    get(e0, m);
    MS_CHECK_LAUNCH();
    MS_HIP(hipMemcpyAsync(h + e0, s.af.p, m * sizeof(double), hipMemcpyDeviceToHost, stream()));
    MS_HIP(hipStreamSynchronize(stream()));
  }
}
template <class Set>
void pieces_in(System &s, long long n, const double *h, Set set) {
  const long long step = (long long)s.af.n;
  for (long long e0 = 0; e0 < n; e0 += step) {
    const long long m = std::min(step, n - e0);
    MS_HIP(hipMemcpyAsync(s.af.p, h + e0, m * sizeof(double), hipMemcpyHostToDevice, stream()));
    set(e0, m);
    MS_CHECK_LAUNCH();
    MS_HIP(hipStreamSynchronize(stream()));
  }
}
dim3 grid(long long m) { return dim3((unsigned)((m + kBlock - 1) / kBlock)); }

}  // namespace

// cell array of w values per cell, device order, to and from natural order; a
// forked system uses its base's numbering
void cells_out(System &s, const DBuf<double> &buf, int w, double *h) {
  const System &t = s.base ? *s.base : s;
  const long long n = (long long)s.nc * w;
  if (buf.n < (size_t)n) fail(MS_EINVAL, "internal: cell array not allocated");
  const double *dev = buf.p;
  if (!s.renumbered) {
    MS_HIP(hipMemcpyAsync(h, dev, n * sizeof(double), hipMemcpyDeviceToHost, stream()));
    MS_HIP(hipStreamSynchronize(stream()));
    return;
  }
  pieces_out(s, n, h, [&](long long e0, long long m) {
    hipLaunchKernelGGL(k_get_cells, grid(m), dim3(kBlock), 0, stream(), m, e0, w, t.d_o2n.p, dev, s.af.p);
  });
}
void cells_in(System &s, const double *h, int w, DBuf<double> &buf) {
  const System &t = s.base ? *s.base : s;
  const long long n = (long long)s.nc * w;
  if (buf.n < (size_t)n) buf.alloc(n);   // zone properties get their arrays when they are set
  double *dev = buf.p;
  if (!s.renumbered) {
    MS_HIP(hipMemcpyAsync(dev, h, n * sizeof(double), hipMemcpyHostToDevice, stream()));
    MS_HIP(hipStreamSynchronize(stream()));
    return;
  }
  pieces_in(s, n, h, [&](long long e0, long long m) {
    hipLaunchKernelGGL(k_set_cells, grid(m), dim3(kBlock), 0, stream(), m, e0, w, t.d_o2n.p, s.af.p, dev);
  });
}

// face array, device face order, to and from face order; on the way out a
// periodic shadow face carries its joined face's value, oriented out of its
// own cell
void faces_out(System &s, const DBuf<double> &buf, double *h) {
  if (buf.n < (size_t)s.nf) fail(MS_EINVAL, "internal: face array not allocated");
  const double *dev = buf.p;
  if (!s.d_face_get.n) {
    std::vector<int> idx(s.nf);
    for (int g = 0; g < s.nf; g++) idx[g] = s.shadow[g] >= 0 ? ~s.fo2d[s.shadow[g]] : s.fo2d[g];
    s.d_face_get.upload(idx);
    MS_HIP(hipStreamSynchronize(stream()));
  }
  pieces_out(s, s.nf, h, [&](long long e0, long long m) {
    hipLaunchKernelGGL(k_get_faces, grid(m), dim3(kBlock), 0, stream(), m, s.d_face_get.p + e0, dev, s.af.p);
  });
}
void faces_in(System &s, const double *h, DBuf<double> &buf) {
  if (buf.n < (size_t)s.nf) buf.alloc(s.nf);
  double *dev = buf.p;
  if (!s.d_fo2d.n) s.d_fo2d.upload(s.fo2d);
  pieces_in(s, s.nf, h, [&](long long e0, long long m) {
    hipLaunchKernelGGL(k_set_faces, grid(m), dim3(kBlock), 0, stream(), m, s.d_fo2d.p + e0, s.af.p, dev);
  });
}

// the matrix in the caller's CSR order
void matrix_values_out(System &s, double *h) {
  if (!s.d_ref2dev.n) s.d_ref2dev.upload(s.ref2dev);
  pieces_out(s, (long long)s.ref2dev.size(), h, [&](long long e0, long long m) {
    hipLaunchKernelGGL(k_get_slots, grid(m), dim3(kBlock), 0, stream(), m, s.d_ref2dev.p + e0, s.val.p, s.af.p);
  });
}

}  // namespace ms

// ms_io.hip -- fields and matrices across the API boundary: the caller's
// natural order on one side, the device numbering on the other.
//
// The reordering runs on the device, in the order of the caller's array, and
// the copy goes straight between the caller's memory and a staging buffer.
// On the host it was one random access per value on one thread, beside a
// temporary copy: a 2M-cell velocity field took 15 ms to set and 20 ms to
// get, now 1.7 and 4.8 ms, of which the copy over PCIe is most.
//
// A launch takes longer than the host needs for some ten thousand values, so
// small arrays are reordered on the host, as are all when the device has no
// memory left for staging.  Microseconds per call, host / device: reading 945
// values 23 / 24, 3,025 12 / 25, 9,600 16 / 27, 28,800 25 / 33, 75,000 49 / 48;
// setting 3,025 values 12 / 22, 9,600 15 / 24, 28,800 22 / 28, 75,000 43 / 41;
// 79,000 faces 72 / 48 and 52 / 42.
//
// Every transfer has a staging buffer of its own, from a small pool, so a
// thread that reads fields while another runs the solver, or reads other
// fields, takes nothing of theirs.  The face and matrix maps are held by the
// system from their first use (4 bytes per face and direction, 8 per nonzero).
#include <mutex>
#include <type_traits>

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

// A device buffer of kStageValues, from the idle ones or new (p null: no memory).  It goes back
// with keep(), once its work has been waited for; a transfer that fails frees
// it instead, which waits for the device.  At most kIdleStages are kept (64
// MB).  Never part of a thread's slab, which ends with its owner.
constexpr long long kStageValues = 1 << 21;
constexpr long long kHostValues = 32768;   // largest arrays reordered on the host
constexpr size_t kIdleStages = 4;
std::mutex g_stage_mu;
std::vector<std::pair<int, double *>> g_idle_stages;   // (device, buffer)
class Stage {
 public:
  Stage() : dev_(runtime_device()) {
    MS_HIP(hipSetDevice(dev_));   // a reader's thread may not have chosen the library's device
    {
      std::lock_guard<std::mutex> g(g_stage_mu);
      for (size_t i = 0; i < g_idle_stages.size(); i++)
        if (g_idle_stages[i].first == dev_) {
          p = g_idle_stages[i].second;
          g_idle_stages.erase(g_idle_stages.begin() + i);
          return;
        }
    }
    std::lock_guard<std::recursive_mutex> g(device_alloc_mutex());
    if (hipMalloc(&p, kStageValues * sizeof(double)) != hipSuccess) {
      p = nullptr;
      (void)hipGetLastError();
    }
  }
  Stage(const Stage &) = delete;
  Stage &operator=(const Stage &) = delete;
  void keep() {
    std::lock_guard<std::mutex> g(g_stage_mu);
    if (g_idle_stages.size() >= kIdleStages) return;
    g_idle_stages.push_back({dev_, p});
    p = nullptr;
  }
  ~Stage() {
    if (!p) return;
    std::lock_guard<std::recursive_mutex> g(device_alloc_mutex());
    (void)hipFree(p);
  }
  double *p = nullptr;

 private:
  int dev_;
};

// the caller's n values in pieces of the staging buffer's size; false: no
// staging buffer, nothing done
template <class Get>
bool pieces_out(long long n, double *h, Get get) {
  const auto lk = library_stream_lock();
  Stage st;
  if (!st.p) return false;
  for (long long e0 = 0; e0 < n; e0 += kStageValues) {
    const long long m = std::min(kStageValues, n - e0);
    get(e0, m, st.p);
    MS_CHECK_LAUNCH();
    MS_HIP(hipMemcpyAsync(h + e0, st.p, m * sizeof(double), hipMemcpyDeviceToHost, stream()));
    MS_HIP(hipStreamSynchronize(stream()));
  }
  st.keep();
  return true;
}
template <class Set>
bool pieces_in(long long n, const double *h, Set set) {
  const auto lk = library_stream_lock();
  Stage st;
  if (!st.p) return false;
  for (long long e0 = 0; e0 < n; e0 += kStageValues) {
    const long long m = std::min(kStageValues, n - e0);
    MS_HIP(hipMemcpyAsync(st.p, h + e0, m * sizeof(double), hipMemcpyHostToDevice, stream()));
    set(e0, m, st.p);
    MS_CHECK_LAUNCH();
    MS_HIP(hipStreamSynchronize(stream()));
  }
  st.keep();
  return true;
}
// the device copy of a map, made on its first use (null: no memory for it); calls on one system may come from several threads
template <class T, class Host>
const T *map_on_device(System &s, DBuf<T> &d, Host host) {
  std::lock_guard<std::mutex> g(s.map_mu);
  if (!d.n) {
    const std::vector<T> &h = host();
    const auto lk = library_stream_lock();
    MS_HIP(hipSetDevice(runtime_device()));
    DBuf<T> t;
    try {
      t.alloc(h.size());
    } catch (const Error &) {
      (void)hipGetLastError();
      return nullptr;
    }
    t.upload(h);
    MS_HIP(hipStreamSynchronize(stream()));
    d = std::move(t);
  }
  return d.p;
}
// the host's route: the whole array as it is on the device
template <class Put>
void host_out(const double *dev, size_t n, Put put) {
  std::vector<double> d(n);
  {
    const auto lk = library_stream_lock();
    MS_HIP(hipMemcpyAsync(d.data(), dev, n * sizeof(double), hipMemcpyDeviceToHost, stream()));
    MS_HIP(hipStreamSynchronize(stream()));
  }
  put(d.data());
}
template <class Fill>
void host_in(double *dev, size_t n, Fill fill) {
  std::vector<double> d(n);
  fill(d.data());
  const auto lk = library_stream_lock();
  MS_HIP(hipMemcpyAsync(dev, d.data(), n * sizeof(double), hipMemcpyHostToDevice, stream()));
  MS_HIP(hipStreamSynchronize(stream()));
}
// values per cell as a constant
template <class F>
void by_width(int w, F f) {
  if (w == 1) f(std::integral_constant<int, 1>{});
  else if (w == 3) f(std::integral_constant<int, 3>{});
  else if (w == 9) f(std::integral_constant<int, 9>{});
  else fail(MS_EINVAL, "internal: values per cell");
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
    const auto lk = library_stream_lock();
    MS_HIP(hipMemcpyAsync(h, dev, n * sizeof(double), hipMemcpyDeviceToHost, stream()));
    MS_HIP(hipStreamSynchronize(stream()));
    return;
  }
  if (n > kHostValues && pieces_out(n, h, [&](long long e0, long long m, double *stage) {
        hipLaunchKernelGGL(k_get_cells, grid(m), dim3(kBlock), 0, stream(), m, e0, w, t.d_o2n.p, dev, stage);
      }))
    return;
  host_out(dev, n, [&](const double *d) {
    by_width(w, [=, o2n = t.o2n.data(), nc = s.nc](auto W) {
      for (int i = 0; i < nc; i++)
        for (int j = 0; j < W; j++) h[(size_t)i * W + j] = d[(size_t)o2n[i] * W + j];
    });
  });
}
void cells_in(System &s, const double *h, int w, DBuf<double> &buf) {
  const System &t = s.base ? *s.base : s;
  const long long n = (long long)s.nc * w;
  if (buf.n < (size_t)n) buf.alloc(n);   // zone properties get their arrays when they are set
  double *dev = buf.p;
  if (!s.renumbered) {
    const auto lk = library_stream_lock();
    MS_HIP(hipMemcpyAsync(dev, h, n * sizeof(double), hipMemcpyHostToDevice, stream()));
    MS_HIP(hipStreamSynchronize(stream()));
    return;
  }
  if (n > kHostValues && pieces_in(n, h, [&](long long e0, long long m, const double *stage) {
        hipLaunchKernelGGL(k_set_cells, grid(m), dim3(kBlock), 0, stream(), m, e0, w, t.d_o2n.p, stage, dev);
      }))
    return;
  host_in(dev, n, [&](double *d) {
    by_width(w, [=, o2n = t.o2n.data(), nc = s.nc](auto W) {
      for (int i = 0; i < nc; i++)
        for (int j = 0; j < W; j++) d[(size_t)o2n[i] * W + j] = h[(size_t)i * W + j];
    });
  });
}

// face array, device face order, to and from face order; on the way out a
// periodic shadow face carries its joined face's value, oriented out of its
// own cell
void faces_out(System &s, const DBuf<double> &buf, double *h) {
  if (buf.n < (size_t)s.nf) fail(MS_EINVAL, "internal: face array not allocated");
  const double *dev = buf.p;
  auto place = [&](int g) { return s.shadow[g] >= 0 ? ~s.fo2d[s.shadow[g]] : s.fo2d[g]; };
  const int *map = s.nf <= kHostValues ? nullptr : map_on_device(s, s.d_face_get, [&] {
    std::vector<int> idx(s.nf);
    for (int g = 0; g < s.nf; g++) idx[g] = place(g);
    return idx;
  });
  if (map && pieces_out(s.nf, h, [&](long long e0, long long m, double *stage) {
        hipLaunchKernelGGL(k_get_faces, grid(m), dim3(kBlock), 0, stream(), m, map + e0, dev, stage);
      }))
    return;
  host_out(dev, s.nf, [&](const double *d) {
    for (int g = 0; g < s.nf; g++) {
      const int f = place(g);
      h[g] = f >= 0 ? d[f] : -d[~f];
    }
  });
}
void faces_in(System &s, const double *h, DBuf<double> &buf) {
  if (buf.n < (size_t)s.nf) buf.alloc(s.nf);
  double *dev = buf.p;
  const int *map = s.nf <= kHostValues ? nullptr : map_on_device(s, s.d_fo2d, [&]() -> const std::vector<int> & {
    return s.fo2d;
  });
  if (map && pieces_in(s.nf, h, [&](long long e0, long long m, const double *stage) {
        hipLaunchKernelGGL(k_set_faces, grid(m), dim3(kBlock), 0, stream(), m, map + e0, stage, dev);
      }))
    return;
  host_in(dev, s.nf, [&](double *d) {
    for (int g = 0; g < s.nf; g++) d[s.fo2d[g]] = h[g];
  });
}

// the matrix in the caller's CSR order
void matrix_values_out(System &s, double *h) {
  const long long n = (long long)s.ref2dev.size();
  const long long *map = n <= kHostValues ? nullptr : map_on_device(s, s.d_ref2dev, [&]() -> const std::vector<long long> & {
    return s.ref2dev;
  });
  if (map && pieces_out(n, h, [&](long long e0, long long m, double *stage) {
        hipLaunchKernelGGL(k_get_slots, grid(m), dim3(kBlock), 0, stream(), m, map + e0, s.val.p, stage);
      }))
    return;
  host_out(s.val.p, s.pat.nstore, [&](const double *d) {
    for (long long k = 0; k < n; k++) h[k] = d[s.ref2dev[k]];
  });
}

}  // namespace ms

// sac_xfer.hip -- states between host memory and the device (sac_xfer.h).
//
// The host keeps unpadded arrays in ordinary memory, the device padded rows.
// A 2-D copy between the two (hipMemcpy2D) moved row after row through the
// runtime's own staging, about 9 us a row: 8.0 s up and 6.1 s down for a
// 256^3 state of 1.85 GB, 0.16 and 0.11 s for 32^3.  Here the state goes in
// chunks: a kernel reads or writes the padded rows and a pinned buffer in the
// host's order (over the bus, coalesced), and a few host threads, each with a
// buffer of its own, copy between the buffers and the caller's array while
// the other chunks move.  One thread alone fills fresh pages at 2.7 GB/s, the
// bus takes 57.  Now 36 ms up and 37 ms down for the 256^3 state, 0.4 and 0.5 ms for
// 31x27x35 (0.16 and 0.11 s before), 12 ms for the states of 4096 tubes (150).
#include "sac_xfer.h"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

namespace sac {
namespace xfer {

namespace {

constexpr int kWorkers = 8;
constexpr size_t kChunk = size_t(4) << 20;  // bytes of a pinned buffer

// n elements in host order from element x0 of row R0 on (rows of all fields
// counted through), between padded rows and contiguous memory
template <typename T, bool OUT>
__global__ void __launch_bounds__(256) k_rows(T* dev, T* flat, unsigned n, unsigned x0, unsigned R0,
                                              unsigned G0, unsigned rows, long long pitch,
                                              long long fs) {
  const unsigned i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const unsigned r = (x0 + i) / G0, x = x0 + i - r * G0;
  const unsigned R = R0 + r, f = R / rows;
  T* p = dev + (long long)f * fs + (long long)(R - f * rows) * pitch + x;
  if (OUT)
    flat[i] = *p;
  else
    *p = flat[i];
}

template <bool OUT>
hipError_t launch_rows(const GridDesc& g, const Fields& f, long long first, unsigned n, void* flat,
                 hipStream_t st) {
  const unsigned G0 = (unsigned)g.G[0], rows = (unsigned)g.G[1] * (unsigned)g.G[2];
  const unsigned R0 = (unsigned)(first / G0), x0 = (unsigned)(first % G0);
  const dim3 nb((n + 255) / 256), bs(256);
  if (f.esz == 8)
    return launch(k_rows<uint64_t, OUT>, nb, bs, st, (uint64_t*)f.dev, (uint64_t*)flat, n, x0, R0,
                  G0, rows, g.st[1], g.fs);
  return launch(k_rows<uint32_t, OUT>, nb, bs, st, (uint32_t*)f.dev, (uint32_t*)flat, n, x0, R0, G0,
                rows, g.st[1], g.fs);
}

// fn(begin, end) on slices of [0, n), on several threads where it pays
template <typename F>
void parallel_slices(size_t n, size_t per_thread, const F& fn) {
  const size_t hw = std::max(1u, std::thread::hardware_concurrency());
  const size_t nt = std::min<size_t>({(size_t)kWorkers, hw, n / per_thread + 1});
  std::vector<std::thread> th;
  auto slice = [&](size_t t) { fn(n * t / nt, n * (t + 1) / nt); };
  size_t t = 1;
  try {
    th.reserve(nt);
    for (; t < nt; t++) th.emplace_back(slice, t);
  } catch (const std::exception&) {  // no more threads, or memory for them: the rest here
  }
  slice(0);
  for (; t < nt; t++) slice(t);
  for (auto& x : th) x.join();
}

// between the host's FP64 and a buffer of elements of esz bytes
void from_pinned(double* h, const void* pin, int esz, size_t m) {
  if (esz == 8) {
    memcpy(h, pin, sizeof(double) * m);
  } else {
    const float* p = (const float*)pin;
    for (size_t i = 0; i < m; i++) h[i] = (double)p[i];
  }
}
void to_pinned(void* pin, const double* h, int esz, size_t m) {
  if (esz == 8) {
    memcpy(pin, h, sizeof(double) * m);
  } else {
    float* p = (float*)pin;
    for (size_t i = 0; i < m; i++) p[i] = (float)h[i];
  }
}

int hip_err(hipError_t e, const char* what, std::string& err) {
  if (e == hipSuccess) return 0;
  err = std::string(what) + ": " + hipGetErrorString(e);
  return SAC_E_HIP;
}

}  // namespace

void host_copy(double* dst, const double* src, size_t n) {
  parallel_slices(n, size_t(1) << 18, [&](size_t b, size_t e) {
    memcpy(dst + b, src + b, sizeof(double) * (e - b));
  });
}

void host_copy(double* dst, const float* src, size_t n) {
  parallel_slices(n, size_t(1) << 18, [&](size_t b, size_t e) {
    for (size_t i = b; i < e; i++) dst[i] = (double)src[i];
  });
}

static int run_chunks(int device, long long n, size_t bytes, const ChunkFn& fn,
                      std::string& err) {
  const long long hw = std::max(1u, std::thread::hardware_concurrency());
  const int nt = (int)std::min<long long>({(long long)kWorkers, hw, n});
  std::vector<std::string> errs((size_t)nt);
  std::vector<int> rcs((size_t)nt, 0);
  std::atomic<long long> next{0};
  std::atomic<bool> stop{false};
  auto work = [&](int t) {
    void* pin = nullptr;
    hipEvent_t ev = nullptr;
    int rc = hip_err(hipSetDevice(device), "hipSetDevice", errs[t]);
    if (!rc && hipHostMalloc(&pin, bytes, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      return;  // the other threads take the chunks
    }
    if (!rc) rc = hip_err(hipEventCreateWithFlags(&ev, hipEventDisableTiming), "hipEventCreate", errs[t]);
    while (!rc && !stop) {
      const long long c = next.fetch_add(1);
      if (c >= n) break;
      rc = guarded(errs[t], [&] { return fn(c, pin, ev, errs[t]); });
    }
    // the buffer's last chunk may still be on its way to the device
    if (ev) {
      const int e = hip_err(hipEventSynchronize(ev), "hipEventSynchronize", errs[t]);
      if (!rc) rc = e;
      hipEventDestroy(ev);
    }
    if (pin) hipHostFree(pin);
    if (rc) stop = true;
    rcs[t] = rc;
  };
  auto worker = [&](int t) {
    if (int rc = guarded(errs[t], [&] { return work(t), 0; })) {
      rcs[t] = rc;
      stop = true;
    }
  };
  std::vector<std::thread> th;
  try {
    th.reserve((size_t)nt);
    for (int t = 1; t < nt; t++) th.emplace_back(worker, t);
  } catch (const std::exception&) {  // the threads there are take the chunks
  }
  // this thread is the caller's: its current device comes back
  int current = device;
  const bool known = hipGetDevice(&current) == hipSuccess;
  worker(0);
  if (known && current != device) (void)hipSetDevice(current);
  for (auto& x : th) x.join();
  for (int t = 0; t < nt; t++)
    if (rcs[t]) {
      err = errs[t];
      return rcs[t];
    }
  return next ? 0 : kNoPinned;  // a thread with a buffer takes chunks until there are none
}

int for_chunks(int device, long long n, size_t bytes, const ChunkFn& fn, std::string& err) {
  if (n <= 0) return 0;
  return guarded(err, [&] { return run_chunks(device, n, bytes, fn, err); });
}

// Without pinned memory: field by field with the runtime's own copies of rows,
// FP32 elements by way of a buffer
static int copy_plain(const GridDesc& g, hipStream_t stream, const Fields* f, int n, bool to_host,
                      std::string& err) {
  const size_t ncell = (size_t)g.G[0] * g.G[1] * g.G[2], rows = (size_t)g.G[1] * g.G[2];
  std::vector<float> tmp;
  for (int k = 0; k < n; k++) {
    const size_t esz = (size_t)f[k].esz, w = esz * g.G[0], pitch = esz * (size_t)g.st[1];
    for (int v = 0; v < f[k].nfield; v++) {
      double* h = f[k].host + v * ncell;
      char* dev = (char*)f[k].dev + esz * (size_t)v * g.fs;
      if (esz == 4) tmp.resize(ncell);
      void* flat = esz == 4 ? (void*)tmp.data() : (void*)h;
      if (!to_host && esz == 4) to_pinned(flat, h, 4, ncell);
      hipError_t e = to_host ? hipMemcpy2DAsync(flat, w, dev, pitch, w, rows, hipMemcpyDeviceToHost, stream)
                             : hipMemcpy2DAsync(dev, pitch, flat, w, w, rows, hipMemcpyHostToDevice, stream);
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
      if (int rc = hip_err(e, "copy", err)) return rc;
      if (to_host && esz == 4) from_pinned(h, flat, 4, ncell);
    }
  }
  return 0;
}

// a copy that fits one buffer: all groups' kernels, one wait (a tube of
// 800 cells: 20 us each way, 180 with a thread and a buffer of its own)
static int copy_small(const GridDesc& g, hipStream_t stream, const Fields* f, int n, bool to_host,
                      void** small, std::string& err) {
  const size_t ncell = (size_t)g.G[0] * g.G[1] * g.G[2];
  if (!*small && hipHostMalloc(small, kSmall, hipHostMallocDefault) != hipSuccess) {
    *small = nullptr;
    (void)hipGetLastError();
    return copy_plain(g, stream, f, n, to_host, err);
  }
  size_t at = 0;
  int rc = 0;
  for (int k = 0; k < n && !rc; k++) {
    const size_t m = ncell * f[k].nfield;
    char* p = (char*)*small + at;
    if (!to_host) to_pinned(p, f[k].host, f[k].esz, m);
    rc = hip_err(to_host ? launch_rows<true>(g, f[k], 0, (unsigned)m, p, stream)
                         : launch_rows<false>(g, f[k], 0, (unsigned)m, p, stream),
                 "copy kernel", err);
    at += (m * f[k].esz + 15) / 16 * 16;
  }
  const int e = hip_err(hipStreamSynchronize(stream), "copy", err);
  if (rc || e) return rc ? rc : e;
  at = 0;
  for (int k = 0; k < n && to_host; k++) {
    const size_t m = ncell * f[k].nfield;
    from_pinned(f[k].host, (char*)*small + at, f[k].esz, m);
    at += (m * f[k].esz + 15) / 16 * 16;
  }
  return 0;
}

static int copy_any(const GridDesc& g, int device, hipStream_t stream, const Fields* f, int n,
                    bool to_host, void** small, std::string& err) {
  const long long ncell = (long long)g.G[0] * g.G[1] * g.G[2];
  size_t all = 0;
  for (int k = 0; k < n; k++) all += (size_t)ncell * f[k].nfield * f[k].esz + 16;
  if (small && all <= kSmall) return copy_small(g, stream, f, n, to_host, small, err);
  // chunks of each group, one after another
  std::vector<long long> first((size_t)n + 1, 0);
  size_t bytes = 0;
  for (int k = 0; k < n; k++) {
    const long long total = ncell * f[k].nfield, per = (long long)(kChunk / f[k].esz);
    first[k + 1] = first[k] + (total + per - 1) / per;
    bytes = std::max(bytes, (size_t)std::min(total, per) * f[k].esz);
  }
  auto fn = [&](long long c, void* pin, hipEvent_t ev, std::string& e) -> int {
    const int k = (int)(std::upper_bound(first.begin(), first.end(), c) - first.begin()) - 1;
    const Fields& s = f[k];
    const long long per = (long long)(kChunk / s.esz), lo = (c - first[k]) * per;
    const unsigned m = (unsigned)std::min(per, ncell * s.nfield - lo);
    double* h = s.host + lo;
    if (to_host) {
      if (int rc = hip_err(launch_rows<true>(g, s, lo, m, pin, stream), "copy kernel", e)) return rc;
      if (int rc = hip_err(hipEventRecord(ev, stream), "hipEventRecord", e)) return rc;
      if (int rc = hip_err(hipEventSynchronize(ev), "download", e)) return rc;
      from_pinned(h, pin, s.esz, m);
      return 0;
    }
    // the buffer is free once its previous chunk has been read
    if (int rc = hip_err(hipEventSynchronize(ev), "upload", e)) return rc;
    to_pinned(pin, h, s.esz, m);
    if (int rc = hip_err(launch_rows<false>(g, s, lo, m, pin, stream), "copy kernel", e)) return rc;
    return hip_err(hipEventRecord(ev, stream), "hipEventRecord", e);
  };
  const int rc = for_chunks(device, first[n], bytes, fn, err);
  return rc == kNoPinned ? copy_plain(g, stream, f, n, to_host, err) : rc;
}

int copy(const GridDesc& g, int device, hipStream_t stream, const Fields* f, int n, bool to_host,
         void** small, std::string& err) {
  return guarded(err, [&] { return copy_any(g, device, stream, f, n, to_host, small, err); });
}

hipError_t launch_pack(const GridDesc& g, const Fields& f, void* out, hipStream_t stream) {
  const long long ncell = (long long)g.G[0] * g.G[1] * g.G[2], total = ncell * f.nfield;
  const long long per = 1LL << 30;  // elements of a launch (32-bit thread numbers)
  hipError_t e = hipSuccess;
  for (long long lo = 0; lo < total && e == hipSuccess; lo += per)
    e = launch_rows<true>(g, f, lo, (unsigned)std::min(per, total - lo), (char*)out + lo * f.esz,
                          stream);
  return e;
}

}  // namespace xfer
}  // namespace sac

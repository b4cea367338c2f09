// sac_xfer.h -- states between host memory and the device (uploads,
// downloads, saves): kernels that pack padded device rows to the host's
// layout, pinned buffers, and host threads that copy.
#pragma once
#include <algorithm>
#include <exception>
#include <functional>
#include <string>
#include <tuple>

#include "../../include/sac_amd.h"
#include "sac_common.h"

namespace sac {
namespace xfer {

// `nfield` fields of a grid: on the device in elements of esz bytes (4 or 8)
// with padded rows (dev: element (0,0,0) of the first field), on the host
// (host) in FP64, unpadded, one field after another.
struct Fields {
  void* dev;
  int esz;
  int nfield;
  double* host;
};

// Copy n groups of fields of grid g to the host or to the device, on
// `stream`; returns when the copy is done.  0, or a SAC_E_* code with the
// message in err.  small: a pinned buffer of kSmall bytes for copies that fit
// in it, of one caller at a time, or null (allocated on first use; the caller
// frees it with hipHostFree).  Where there is no pinned memory the rows are
// copied from and to ordinary memory.
constexpr size_t kSmall = size_t(1) << 19;
int copy(const GridDesc& g, int device, hipStream_t stream, const Fields* f, int n, bool to_host,
         void** small, std::string& err);

// f() with what it throws made an error: nothing may leave a C entry point
template <typename F>
int guarded(std::string& err, const F& f) {
  try {
    return f();
  } catch (const std::exception&) {
    err = "no host memory";  // short enough for a string without memory of its own
    return SAC_E_NOMEM;
  }
}

// Launch a kernel and return this launch's own error.  The last error that the
// runtime keeps is one per thread, so that of a worker is not seen by the
// caller, and it may be one that another call left there.
template <typename... P, typename... A>
hipError_t launch(void (*kernel)(P...), dim3 grid, dim3 block, hipStream_t st, A... a) {
  std::tuple<P...> p(a...);
  void* args[sizeof...(P)];
  std::apply([&](P&... x) {
    void* v[] = {&x...};
    std::copy(v, v + sizeof...(P), args);
  }, p);
  const hipError_t e = hipLaunchKernel((const void*)kernel, grid, block, args, 0, st);
  if (e != hipSuccess) (void)hipGetLastError();  // the caller gets it
  return e;
}

// pack the fields of f (f.host unused) into contiguous device memory at `out`
hipError_t launch_pack(const GridDesc& g, const Fields& f, void* out, hipStream_t stream);

// memcpy / FP32 to FP64 by several host threads
void host_copy(double* dst, const double* src, size_t n);
void host_copy(double* dst, const float* src, size_t n);

// Work in `n` chunks of at most `bytes` each: on up to kWorkers host threads,
// each with a pinned buffer of its own, fn(chunk, buffer, event) for every
// chunk; fn returns 0 or a SAC_E_* code (message in the string it is given).
// kNoPinned, and nothing done, if no thread could get a buffer.
constexpr int kNoPinned = -1;
using ChunkFn = std::function<int(long long chunk, void* pinned, hipEvent_t ev, std::string& err)>;
int for_chunks(int device, long long n, size_t bytes, const ChunkFn& fn, std::string& err);

}  // namespace xfer
}  // namespace sac

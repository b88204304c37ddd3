// readback.hip -- reads of large arrays by the host.  No counterpart in the reference.
//
// A copy into pageable memory goes through the runtime's own staging on one
// thread, 17 GB/s into pages that are there and 10 into new ones, whose first
// touch falls on that thread too (and 0.25 ms for 0.6 MB of new ones).  Here up to six
// threads take the chunks in turn: each has two pinned chunks, one filled by the
// GPU while it empties the other.  102 MB of new pages 10.0 -> 3.0 ms, 34 MB 3.4 -> 1.4,
// 0.6 MB 0.05.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

#include "readback.h"

namespace picard {
namespace {

// a copy of 1 MB costs 36 us, 28 GB/s, of 2 MB 35 to 48; arrays of a few MB need
// the smaller one to overlap at all
constexpr int64_t kPin = int64_t(2) << 20;
constexpr int64_t kBig = int64_t(16) << 20;
// memory that the GPU does not reach: the host's alone
bool pageable(const void *host) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, host) != hipSuccess) {
    (void)hipGetLastError();             // unknown to the runtime
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

}  // namespace

Readback::~Readback() {
  for (Worker &w : w_)
    for (int b = 0; b < 2; ++b) {
      if (w.pin[b]) (void)hipHostFree(w.pin[b]);
      if (w.ev[b]) (void)hipEventDestroy(w.ev[b]);
    }
}

// Chunks first, first + step, ...
template <typename OUT>
hipError_t Readback::work(Worker &w, int device, hipStream_t stream, const char *dev, int64_t bytes,
                          int64_t chunk, int first, int step, const OUT &out) {
  hipError_t rc = hipSetDevice(device);
  auto fetch = [&](int64_t at, int b) {
    const int64_t m = std::min(chunk, bytes - at);
    if (rc == hipSuccess) rc = hipMemcpyAsync(w.pin[b], dev + at, m, hipMemcpyDeviceToHost, stream);
    if (rc == hipSuccess) rc = hipEventRecord(w.ev[b], stream);
  };
  int b = 0;
  if (first * chunk < bytes) fetch(first * chunk, 0);
  for (int64_t at = first * chunk; at < bytes && rc == hipSuccess; at += step * chunk, b ^= 1) {
    if (at + step * chunk < bytes) fetch(at + step * chunk, b ^ 1);
    if (rc == hipSuccess) rc = hipEventSynchronize(w.ev[b]);
    if (rc == hipSuccess) out(w.pin[b], at, std::min(chunk, bytes - at));
  }
  return rc;
}

template <typename OUT>
int Readback::run(int device, hipStream_t stream, const char *dev, int64_t bytes, const OUT &out) {
  std::lock_guard<std::mutex> lk(mu_);
  const int64_t chunk = bytes < kBig ? kPin / 2 : kPin;
  const int cpus = std::max(1, (int)std::thread::hardware_concurrency());
  int workers = (int)std::min<int64_t>(std::min(kMaxWorkers, cpus), std::max<int64_t>(1, bytes / kPin));
  // as many as there is pinned memory for
  auto ready = [](Worker &w) {
    for (int b = 0; b < 2; ++b) {
      if (!w.pin[b] && hipHostMalloc(reinterpret_cast<void **>(&w.pin[b]), kPin) != hipSuccess) return false;
      if (!w.ev[b] && hipEventCreateWithFlags(&w.ev[b], hipEventDisableTiming) != hipSuccess) return false;
    }
    return true;
  };
  int have = 0;
  while (have < workers && ready(w_[have])) ++have;
  if (have < workers) (void)hipGetLastError();
  if (!have) return kNoChunks;
  workers = have;
  hipError_t rc[kMaxWorkers] = {};
  std::thread threads[kMaxWorkers];
  int started = 1;
  try {
    for (; started < workers; ++started) {
      const int t = started;
      threads[t] = std::thread([&, t] {
        rc[t] = work(w_[t], device, stream, dev, bytes, chunk, t, workers, out);
      });
    }
  } catch (const std::system_error &) {  // no more threads: the caller takes those chunks
  }
  rc[0] = work(w_[0], device, stream, dev, bytes, chunk, 0, workers, out);
  for (int t = started; t < workers; ++t)
    rc[t] = work(w_[t], device, stream, dev, bytes, chunk, t, workers, out);
  for (int t = 1; t < started; ++t) threads[t].join();
  for (int t = 0; t < workers; ++t)
    if (rc[t] != hipSuccess) {
      (void)hipStreamSynchronize(stream);           // copies into the chunks have ended
      PICARD_HIP(rc[t]);
    }
  return PICARD_OK;
}

int Readback::copy(int device, hipStream_t stream, void *host, const void *dev, int64_t bytes) {
  if (bytes >= direct_copy_ && pageable(host)) {
    const int rc = run(device, stream, static_cast<const char *>(dev), bytes,
                       [host](const char *pin, int64_t at, int64_t m) {
                         std::memcpy(static_cast<char *>(host) + at, pin, m);
                       });
    if (rc != kNoChunks) return rc;
  }
  PICARD_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream));
  PICARD_HIP(hipStreamSynchronize(stream));
  return PICARD_OK;
}

int Readback::widen(int device, hipStream_t stream, double *host, const float4 *E, int64_t n,
                    bool *taken) {
  *taken = n * (int64_t)sizeof(float4) >= direct_widen_ && pageable(host);
  if (!*taken) return PICARD_OK;
  const int rc = run(device, stream, reinterpret_cast<const char *>(E), n * (int64_t)sizeof(float4),
             [host](const char *pin, int64_t at, int64_t m) {
               const float *e = reinterpret_cast<const float *>(pin);
               double *o = host + 3 * (at / (int64_t)sizeof(float4));
               for (int64_t q = 0; q < m / (int64_t)sizeof(float4); ++q)
                 for (int d = 0; d < 3; ++d) o[3 * q + d] = e[4 * q + d];
             });
  *taken = rc != kNoChunks;
  return *taken ? rc : PICARD_OK;
}

}  // namespace picard

// readback.h -- device arrays to pageable host memory through pinned chunks,
// several host threads copying out of them.
#pragma once
#include <mutex>

#include "picard_internal.h"

namespace picard {

class Readback {
 public:
  // copies of fewer than `copy` bytes and E of fewer than `widen` go the runtime's way
  Readback(int64_t copy, int64_t widen) : direct_copy_(copy), direct_widen_(widen) {}
  ~Readback();
  // host[0 .. bytes) = dev, in the stream's order; returns when it is there
  int copy(int device, hipStream_t stream, void *host, const void *dev, int64_t bytes);
  // host[3 q + d] = component d of E[q], q < n.  *taken = false, and nothing done, for
  // few, where `host` is memory that the GPU reaches itself, and without pinned memory.
  int widen(int device, hipStream_t stream, double *host, const float4 *E, int64_t n, bool *taken);

 private:
  static constexpr int kMaxWorkers = 6;
  struct Worker {
    char *pin[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
  };
  // kNoChunks, and nothing done, where there is no pinned memory
  template <typename OUT>
  int run(int device, hipStream_t stream, const char *dev, int64_t bytes, const OUT &out);
  static constexpr int kNoChunks = 1;
  template <typename OUT>
  hipError_t work(Worker &w, int device, hipStream_t stream, const char *dev, int64_t bytes,
                  int64_t chunk, int first, int step, const OUT &out);
  const int64_t direct_copy_, direct_widen_;
  std::mutex mu_;
  Worker w_[kMaxWorkers];
};

}  // namespace picard

// Host-side helpers of the HIP backend: owning device and pinned-host buffers and the
// error-check macros (runtime failures become std::runtime_error, as relay's CUDA
// backend does with its CUDA_CHECK).
#pragma once

#include <hip/hip_runtime_api.h>

#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "relay_hip.h"

#define HIP_CHECK(x)                                                                          \
  do {                                                                                        \
    hipError_t _e = (x);                                                                      \
    if (_e != hipSuccess) throw std::runtime_error(std::string("HIP: ") + hipGetErrorString(_e) + " at " #x); \
  } while (0)

#define RH_CHECK(x)                                                                           \
  do {                                                                                        \
    if ((x) != 0) throw std::runtime_error(std::string("relay_hip: ") + rh_last_error() + " at " #x); \
  } while (0)

namespace relay_hip_host {

// An owning device allocation of n elements.
template <class T>
struct DeviceArray {
  T* p = nullptr;
  std::size_t n = 0;
  DeviceArray() = default;
  explicit DeviceArray(std::size_t count) : n(count) {
    if (count) HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&p), count * sizeof(T)));
  }
  ~DeviceArray() { reset(); }
  DeviceArray(const DeviceArray&) = delete;
  DeviceArray& operator=(const DeviceArray&) = delete;
  DeviceArray(DeviceArray&& o) noexcept : p(o.p), n(o.n) {
    o.p = nullptr;
    o.n = 0;
  }
  DeviceArray& operator=(DeviceArray&& o) noexcept {
    if (this != &o) {
      reset();
      p = o.p;
      n = o.n;
      o.p = nullptr;
      o.n = 0;
    }
    return *this;
  }
  void reset() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
};

// Page-locked host memory that only grows (copies from it run asynchronously).
struct PinnedBuffer {
  void* p = nullptr;
  std::size_t bytes = 0;
  PinnedBuffer() = default;
  PinnedBuffer(const PinnedBuffer&) = delete;
  PinnedBuffer& operator=(const PinnedBuffer&) = delete;
  ~PinnedBuffer() {
    if (p) (void)hipHostFree(p);
  }
  void reserve(std::size_t want) {
    if (want <= bytes) return;
    if (p) HIP_CHECK(hipHostFree(p));
    p = nullptr;
    const std::size_t grow = want + want / 2;
    HIP_CHECK(hipHostMalloc(&p, grow, hipHostMallocDefault));
    bytes = grow;
  }
};

// What the per-layer events of wait_kv_written stand for. A pass records them (an event after
// each layer's KV write) on a backend whose layers are waited for: from its first pass with an
// observer, or from the first wait that found a pass running. On other backends the passes go
// without, since an event between two kernels costs 3 us on the device and 4 us of the
// launching thread (SmolLM2-135M, one token, 30 layers: 910 us a step with them, 777 without).
class KvProgress {
 public:
  explicit KvProgress(int layers) : written_(layers, 0) {}

  // A pass, between its construction and its end, by the thread that runs it.
  class Pass {
   public:
    Pass(KvProgress& p, bool observed) : p_(p) {
      std::lock_guard<std::mutex> lock(p_.mu_);
      ++p_.begun_;
      p_.observed_ = observed;
      if (observed) p_.record_ = true;
    }
    ~Pass() {
      {
        std::lock_guard<std::mutex> lock(p_.mu_);
        p_.over_ = p_.begun_;
      }
      p_.moved_.notify_all();
    }
    Pass(const Pass&) = delete;
    Pass& operator=(const Pass&) = delete;

   private:
    KvProgress& p_;
  };

  // Whether the pass records its layers' events; recorded() follows each of them.
  bool record() const { return record_.load(std::memory_order_relaxed); }
  void recorded(int layer) {
    {
      std::lock_guard<std::mutex> lock(mu_);
      written_[layer] = begun_;
    }
    moved_.notify_all();
  }

  bool running() const {
    std::lock_guard<std::mutex> lock(mu_);
    return over_ < begun_;
  }

  // Returns once the layer's event may be waited for. In a pass with an observer that is at once:
  // the observer has named the layer, or the caller means an earlier pass (and the observer may
  // itself wait for the caller). A pass without one has no such order, so it is the moment that
  // pass has recorded the event, or is over; passes that begin meanwhile do not prolong it.
  void reach(int layer) {
    std::unique_lock<std::mutex> lock(mu_);
    if (over_ == begun_ || observed_) return;
    record_ = true;
    const std::uint64_t pass = begun_;
    moved_.wait(lock, [&] { return over_ >= pass || written_[layer] >= pass; });
  }

 private:
  mutable std::mutex mu_;
  std::condition_variable moved_;
  std::uint64_t begun_ = 0, over_ = 0;  // passes
  std::vector<std::uint64_t> written_;  // the pass of each layer's last event
  bool observed_ = false;               // of the pass running
  std::atomic<bool> record_{false};
};

}  // namespace relay_hip_host

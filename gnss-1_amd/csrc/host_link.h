// host_link.h — fields between device arrays and a caller's host buffers.
//
// The ABI's buffers are pageable FP64 in the reference's order; the device holds T in its own layout.  A
// kernel writes one chunk at a time in the ABI's order straight into pinned host memory (or reads it
// from there), and several host threads, each with a pinned slot of its own, widen or narrow the
// chunks from and to the caller's pages, so that the bus, the conversion and the page faults of a
// fresh buffer run side by side.  (One thread through pageable copies: four 256^3 FP32 fields took 70 to
// 118 ms, now 35 to 39 with the reader's own use of them; four 192 x 256 x 128 FP64 fields in and out 130 ms,
// now 12.5.)
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "engine.h"

namespace gnss {

class HostLink {
 public:
  static constexpr size_t SLOT = 2u << 20;  // bytes of a slot: a large page, and 40 us of the bus
  static constexpr int SLOTS = 8;

  // Pinned memory for transfers of up to `most` bytes at a time: as many slots as such a transfer fills, and
  // one word beside them (flag()).
  void allocate(int dev, size_t most) {
    dev_ = dev;
    n_ = (int)std::min<size_t>(SLOTS, std::max<size_t>(1, (most + SLOT - 1) / SLOT));
    const size_t bytes = n_ == 1 ? std::max<size_t>(most, 1) : n_ * SLOT;
    slot_ = n_ == 1 ? bytes : SLOT;
    flag_at_ = (bytes + 63) / 64 * 64;
    if (hipHostMalloc(&base_, flag_at_ + 64, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      base_ = nullptr;
      throw Error(GNSS_ERR_ALLOC, "hipHostMalloc of " + std::to_string(bytes) + " bytes failed");
    }
    for (int i = 0; i < n_; ++i) GNSS_HIP(hipEventCreateWithFlags(&ev_[i], hipEventDisableTiming));
  }
  void release() {
    for (hipEvent_t& e : ev_)
      if (e) (void)hipEventDestroy(e);
    for (hipEvent_t& e : ev_) e = nullptr;
    if (base_) (void)hipHostFree(base_);
    base_ = nullptr;
  }
  size_t slot_bytes() const { return slot_; }
  int* flag() const { return reinterpret_cast<int*>((char*)base_ + flag_at_); }

  // fn(chunk, slot memory, the slot's event) for every chunk, on up to one thread per slot; the caller's
  // thread takes part.  An exception stops the chunks not yet begun and is thrown here.
  template <typename Fn> void each(int nchunks, Fn&& fn) {
    std::atomic<int> next{0};
    std::exception_ptr err;
    std::mutex mu;
    auto work = [&](int slot) {
      try {
        if (slot) GNSS_HIP(hipSetDevice(dev_));
        for (int c = next++; c < nchunks; c = next++) fn(c, (char*)base_ + slot * slot_, ev_[slot]);
      } catch (...) {
        next = nchunks;
        std::lock_guard<std::mutex> lk(mu);
        if (!err) err = std::current_exception();
      }
    };
    std::vector<std::thread> th;
    const int cpus = (int)std::max(1u, std::thread::hardware_concurrency());
    const int want = std::min({n_, nchunks, cpus});
    try {
      for (int i = 1; i < want; ++i) th.emplace_back(work, i);
    } catch (const std::system_error&) {  // fewer threads then
    }
    work(0);
    for (std::thread& t : th) t.join();
    if (err) std::rethrow_exception(err);
  }

 private:
  int dev_ = 0, n_ = 0;
  size_t slot_ = 0, flag_at_ = 0;
  void* base_ = nullptr;
  hipEvent_t ev_[SLOTS] = {};
};

}  // namespace gnss

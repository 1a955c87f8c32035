// transfer.hpp — copies between device memory and a caller's pageable arrays
// through pinned slots.
//
// The runtime copies pageable memory through one thread, which also takes the
// page faults of a caller's fresh array: 5 GB/s for the three macro arrays of
// a 4097^2 lattice.  Here up to THREADS threads own two pinned slots each:
// while the device fills (or reads) one, its thread moves the other's items to
// (or from) the caller's arrays.  A transfer that fits one slot stays on the
// calling thread.  A Staging belongs to one handle, whose calls come from one
// host thread at a time; its threads end with the call, and its slots are
// freed with the handle.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <functional>
#include <thread>
#include <vector>

namespace lbmhost {

class Staging {
 public:
  static constexpr size_t SLOT = (size_t)1 << 19;  // bytes per slot
  static constexpr int THREADS = 8;                // at most; two slots each
  static constexpr int MAX_PARTS = 9;

  Staging() = default;
  Staging(const Staging&) = delete;
  Staging& operator=(const Staging&) = delete;
  ~Staging() { release(); }

  // Items [off, off + len) of a transfer, each of `unit` bytes of the slot.
  // A Device queues their copy between the device and the slot on a stream; a
  // Host moves them between the slot and the caller's arrays.  Both are called
  // by several threads, for disjoint ranges.
  using Device = std::function<hipError_t(size_t off, size_t len, char* slot)>;
  using Host = std::function<void(size_t off, size_t len, char* slot)>;

  // Queues the copy of `count` parts of `bytes` each to dst, dst + bytes, ...;
  // dst or the parts lie in a slot.
  hipError_t copy(void* dst, const void* const* src, int count, size_t bytes,
                  hipStream_t st) const;

  // Returns when the caller's arrays hold everything.
  hipError_t to_host(hipStream_t st, size_t count, size_t unit, const Device& fetch,
                     const Host& put) {
    return run(st, count, unit, fetch, put, true);
  }
  // Returns when the caller's arrays have been read; the copies to the device
  // are queued on st.
  hipError_t to_device(hipStream_t st, size_t count, size_t unit, const Host& get,
                       const Device& send) {
    return run(st, count, unit, send, get, false);
  }

 private:
  char* buf_ = nullptr;
  size_t slot_ = 0;
  int slots_ = 0;
  std::vector<hipEvent_t> ev_;  // one per slot: its last device copy
  std::vector<char> busy_;      // a copy to the device may still read the slot

  bool pinned_ = false;

  void release() {
    for (size_t i = 0; i < ev_.size(); i++) {
      if (busy_[i]) (void)hipEventSynchronize(ev_[i]);
      (void)hipEventDestroy(ev_[i]);
    }
    ev_.clear();
    busy_.clear();
    if (buf_ && pinned_) (void)hipHostFree(buf_);
    if (buf_ && !pinned_) std::free(buf_);
    buf_ = nullptr;
    slots_ = 0;
    slot_ = 0;
  }

  // Slots for a transfer of `total` bytes: a small one takes one slot of its
  // own size, so that a small handle pins little.
  hipError_t reserve(size_t total) {
    const size_t want = std::min(SLOT, (total + 4095) / 4096 * 4096);
    const int n = total <= SLOT ? 1 : (int)std::min<size_t>(2 * THREADS, (total + SLOT - 1) / SLOT);
    if (slot_ >= want && slots_ >= n) return hipSuccess;
    release();
    pinned_ = hipHostMalloc((void**)&buf_, want * (size_t)n, hipHostMallocDefault) == hipSuccess;
    if (!pinned_) {  // no pinned memory left: the runtime stages the slots itself
      (void)hipGetLastError();
      buf_ = (char*)std::malloc(want * (size_t)n);
      if (!buf_) return hipErrorOutOfMemory;
    }
    for (int i = 0; i < n; i++) {
      hipEvent_t v;
      const hipError_t e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
      if (e != hipSuccess) return e;
      ev_.push_back(v);
      busy_.push_back(0);
    }
    slot_ = want;
    slots_ = n;
    return hipSuccess;
  }

  hipError_t run(hipStream_t st, size_t count, size_t unit, const Device& dev, const Host& host,
                 bool down) {
    if (count == 0) return hipSuccess;
    hipError_t e = reserve((count + 63) / 64 * 64 * unit);
    if (e != hipSuccess) return e;
    int device = 0;
    e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    const size_t chunk = slot_ / unit / 64 * 64;  // whole 64 items keep the parts aligned
    const size_t chunks = (count + chunk - 1) / chunk;
    const int nt = (int)std::min<size_t>((size_t)(slots_ + 1) / 2, chunks);
    const int per = slots_ / nt;  // slots per thread
    std::vector<hipError_t> err((size_t)nt, hipSuccess);
    auto work = [&](int k) {
      hipError_t& r = err[(size_t)k];
      if (k) r = hipSetDevice(device);
      const size_t mine = (chunks - 1 - (size_t)k) / (size_t)nt + 1;  // k, k + nt, ...
      auto slot = [&](size_t j) { return (size_t)k * per + j % (size_t)per; };
      auto at = [&](size_t j) { return buf_ + slot(j) * slot_; };
      auto off = [&](size_t j) { return ((size_t)k + j * (size_t)nt) * chunk; };
      auto len = [&](size_t j) { return std::min(chunk, count - off(j)); };
      auto wait = [&](size_t j) {
        if (r == hipSuccess && busy_[slot(j)]) r = hipEventSynchronize(ev_[slot(j)]);
        busy_[slot(j)] = 0;
      };
      auto queue = [&](size_t j) {
        if (r == hipSuccess) r = dev(off(j), len(j), at(j));
        if (r == hipSuccess) r = hipEventRecord(ev_[slot(j)], st);
        busy_[slot(j)] = r == hipSuccess;
      };
      if (down)
        for (size_t j = 0; j < mine && j < (size_t)per; j++) {
          wait(j);
          queue(j);
        }
      for (size_t j = 0; j < mine; j++) {
        wait(j);
        if (r != hipSuccess) return;
        host(off(j), len(j), at(j));
        if (!down) queue(j);
        if (down && j + (size_t)per < mine) queue(j + (size_t)per);
      }
    };
    std::vector<std::thread> th;
    int started = 1;
    try {
      th.reserve((size_t)nt);
      for (; started < nt; started++) th.emplace_back(work, started);
    } catch (...) {  // no more threads: this one does their share
    }
    work(0);
    for (int k = started; k < nt; k++) work(k);
    for (std::thread& x : th) x.join();
    for (hipError_t r : err)
      if (r != hipSuccess) return r;
    return hipSuccess;
  }
};

}  // namespace lbmhost

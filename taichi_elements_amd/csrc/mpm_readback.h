// Device to host copies into the caller's (pageable) memory.
//
// A copy into pageable memory goes through pinned memory in any case, and what
// costs is its second half: the pages of a fresh numpy array are touched for
// the first time, by one thread.  Here the device writes into pinned slots of
// this object while several threads move the previous ones on (3D 1M
// particles, 32 MB into new arrays: 2.5-4 ms -> 0.9 ms; 16M, 512 MB: 46-51 ms
// -> 12.6).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

namespace mpm {

class Readback {
 public:
  // bytes from src (device, or host memory if on_host) to dst
  struct Segment {
    const void* src;
    void* dst;
    size_t bytes;
    bool on_host;
  };

  // Waits for the stream's work so far and for the copies.  Without pinned
  // memory (or host memory for the bookkeeping) they are plain ones.
  hipError_t copy(const std::vector<Segment>& segments, hipStream_t st) {
    if (again_) {  // a single read does not pay for pinned memory (~0.2 ms per MiB)
      bool began = false;
      const hipError_t e = through_slots(segments, st, began);
      if (began) return e;
      (void)hipGetLastError();
    }
    again_ = true;
    hipError_t e = hipStreamSynchronize(st);
    if (e != hipSuccess) return e;
    for (const Segment& s : segments) {
      if (s.bytes == 0) continue;
      if (s.on_host)
        std::memcpy(s.dst, s.src, s.bytes);
      else if ((e = hipMemcpy(s.dst, s.src, s.bytes, hipMemcpyDeviceToHost)) != hipSuccess)
        return e;
    }
    return hipSuccess;
  }

  void release() {
    for (int k = 0; k < kSlots; k++) {
      if (done_[k]) hipEventDestroy(done_[k]);
      if (slot_[k]) hipHostFree(slot_[k]);
      done_[k] = nullptr;
      slot_[k] = nullptr;
    }
  }

 private:
  static constexpr int kSlots = 4;
  static constexpr size_t kSlotBytes = 2u << 20;
  struct Piece {
    const char* src;
    char* dst;
    size_t bytes;
    bool on_host;
  };

  // began: everything the copies need is there.
  hipError_t through_slots(const std::vector<Segment>& segments, hipStream_t st, bool& began) {
    size_t device = 0, all = 0;
    for (const Segment& s : segments) {
      if (!s.on_host) device += s.bytes;
      all += s.bytes;
    }
    hipError_t e = reserve(device <= kSlotBytes ? 1 : kSlots);
    if (e != hipSuccess) return e;
    if (device <= kSlotBytes) {  // one slot holds everything
      began = true;
      size_t at = 0;
      for (size_t i = 0; i < segments.size();) {  // neighbours on the device in one copy
        const Segment& s = segments[i++];
        if (s.on_host || s.bytes == 0) continue;
        size_t run = s.bytes;
        for (; i < segments.size() && !segments[i].on_host &&
               segments[i].src == (const char*)s.src + run;
             i++)
          run += segments[i].bytes;
        e = hipMemcpyAsync(slot_[0] + at, s.src, run, hipMemcpyDeviceToHost, st);
        if (e != hipSuccess) return e;
        at += run;
      }
      e = hipStreamSynchronize(st);
      if (e != hipSuccess) return e;
      at = 0;
      for (const Segment& s : segments) {
        if (s.bytes == 0) continue;
        std::memcpy(s.dst, s.on_host ? s.src : slot_[0] + at, s.bytes);
        if (!s.on_host) at += s.bytes;
      }
      return hipSuccess;
    }
    std::vector<Piece> pieces;
    std::vector<std::atomic<int>> moved;
    try {
      for (const Segment& s : segments)
        for (size_t at = 0; at < s.bytes; at += kSlotBytes)
          pieces.push_back({(const char*)s.src + at, (char*)s.dst + at,
                            std::min(kSlotBytes, s.bytes - at), s.on_host});
      moved = std::vector<std::atomic<int>>(pieces.size());
    } catch (const std::bad_alloc&) {
      return hipErrorOutOfMemory;
    }
    began = true;
    e = hipStreamSynchronize(st);  // no thread waits for kernels
    if (e != hipSuccess) return e;
    return pipeline(pieces, moved, st, all);
  }

  // The first n slots and their events.
  hipError_t reserve(int n) {
    hipError_t e = hipSuccess;
    for (int k = 0; k < n; k++) {
      if (!slot_[k] && (e = hipHostMalloc((void**)&slot_[k], kSlotBytes)) != hipSuccess) {
        slot_[k] = nullptr;
        return e;
      }
      if (!done_[k] &&
          (e = hipEventCreateWithFlags(&done_[k], hipEventDisableTiming)) != hipSuccess) {
        done_[k] = nullptr;
        return e;
      }
    }
    return e;
  }

  // Piece k passes through slot k % kSlots.  Every mover copies its share of
  // each piece once the piece has arrived; a slot is refilled when all movers
  // are done with it.
  hipError_t pipeline(const std::vector<Piece>& pieces, std::vector<std::atomic<int>>& moved,
                      hipStream_t st, size_t bytes) {
    const int n = (int)pieces.size();
    std::atomic<int> arrived{0};
    for (auto& m : moved) m.store(0, std::memory_order_relaxed);
    const int hw = (int)std::max(2u, std::thread::hardware_concurrency());
    const int want = (int)std::min<size_t>({(size_t)kMovers, (size_t)hw / 2, 1 + bytes / (4u << 20)});
    std::atomic<int> movers{0};  // decided below; movers wait for it
    const auto move = [&](int me) {
      int count;
      while ((count = movers.load(std::memory_order_acquire)) == 0) std::this_thread::yield();
      for (int k = 0; k < n; k++) {
        while (arrived.load(std::memory_order_acquire) <= k) std::this_thread::yield();
        const Piece& p = pieces[k];
        const size_t share = ((p.bytes + count - 1) / count + 4095) & ~(size_t)4095;
        const size_t a = std::min(p.bytes, share * me), b = std::min(p.bytes, a + share);
        if (b > a) std::memcpy(p.dst + a, slot(p, k) + a, b - a);
        moved[k].fetch_add(1, std::memory_order_release);
      }
    };
    std::vector<std::thread> threads;
    try {
      threads.reserve(want);
      for (int m = 0; m < want; m++) threads.emplace_back(move, m);
    } catch (...) {  // fewer threads, or none: the movers there are share the work
    }
    const int count = (int)threads.size();
    movers.store(std::max(count, 1), std::memory_order_release);
    hipError_t err = hipSuccess;
    const auto fetch = [&](int k) {
      if (pieces[k].on_host || err != hipSuccess) return;
      err = hipMemcpyAsync(slot_[k % kSlots], pieces[k].src, pieces[k].bytes,
                           hipMemcpyDeviceToHost, st);
      if (err == hipSuccess) err = hipEventRecord(done_[k % kSlots], st);
    };
    for (int k = 0; k < std::min(n, kSlots); k++) fetch(k);
    for (int k = 0; k < n; k++) {
      if (!pieces[k].on_host && err == hipSuccess) err = hipEventSynchronize(done_[k % kSlots]);
      if (count == 0 && err == hipSuccess)
        std::memcpy(pieces[k].dst, slot(pieces[k], k), pieces[k].bytes);
      arrived.store(k + 1, std::memory_order_release);
      if (k >= 1 && k - 1 + kSlots < n) {  // the previous piece's slot
        while (moved[k - 1].load(std::memory_order_acquire) < count) std::this_thread::yield();
        fetch(k - 1 + kSlots);
      }
    }
    for (auto& t : threads) t.join();
    return err;
  }
  const char* slot(const Piece& p, int k) const {
    return p.on_host ? p.src : slot_[k % kSlots];
  }

  static constexpr int kMovers = 6;
  bool again_ = false;
  char* slot_[kSlots] = {};
  hipEvent_t done_[kSlots] = {};
};

}  // namespace mpm

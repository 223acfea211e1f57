// cs_transfer.h -- copies of a whole state between the caller's (pageable)
// arrays and the device through pinned staging slots.
//
// The runtime's copy down to pageable memory moves one chunk at a time on the
// calling thread, and a fresh destination array costs that thread the page
// faults and the clearing of every page besides.  Here the calling thread
// only puts the slots' copies on the handle's stream and waits for them, and
// up to kWorkers threads move the words between the slots and the caller's
// arrays, so the page faults are taken side by side.  The threads make no
// runtime call (a thread's first one costs about 0.2 ms).
// Milliseconds down (into a new array) / up, runtime's copy -> staged: 28 MiB
// 2.4 -> 1.8, 48 MiB 4.2 -> 2.6, 125 MiB 12.1 -> 4.4 / 5.0 -> 3.7, 225 MiB
// 22 -> 7.8 / 8.8 -> 6.3, 823 MiB 85 -> 23 / 32 -> 22 (40 GB/s, the link).
// Below the thresholds the threads cost what they gain.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>

namespace cs {

constexpr int kWorkers = 8;                        // host threads of one transfer at most
constexpr int kSlots = 16;                         // pinned slots
constexpr size_t kSlotMin = (size_t)1 << 20;       // a slot: a 32nd of the state, between
constexpr size_t kSlotMax = (size_t)2 << 20;       // 1 and 2 MiB
constexpr size_t kStagedDown = (size_t)24 << 20;   // smallest staged transfers (transfer())
constexpr size_t kStagedUp = (size_t)64 << 20;
constexpr size_t kStagedAtOnce = (size_t)64 << 20; // smaller ones: from the second transfer on (StagingPool)

struct Segment {
  char* dev;
  char* host;
  size_t bytes;
};

inline size_t slot_bytes(size_t total) {
  return std::min(kSlotMax, std::max(kSlotMin, total / 32 & ~(size_t)4095));
}

// Pinned slots of one transfer at a time (16 to 32 MiB) with their events.
struct Staging {
  char* pin = nullptr;
  size_t slot = 0;
  int device = -1;
  hipEvent_t ev[kSlots] = {};
  // for streams of device dev, whichever is the calling thread's: an event can
  // only be recorded on a stream of the device that was current when it was made
  bool make(int dev, size_t bytes) {
    device = dev;
    slot = bytes;
    int was = dev;
    bool ok = hipGetDevice(&was) == hipSuccess && (was == dev || hipSetDevice(dev) == hipSuccess);
    ok = ok && hipHostMalloc((void**)&pin, kSlots * slot, hipHostMallocDefault) == hipSuccess;
    if (!ok) pin = nullptr;
    for (hipEvent_t& e : ev)
      if (ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        e = nullptr;
        ok = false;
      }
    if (was != dev) (void)hipSetDevice(was);
    if (!ok) (void)hipGetLastError();
    return ok;
  }
  ~Staging() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (pin) (void)hipHostFree(pin);
  }
};

// The slot sets not in use, kept for the next transfer of any handle of their
// device: at most kIdleSets of them, released when the last handle is
// destroyed.  A transfer owns its set alone.  A MiB of slots costs 70 us to
// have and give back, so a set has what its transfer needs, one that needs
// more replaces it, and below 64 MiB, where a transfer gains less than its
// set costs, the first one takes plain copies: a program that brings one
// state back pays nothing (handle made, 28 MiB up, down, handle gone: 10.4 ms,
// with a set of 32 MiB made at once 12.9), and one that goes on has its slots
// from the second transfer.
class StagingPool {
 public:
  static constexpr size_t kIdleSets = 2;
  void enter() {
    std::lock_guard<std::mutex> l(mu_);
    ++handles_;
  }
  void leave() {
    std::unique_ptr<Staging> drop[kIdleSets];
    std::lock_guard<std::mutex> l(mu_);
    if (--handles_ == 0) {
      for (size_t q = 0; q < kIdleSets; ++q) drop[q] = std::move(idle_[q]);
      small_ = 0;
    }
  }
  std::unique_ptr<Staging> take(hipStream_t st, size_t total) {
    const size_t slot = slot_bytes(total);
    int dev = 0;
    if (hipStreamGetDevice(st, &dev) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    std::unique_ptr<Staging> s;
    {
      std::lock_guard<std::mutex> l(mu_);
      for (auto& q : idle_)
        if (q && q->device == dev && (!s || s->slot < q->slot)) std::swap(s, q);
      if (s && s->slot >= slot) return s;
      if (!s && total < kStagedAtOnce && small_++ == 0) return nullptr;
    }
    s.reset(new (std::nothrow) Staging());
    if (s && !s->make(dev, slot)) s.reset();
    return s;
  }
  void give(std::unique_ptr<Staging> s) {
    std::lock_guard<std::mutex> l(mu_);
    for (auto& q : idle_)
      if (!q) {
        q = std::move(s);
        return;
      }
  }

 private:
  std::mutex mu_;
  int handles_ = 0;
  unsigned small_ = 0;  // transfers below kStagedAtOnce that found no set
  std::unique_ptr<Staging> idle_[kIdleSets];
};
// never destroyed: the runtime may be gone by the time static objects are
inline StagingPool& staging_pool() {
  alignas(StagingPool) static char mem[sizeof(StagingPool)];
  static StagingPool* p = new (mem) StagingPool();
  return *p;
}

// One transfer: chunk c of the segments goes through slot c % kSlots.
struct Transfer {
  const Segment* seg;
  int nseg;
  size_t slot;
  char* pin;
  bool down;
  int64_t n = 0;                       // chunks
  std::atomic<int64_t> taken{0};       // chunks handed to a worker
  std::atomic<int64_t> opened{0};      // chunks below it: down, their copy has finished; up, their slot may be filled
  std::atomic<int64_t> moved[kSlots];  // the last chunk whose words a worker moved through the slot, plus one
  std::atomic<bool> stop{false};

  Transfer(const Segment* s, int ns, size_t slot_, const Staging& S, bool to_host)
      : seg(s), nseg(ns), slot(slot_), pin(S.pin), down(to_host) {
    for (int q = 0; q < ns; ++q) n += (int64_t)((s[q].bytes + slot - 1) / slot);
    for (auto& m : moved) m.store(0, std::memory_order_relaxed);
    if (!down) opened.store(kSlots, std::memory_order_relaxed);
  }
  Segment chunk(int64_t c) const {
    for (int q = 0; q < nseg; ++q) {
      const int64_t have = (int64_t)((seg[q].bytes + slot - 1) / slot);
      if (c < have) {
        const size_t off = (size_t)c * slot;
        return Segment{seg[q].dev + off, seg[q].host + off, std::min(slot, seg[q].bytes - off)};
      }
      c -= have;
    }
    return Segment{nullptr, nullptr, 0};
  }
  void work() {
    for (;;) {
      const int64_t c = taken.fetch_add(1, std::memory_order_relaxed);
      if (c >= n) return;
      while (opened.load(std::memory_order_acquire) <= c) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      const Segment k = chunk(c);
      char* p = pin + (size_t)(c % kSlots) * slot;
      if (down) memcpy(k.host, p, k.bytes);
      else memcpy(p, k.host, k.bytes);
      moved[c % kSlots].store(c + 1, std::memory_order_release);
    }
  }
  bool has_moved(int64_t c) const { return c < 0 || moved[c % kSlots].load(std::memory_order_acquire) == c + 1; }
  // the calling thread: copies put on the stream up to `put`, finished up to `fin`
  hipError_t drive(hipStream_t st, hipEvent_t* ev) {
    int64_t put = 0, fin = 0;
    while (fin < n) {
      const bool room = put < n && put - fin < kSlots && has_moved(down ? put - kSlots : put);
      hipError_t e = hipSuccess;
      if (room) {
        const Segment k = chunk(put);
        char* p = pin + (size_t)(put % kSlots) * slot;
        e = down ? hipMemcpyAsync(p, k.dev, k.bytes, hipMemcpyDeviceToHost, st)
                 : hipMemcpyAsync(k.dev, p, k.bytes, hipMemcpyHostToDevice, st);
        if (e == hipSuccess) e = hipEventRecord(ev[put % kSlots], st);
        ++put;
      } else if (fin < put) {
        e = hipEventSynchronize(ev[fin % kSlots]);
        ++fin;
        opened.store(down ? fin : fin + kSlots, std::memory_order_release);
      } else {
        std::this_thread::yield();
      }
      if (e != hipSuccess) {
        stop.store(true, std::memory_order_relaxed);
        (void)hipStreamSynchronize(st);  // no copy may still use the slots or the caller's arrays
        return e;
      }
    }
    return hipSuccess;
  }
};

// memory that the runtime knows nothing of
inline bool pageable(const char* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}
inline hipError_t plain_copy(hipStream_t st, const Segment& s, bool to_host) {
  return to_host ? hipMemcpyAsync(s.host, s.dev, s.bytes, hipMemcpyDeviceToHost, st)
                 : hipMemcpyAsync(s.dev, s.host, s.bytes, hipMemcpyHostToDevice, st);
}

// Copies the segments (kSegments at most) on `st` and waits for them.  Pinned
// arrays, and others that the runtime knows, are its own to copy: the link
// reaches them without a second pass (225 MiB of them up 4.4 ms and down 4.2,
// through the slots 6.3 and 6.1).  Pageable ones are staged down from 24 MiB
// and up from 64 MiB in all; below, and where no slots or threads are to be
// had or the staging fails, they take the runtime's copies too.
constexpr int kSegments = 5;
inline hipError_t transfer(hipStream_t st, const Segment* all, int nall, bool to_host) {
  Segment seg[kSegments];
  int nseg = 0;
  size_t total = 0;
  for (int q = 0; q < nall; ++q) {
    if (pageable(all[q].host)) {
      total += all[q].bytes;
      seg[nseg++] = all[q];
    } else {
      const hipError_t e = plain_copy(st, all[q], to_host);
      if (e != hipSuccess) return e;
    }
  }
  std::unique_ptr<Staging> S;
  if (total >= (to_host ? kStagedDown : kStagedUp)) S = staging_pool().take(st, total);
  if (S) {
    Transfer T(seg, nseg, slot_bytes(total), *S, to_host);
    std::thread th[kWorkers];
    const int want = (int)std::min<int64_t>(std::min<int64_t>(kWorkers, T.n),
                                            std::max(1u, std::thread::hardware_concurrency()));
    int have = 0;
    try {
      for (; have < want; ++have) th[have] = std::thread(&Transfer::work, &T);
    } catch (const std::exception&) {  // no thread or no memory for its start: fewer share the chunks
    }
    if (have > 0) {
      const hipError_t e = T.drive(st, S->ev);
      for (int t = 0; t < have; ++t) th[t].join();
      staging_pool().give(std::move(S));
      if (e == hipSuccess) return e;
      (void)hipGetLastError();  // the plain copies below redo the whole transfer, and report what still fails
    } else {
      staging_pool().give(std::move(S));
    }
  }
  for (int q = 0; q < nseg; ++q) {
    const hipError_t e = plain_copy(st, seg[q], to_host);
    if (e != hipSuccess) return e;
  }
  return hipStreamSynchronize(st);
}

}  // namespace cs

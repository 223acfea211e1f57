// Host check of the state transfers' staging (cs_transfer.h) over the fake
// runtime of fake_hip/: argument 1 names the check, "ok" is printed when it holds.
#include "cs_transfer.h"

#include <stdio.h>
#include <stdlib.h>

#include <string>
#include <vector>

using namespace cs;

// operator new fails once `budget` more allocations have been made (-1: never)
static std::atomic<int> budget{-1};
void* operator new(size_t n) {
  if (budget.load() >= 0 && budget.fetch_sub(1) <= 0) throw std::bad_alloc();
  if (void* p = malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

static int fail(const char* what) {
  printf("%s\n", what);
  return 1;
}

// a state in three arrays of uneven size, past the threshold of its direction
struct State {
  std::vector<char> dev[3], host[3];
  Segment seg[3];
  explicit State(size_t mib) {
    const size_t n[3] = {(mib << 19) + 24, (mib << 18) + 8, (mib << 18) + 4096};
    for (int q = 0; q < 3; ++q) {
      dev[q].resize(n[q]);
      host[q].resize(n[q]);
      seg[q] = Segment{dev[q].data(), host[q].data(), n[q]};
    }
  }
  size_t bytes() const { return dev[0].size() + dev[1].size() + dev[2].size(); }
  void fill(bool down, int seed) {
    for (int q = 0; q < 3; ++q) {
      auto &a = down ? dev[q] : host[q], &b = down ? host[q] : dev[q];
      for (size_t i = 0; i < a.size(); ++i) a[i] = (char)((i * 2654435761u + seed) >> 7);
      std::fill(b.begin(), b.end(), 0);
    }
  }
  bool same() const { return dev[0] == host[0] && dev[1] == host[1] && dev[2] == host[2]; }
};

// past the first small transfer, which has no slots yet, with slots for any size
static bool warm(FakeStream* st) {
  State S(130);
  return transfer(st, S.seg, 3, true) == hipSuccess;
}

// slots from the second transfer on below 64 MiB, at once from there, anew after the last handle
static int first_small() {
  FakeStream st{0};
  State S(25), L(64);
  for (int round = 0; round < 2; ++round) {
    for (int n = 0; n < 3; ++n) {
      S.fill(true, n);
      fake().direct = fake().staged = 0;
      if (transfer(&st, S.seg, 3, true) != hipSuccess || !S.same()) return fail("words lost");
      if ((n == 0 ? fake().direct : fake().staged) != S.bytes()) return fail("slots not from the second transfer");
    }
    const size_t few = fake().pin.begin()->second;
    if (few > 16 * (size_t)(1 << 20)) return fail("more slots than the transfer needs");
    L.fill(true, 9);
    fake().direct = fake().staged = 0;
    if (transfer(&st, L.seg, 3, true) != hipSuccess || !L.same()) return fail("words lost");
    if (fake().staged != L.bytes()) return fail("a large transfer not staged");
    if (fake().pin.size() != 1 || fake().pin.begin()->second <= few) return fail("the small set was not replaced");
    staging_pool().leave();
    if (!fake().pin.empty()) return fail("slots kept after the last handle");
    staging_pool().enter();
    fake().direct = fake().staged = 0;
    if (transfer(&st, L.seg, 3, true) != hipSuccess || fake().staged != L.bytes())
      return fail("the first large transfer not staged");
    staging_pool().leave();
    staging_pool().enter();
  }
  return 0;
}

// the handle's stream on a device that is not the calling thread's
static int other_device() {
  FakeStream st{1};
  if (!warm(&st)) return fail("a transfer of a handle on another device failed");
  for (bool down : {true, false}) {
    State S(down ? 25 : 66);
    S.fill(down, 3);
    fake().direct = fake().staged = 0;
    if (transfer(&st, S.seg, 3, down) != hipSuccess) return fail("a transfer of a handle on another device failed");
    if (!S.same()) return fail("words lost");
    if (fake().staged != S.bytes()) return fail("not staged");
    if (fake().device != 0) return fail("the calling thread's device was changed");
  }
  return 0;
}

// staging that fails half way: the plain copies take over, and no error is left behind
static int fall_back() {
  FakeStream st{0};
  if (!warm(&st)) return fail("failed");
  for (bool down : {true, false}) {
    State S(down ? 40 : 80);
    S.fill(down, 5);
    fake().fail_record = 1;
    if (transfer(&st, S.seg, 3, down) != hipSuccess) return fail("no fall back to the plain copies");
    if (!S.same()) return fail("words lost");
    if (hipGetLastError() != hipSuccess) return fail("an error is left for the next call");
  }
  return 0;
}

// arrays that the runtime can reach by itself: its own copies, no pass through the slots
static int pinned_arrays() {
  FakeStream st{0};
  if (!warm(&st)) return fail("failed");
  for (bool down : {true, false})
    for (int pin = 0; pin < 3; ++pin) {  // none, one, all of them
      State S(down ? 25 : 66);
      char* own[3] = {};
      for (int q = 0; q < 3; ++q)
        if (pin == 2 || (pin == 1 && q == 1)) {
          if (hipHostMalloc((void**)&own[q], S.seg[q].bytes / 4096 * 4096 + 4088, hipHostMallocDefault) != hipSuccess)
            return fail("no memory");
          S.seg[q].bytes = S.seg[q].bytes / 4096 * 4096;
          S.seg[q].host = own[q];
          S.host[q].resize(S.seg[q].bytes);
          S.dev[q].resize(S.seg[q].bytes);
          S.seg[q].dev = S.dev[q].data();
        }
      S.fill(down, 7);
      if (!down)
        for (int q = 0; q < 3; ++q)
          if (own[q]) memcpy(own[q], S.host[q].data(), S.seg[q].bytes);
      fake().direct = fake().staged = 0;
      if (transfer(&st, S.seg, 3, down) != hipSuccess) return fail("failed");
      size_t direct = 0;
      for (int q = 0; q < 3; ++q)
        if (own[q]) {
          direct += S.seg[q].bytes;
          if (down) memcpy(S.host[q].data(), own[q], S.seg[q].bytes);
        }
      if (!S.same()) return fail("words lost");
      if (pin == 0 && fake().staged != S.bytes()) return fail("pageable arrays not staged");
      if (fake().direct < direct) return fail("a pinned array went through the slots");
      for (char* p : own)
        if (p) hipHostFree(p);
    }
  return 0;
}

// no memory for any thread's start, or after the first or the third (the slots are in the pool)
static int no_thread_memory() {
  FakeStream st{0};
  if (!warm(&st)) return fail("failed");
  for (bool down : {true, false})
    for (int have : {0, 1, 3}) {
      State S(down ? 25 : 66);
      S.fill(down, 11);
      budget = have;
      const hipError_t e = transfer(&st, S.seg, 3, down);
      budget = -1;
      if (e != hipSuccess) return fail("failed");
      if (!S.same()) return fail("words lost");
    }
  return 0;
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  int rc = 2;
  staging_pool().enter();
  if (what == "other_device") rc = other_device();
  if (what == "first_small") rc = first_small();
  if (what == "fall_back") rc = fall_back();
  if (what == "pinned_arrays") rc = pinned_arrays();
  if (what == "no_thread_memory") rc = no_thread_memory();
  staging_pool().leave();
  if (rc == 0 && (fake().events != 0 || !fake().pin.empty())) rc = fail("slots kept after the last handle");
  if (rc == 0) printf("ok\n");
  return rc;
}

/*
 * copyout.cpp over a stand-in for the HIP runtime: device memory is host memory, and a stream either runs a launch
 * before the call returns (the device is always ahead of the caller) or hands it to a thread of its own.  Prints a
 * line per run; exits with 1 if any failed.
 */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <deque>
#include <functional>
#include <mutex>
#include <random>
#include <thread>
#include <utility>
#include <vector>

#include "../clovers_amd/csrc/copyout.h"

namespace {

struct Stream {
  bool at_once = true;
  std::mutex m;
  std::condition_variable cv;
  std::deque<std::function<void()>> ops;
  bool busy = false, stop = false;
  std::thread t;
  void start() {
    t = std::thread([this] {
      std::unique_lock<std::mutex> l(m);
      for (;;) {
        cv.wait(l, [this] { return stop || !ops.empty(); });
        if (stop) return;
        auto op = ops.front();
        ops.pop_front();
        busy = true;
        l.unlock();
        op();
        l.lock();
        busy = false;
      }
    });
  }
  ~Stream() {
    if (!t.joinable()) return;
    {
      std::lock_guard<std::mutex> l(m);
      stop = true;
    }
    cv.notify_all();
    t.join();
  }
  void push(std::function<void()> op) {
    if (at_once) return op();
    {
      std::lock_guard<std::mutex> l(m);
      ops.push_back(op);
    }
    cv.notify_all();
  }
  bool idle() {
    std::lock_guard<std::mutex> l(m);
    return ops.empty() && !busy;
  }
} g_stream;

std::vector<std::pair<const char *, size_t>> g_known; /* destinations that the runtime knows */
std::atomic<size_t> g_link{0};                        /* bytes that launches have written */
size_t g_pinned = 0, g_allocs = 0;                    /* bytes of pinned memory now; allocations so far */
std::vector<std::pair<void *, size_t>> g_blocks;

}  // namespace

extern "C" {
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  a->type = hipMemoryTypeUnregistered;
  for (auto &k : g_known)
    if ((const char *)p >= k.first && (const char *)p < k.first + k.second) a->type = hipMemoryTypeHost;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned int) {
  *p = aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  g_blocks.push_back({*p, n});
  g_pinned += n;
  g_allocs++;
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
  for (auto &b : g_blocks)
    if (b.first == p) g_pinned -= std::exchange(b, {}).second;
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  g_stream.push([=] { memcpy(d, s, n); });
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return g_stream.idle() ? hipSuccess : hipErrorNotReady; }
hipError_t hipStreamSynchronize(hipStream_t) {
  while (!g_stream.idle()) std::this_thread::yield();
  return hipSuccess;
}
}

namespace clv {
void launch_copy_out(hipStream_t, const void *src, void *dst, size_t bytes, uint32_t *flags, uint32_t stamp,
                     const uint64_t *stats, uint64_t *stats_out) {
  g_link += bytes;
  g_stream.push([=] {
    for (size_t k = 0; k * COPY_CHUNK < bytes; k++) {
      const size_t at = k * COPY_CHUNK, n = bytes - at < COPY_CHUNK ? bytes - at : COPY_CHUNK;
      if (k == 0 && stats) memcpy(stats_out, stats, 64);
      memcpy((char *)dst + at, (const char *)src + at, n);
      __atomic_store_n(flags + k, stamp, __ATOMIC_RELEASE);
    }
  });
}
}  // namespace clv

/* one array per list; in it, destinations of `bytes`, pinned where `known`, or left out where `skip` */
struct Dst {
  size_t bytes;
  bool known, skip;
};
typedef std::vector<std::vector<Dst>> Case;

static bool one(clv::CopyOut &co, const Case &c, uint32_t seed) {
  std::mt19937 rng(seed);
  std::vector<std::vector<uint32_t>> dev;
  std::vector<clv::CopyArray> arrays;
  std::vector<clv::CopySeg> segs;
  std::vector<std::vector<char>> out;
  g_known.clear();
  for (auto &a : c) {
    size_t n = 0;
    for (auto &d : a) n += d.bytes;
    std::vector<uint32_t> v(n / 4);
    uint32_t word = rng();
    for (auto &x : v) x = word = word * 1664525u + 1013904223u;
    dev.push_back(std::move(v));
  }
  size_t pageable = 0, runs = 0;
  for (uint32_t a = 0; a < c.size(); a++) {
    size_t off = 0;
    arrays.push_back({dev[a].data(), dev[a].size() * 4});
    for (auto &d : c[a]) {
      out.emplace_back(d.bytes + 128, (char)0x5a);
      char *p = out.back().data() + 64;
      if (d.known) g_known.push_back({p, d.bytes});
      if (!d.skip) segs.push_back({a, off, d.bytes, p});
      if (!d.skip && !d.known) {
        pageable += d.bytes;
        runs++;
      }
      off += d.bytes;
    }
  }
  uint64_t stats[8], got[8];
  for (int k = 0; k < 8; k++) stats[k] = rng();
  g_link = 0;
  const hipError_t e = co.run(nullptr, arrays, segs, stats, got);
  if (e != hipSuccess) return printf("FAILED: error %d\n", (int)e), false;
  if (memcmp(stats, got, 64)) return printf("FAILED: counters\n"), false;
  size_t k = 0;
  for (uint32_t a = 0; a < c.size(); a++) {
    const char *src = (const char *)dev[a].data();
    for (auto &d : c[a]) {
      const std::vector<char> &o = out[k++];
      if (!d.skip && memcmp(o.data() + 64, src, d.bytes)) return printf("FAILED: bytes\n"), false;
      for (size_t i = 0; i < o.size(); i++)
        if ((d.skip || i < 64 || i >= 64 + d.bytes) && o[i] != 0x5a) return printf("FAILED: beside\n"), false;
      src += d.bytes;
    }
  }
  /* what the pageable destinations need, in whole chunks */
  if (g_link > pageable + 2 * COPY_CHUNK * runs) return printf("FAILED: %zu bytes sent for %zu\n", g_link.load(), pageable), false;
  printf("ok\n");
  return true;
}

int main(int argc, char **argv) {
  g_stream.at_once = argc > 1 && !strcmp(argv[1], "at-once");
  if (!g_stream.at_once) g_stream.start();
  const size_t MB = 1 << 20, L = 25 * MB - 4, S = 100004;
  const bool P = true, F = false;
  std::vector<Case> cases = {
      {{{L, P, F}}, {{L, F, F}}},                                       /* a pinned image, pageable second moments */
      {{{L, F, F}}, {{L, P, F}}},
      {{{L, F, F}}, {{L, F, F}}},
      {{{L, P, F}}, {{L, P, F}}},
      {{{3 * L, P, F}, {S, F, F}, {17 * MB, F, F}}},                    /* a batch: the first image pinned */
      {{{S, F, F}, {3 * L, P, F}, {S, F, F}}},                          /* one in the middle */
      {{{S, P, F}, {L, F, F}, {17 * MB, P, F}}},
      {{{L, F, F}, {S, F, F}}, {{L, F, P}, {S, F, F}}},                 /* second moments of the later job only */
      {{{4, F, F}, {4, P, F}, {8 * MB, F, F}, {4, F, F}}},
      {{{24, F, F}}},
  };
  std::mt19937 rng(5);
  for (int k = 0; k < 12; k++) {
    Case c(1 + rng() % 2);
    for (uint32_t n = 1 + rng() % 5; n > 0; n--) {
      const size_t b = 4 * (1 + rng() % (rng() % 3 ? 5 * MB : 40000));
      for (auto &a : c) a.push_back({b, rng() % 2 == 0, F});
    }
    cases.push_back(c);
  }
  bool good = true;
  clv::CopyOut kept;
  for (uint32_t k = 0; k < cases.size(); k++) {
    printf("case %u: ", k);
    good = one(kept, cases[k], k) && good; /* a context that has pinned memory by then */
    clv::CopyOut fresh;
    printf("case %u, new context: ", k);
    good = one(fresh, cases[k], k) && good;
    printf("case %u, its next call: ", k);
    good = one(fresh, cases[k], k + 100) && good;
  }
  /* what a context pins: little until it has copied a lot, then the large windows, once */
  {
    const size_t before = g_pinned, allocs = g_allocs;
    clv::CopyOut co;
    for (uint32_t k = 0; k < 40; k++) {
      printf("large call %u: ", k);
      good = one(co, {{{17 * MB, F, F}}}, k) && good;
      const size_t pinned = g_pinned - before;
      if (k < 3 ? pinned > 9 * MB : k == 39 && (pinned < 16 * MB || pinned > 17 * MB)) good = false, printf("FAILED: pinned %zu\n", pinned);
    }
    if (g_allocs - allocs != 2) good = false, printf("FAILED: %zu allocations\n", g_allocs - allocs);
  }
  return good ? 0 : 1;
}

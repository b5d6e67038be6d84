/*
 * copyout.cpp -- results from device arrays into the caller's memory (copyout.h).
 */
#include "copyout.h"

#include <sched.h>
#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <system_error>
#include <utility>

namespace clv {

namespace {

/* a window's half of the pinned memory: two of 8 MB keep the link busy (150 us
 * each) and pin no more than the 16 MB a context may have staged with.  Their
 * pages' first touch costs 2 to 4 ms over the threads where the device does not
 * hide it, which a context that copies once never earns back, so it starts with
 * half of them, and the first copy that these do not hold after GROW_AFTER bytes
 * gets the larger ones.  First hits and normals at 1080p, a new context's calls
 * 1 / 2 / 3: 8.7 / 6.1 / 6.0 ms the runtime's way, 10.7 / 3.4 / 3.4 with 8 MB at
 * once, 8.0 / 5.0 / 3.3 so; with 2 MB first a tenth less in the first call, but
 * results of 3 to 25 MB take a sixth longer until then.  (With 4 MB for good,
 * calls that return 14 MB take 1 to 3% longer.) */
#define HALF_FIRST ((size_t)4 << 20)
#define HALF_BYTES ((size_t)8 << 20)
#define GROW_AFTER ((size_t)48 << 20)
#define MAX_FLAGS (HALF_BYTES / COPY_CHUNK)
#define PIN_HEAD (64 + 2 * MAX_FLAGS * sizeof(uint32_t))

/* parts of at most 2 MB, cut at the destination's 2 MB boundaries: two threads
 * that touch the same unmapped huge page both clear one.  Runs below 4 MB are
 * cut into 256 KB, so that the helpers have something to do. */
#define PART_LARGE ((size_t)2 << 20)
#define PART_SMALL ((size_t)256 << 10)
#define LARGE_RUN ((size_t)4 << 20)

/* from here on the helpers are woken: they take 20 to 50 us to come, the time of
 * a 1 MB host copy */
#define HELP_BYTES ((size_t)1 << 20)
#define HELPERS 3u

/* Pinned memory costs 0.1 ms and 0.03 ms per 64 KB of its first touch.  A render's image and counters earn that back in
 * their first call (the first copies of a process the runtime's way cost 6 ms more, the next ones 0.45 ms where a
 * 200x200 image takes 0.21), and so does a large first-hit probe (640x360: 1.36 ms, 1.75 the runtime's way).  For small
 * probes, which have no counters, it is allocated once the context has sent this many times their size the runtime's
 * way (200x200: first 0.54 ms, pinned at once 0.64; then 0.21 and 0.08). */
#define PIN_LARGE ((size_t)1 << 20)
#define PIN_AFTER 4u

inline void pause_cpu() { __builtin_ia32_pause(); }

/* memory the runtime knows (pinned or device memory): it copies there by itself */
bool known_to_runtime(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

/* maps a range's pages at once; what is in them stays.  False from a kernel that cannot (before 5.14). */
bool map_range(char *p, size_t bytes) {
#ifdef MADV_POPULATE_WRITE
  const uintptr_t page = 4096, at = (uintptr_t)p & ~(page - 1);
  return madvise((void *)at, ((uintptr_t)p + bytes - at + page - 1) & ~(page - 1), MADV_POPULATE_WRITE) == 0;
#else
  return false;
#endif
}

/* destinations that overlap are written one after the other, as they are listed */
bool overlap(const std::vector<CopySeg> &segs) {
  std::vector<std::pair<uintptr_t, uintptr_t>> r;
  for (const CopySeg &s : segs) r.push_back({(uintptr_t)s.dst, (uintptr_t)s.dst + s.bytes});
  std::sort(r.begin(), r.end());
  for (size_t k = 1; k < r.size(); k++)
    if (r[k].first < r[k - 1].second) return true;
  return false;
}

}  // namespace

CopyOut::~CopyOut() {
  {
    std::lock_guard<std::mutex> l(m_);
    stop_ = true;
  }
  cv_.notify_all();
  for (auto &t : helpers_) t.join();
  if (pin_) (void)hipHostFree(pin_);
}

uint32_t *CopyOut::flags(size_t window) const { return (uint32_t *)(pin_ + 64) + (window & 1u) * MAX_FLAGS; }
char *CopyOut::half(size_t window) const { return pin_ + PIN_HEAD + (window & 1u) * cap_; }

/* windows_ and parts_ of a run, in the order in which the parts arrive.  Windows lie where the segments need bytes and
 * nowhere else: every window has parts, so that its half, and the flags that the caller waits for, are free for the
 * window after the next only when all of it has been taken. */
void CopyOut::plan(const std::vector<CopySeg> &segs, size_t total) {
  struct Span {
    uint32_t array;
    size_t off, bytes;
    uint32_t parts;
  };
  std::vector<Span> spans;
  std::vector<CopySeg> in;
  const size_t cut = total >= LARGE_RUN ? PART_LARGE : PART_SMALL;
  parts_.clear();
  for (uint32_t a = 0; a < arrays_->size(); a++) {
    in.clear();
    for (const CopySeg &s : segs)
      if (s.array == a) in.push_back(s);
    std::sort(in.begin(), in.end(), [](const CopySeg &x, const CopySeg &y) { return x.off < y.off; });
    const size_t first = spans.size();
    for (const CopySeg &s : in)
      for (size_t b = s.off, e = s.off + s.bytes; b < e;) {
        /* on in the array's last window while it has room and no chunk or more lies between */
        Span *w = spans.size() > first ? &spans.back() : nullptr;
        if (!w || b >= w->off + half_ || b - (w->off + w->bytes) >= COPY_CHUNK) {
          spans.push_back({a, b & ~(size_t)15, 0, 0});
          w = &spans.back();
        }
        char *dst = (char *)s.dst + (b - s.off);
        const size_t len = std::min(std::min(e, w->off + half_) - b, cut - (uintptr_t)dst % cut);
        parts_.push_back({(uint32_t)spans.size() - 1u, b - w->off, len, dst});
        w->bytes = b + len - w->off;
        w->parts++;
        b += len;
      }
  }
  windows_ = std::vector<Window>(spans.size());
  for (size_t k = 0; k < spans.size(); k++) {
    windows_[k].array = spans[k].array;
    windows_[k].off = spans[k].off;
    windows_[k].bytes = spans[k].bytes;
    windows_[k].stamp = ++stamp_;
    windows_[k].left = spans[k].parts;
  }
}

bool CopyOut::reserve(size_t total) {
  if (pin_ && cap_ >= half_) return true;
  if (!pin_ && !stats_ && total < PIN_LARGE && direct_ < PIN_AFTER * total) return false;
  char *p = nullptr;
  /* coherent: the flags and what is behind them are read while the kernel runs */
  if (hipHostMalloc((void **)&p, PIN_HEAD + 2 * half_, hipHostMallocCoherent) != hipSuccess) {
    (void)hipGetLastError();
    sent_ = 0; /* not again before as much has been sent again */
    half_ = cap_;
    return pin_ != nullptr;
  }
  if (pin_) (void)hipHostFree(pin_);
  memset(p, 0, PIN_HEAD);
  pin_ = p;
  cap_ = half_;
  touched_[0] = touched_[1] = 0;
  return true;
}

/* Has the destination's pages mapped until the first bytes arrive: a fresh
 * array's faults cost more than its copy (25 MB: 1.0 ms with huge pages and 4.7
 * without, against 0.9 of copying), and the device is busy meanwhile.  (Helpers
 * that map their own parts as well only wait for each other: a 2.8 MB image
 * 0.56 ms instead of 0.50.)  Then the pinned pages of the first two windows,
 * where they have not been touched yet. */
void CopyOut::map_pages(const std::vector<CopySeg> &segs) {
  const auto here = [this] { return __atomic_load_n(flags(0), __ATOMIC_RELAXED) == windows_[0].stamp; };
  bool can = true;
  for (const CopySeg &s : segs)
    for (size_t at = 0; can && s.bytes >= HELP_BYTES && at < s.bytes; at += HELP_BYTES) {
      if (here()) return;
      can = map_range((char *)s.dst + at, std::min(HELP_BYTES, s.bytes - at));
    }
  for (size_t w = 0; w < std::min<size_t>(2, windows_.size()); w++)
    for (; touched_[w] < windows_[w].bytes; touched_[w] += 4096) {
      if (here()) return;
      (void)*(const volatile char *)(half(w) + touched_[w]);
    }
}

void CopyOut::start_helpers() {
  if (tried_) return;
  tried_ = true;
  cpu_set_t set;
  const uint32_t cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? (uint32_t)CPU_COUNT(&set) : 1u;
  try {
    helpers_.reserve(HELPERS);
    for (uint32_t k = 0; k < std::min(HELPERS, cpus - 1u); k++) helpers_.emplace_back([this] { helper(); });
  } catch (const std::system_error &) { /* no more threads: those that started, or none */
  }
}

void CopyOut::helper() {
  uint64_t seen = 0;
  std::unique_lock<std::mutex> l(m_);
  for (;;) {
    cv_.wait(l, [&] { return stop_ || (open_ && run_ != seen); });
    if (stop_) return;
    seen = run_;
    inside_++;
    l.unlock();
    work(false);
    l.lock();
    inside_--;
  }
}

/* launches every window whose half is free again; the caller's thread only */
bool CopyOut::pump() {
  for (; launched_ < windows_.size(); launched_++) {
    const size_t w = launched_;
    if (w >= 2 && windows_[w - 2].left.load(std::memory_order_acquire)) return true;
    const Window &win = windows_[w];
    launch_copy_out(st_, (const char *)(*arrays_)[win.array].dev + win.off, half(w), win.bytes, flags(w), win.stamp,
                    w == 0 ? stats_ : nullptr, (uint64_t *)pin_);
    if (hipGetLastError() != hipSuccess) return false;
  }
  return true;
}

/* waits until the window's bytes [off, off + bytes) are in pinned memory */
bool CopyOut::landed(size_t window, size_t off, size_t bytes, bool caller) {
  const uint32_t stamp = windows_[window].stamp, *f = flags(window);
  uint32_t turns = 0;
  for (size_t k = off / COPY_CHUNK; k * COPY_CHUNK < off + bytes; k++)
    while (__atomic_load_n(f + k, __ATOMIC_ACQUIRE) != stamp) {
      if (failed_.load(std::memory_order_relaxed)) return false;
      pause_cpu();
      if (caller && ++turns % 256u == 0 && !alive(window, f + k)) return false;
    }
  return true;
}

/* the caller's look at the stream while it waits for a flag: one that has run
 * everything queued, or is broken, raises no more */
bool CopyOut::alive(size_t window, const uint32_t *flag) {
  hipError_t e = pump() ? hipStreamQuery(st_) : hipErrorLaunchFailure;
  if (e == hipErrorNotReady) return true;
  if (e == hipSuccess) {
    if (window >= launched_ || __atomic_load_n(flag, __ATOMIC_ACQUIRE) == windows_[window].stamp) return true;
    e = hipErrorUnknown;
  }
  failed_ = (int)e;
  return false;
}

void CopyOut::work(bool caller) {
  for (;;) {
    const uint32_t k = next_.fetch_add(1);
    if (k >= parts_.size()) return;
    const Part &p = parts_[k];
    if (!landed(p.window, p.off, p.bytes, caller)) return;
    memcpy(p.dst, half(p.window) + p.off, p.bytes);
    windows_[p.window].left.fetch_sub(1, std::memory_order_release);
  }
}

hipError_t CopyOut::run(hipStream_t st, const std::vector<CopyArray> &arrays, const std::vector<CopySeg> &all,
                        const uint64_t *stats, uint64_t stats_out[8]) {
  std::vector<CopySeg> segs;
  hipError_t err = hipSuccess;
  const auto direct = [&](const CopySeg &s) {
    if (err == hipSuccess)
      err = hipMemcpyAsync(s.dst, (const char *)arrays[s.array].dev + s.off, s.bytes, hipMemcpyDeviceToHost, st);
  };
  const bool in_turn = overlap(all);
  for (const CopySeg &s : all) {
    if (in_turn || known_to_runtime(s.dst)) direct(s);
    else segs.push_back(s);
  }
  st_ = st;
  arrays_ = &arrays;
  stats_ = stats;
  launched_ = 0;
  next_ = 0;
  failed_ = 0;
  size_t total = 0;
  for (const CopySeg &s : segs) total += s.bytes;
  half_ = cap_ == HALF_BYTES || (sent_ >= GROW_AFTER && total > 2 * HALF_FIRST) ? HALF_BYTES : HALF_FIRST;
  if (segs.empty() || !reserve(total)) {
    for (const CopySeg &s : segs) {
      direct(s);
      direct_ += s.bytes;
    }
    if (stats && err == hipSuccess) err = hipMemcpyAsync(stats_out, stats, 64, hipMemcpyDeviceToHost, st);
    const hipError_t e = hipStreamSynchronize(st);
    return err != hipSuccess ? err : e;
  }
  plan(segs, total);
  if (err == hipSuccess && !pump()) err = hipErrorLaunchFailure;
  if (err == hipSuccess) {
    map_pages(segs);
    sent_ += total;
    if (landed(0, 0, 1, true)) {
      if (total >= HELP_BYTES) {
        start_helpers();
        {
          std::lock_guard<std::mutex> l(m_);
          open_ = true;
          run_++;
        }
        cv_.notify_all();
      }
      work(true);
      /* the helpers' last parts, and windows that wait for them */
      for (size_t w = 0; w < windows_.size(); w++)
        for (uint32_t turns = 1; windows_[w].left.load(std::memory_order_acquire) && !failed_; turns++) {
          pause_cpu();
          if (turns % 256u) continue;
          const hipError_t e = pump() ? hipStreamQuery(st_) : hipErrorLaunchFailure;
          if (e != hipSuccess && e != hipErrorNotReady) failed_ = (int)e;
        }
      std::unique_lock<std::mutex> l(m_);
      open_ = false;
      while (inside_) {
        l.unlock();
        std::this_thread::yield();
        l.lock();
      }
    }
    err = (hipError_t)failed_.load();
  }
  const hipError_t e = hipStreamSynchronize(st);
  if (stats && err == hipSuccess) memcpy(stats_out, pin_, 64);
  return err != hipSuccess ? err : e;
}

}  // namespace clv

/*
 * copyout.h -- results from device arrays into the caller's memory.
 */
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace clv {

/* bytes behind one flag of launch_copy_out */
#define COPY_CHUNK ((size_t)65536)
/* k_copy_out (kernels.hip): `bytes` from device to pinned memory; flags[k] becomes `stamp` behind chunk k, and the 8
 * words at `stats` (may be null) go with the first */
void launch_copy_out(hipStream_t st, const void *src, void *dst, size_t bytes, uint32_t *flags, uint32_t stamp,
                     const uint64_t *stats, uint64_t *stats_out);

/* `bytes` of one device array from `off`, to the host address `dst` */
struct CopySeg {
  uint32_t array;
  size_t off, bytes;
  void *dst;
};

/* a device array of results (16-byte aligned, whole 4-byte words) */
struct CopyArray {
  const void *dev;
  size_t bytes;
};

/*
 * One context's way back to the host.  The caller's memory is pageable: the
 * runtime's own copy into it stages 1 MB at a time through pinned memory, a
 * launch, a wait and a host copy one after the other (17 GB/s into mapped
 * memory, 9 into fresh).  Here k_copy_out writes a window of the arrays to
 * pinned memory and raises a flag behind every 64 KB, the calling thread and
 * three helpers copy what has arrived on to the caller's memory meanwhile, and
 * two windows alternate, so that the link's 51 GB/s is what bounds a large copy.
 * While the device is still rendering, the calling thread has the destination's
 * pages mapped.  A context's first small probes go the runtime's way
 * (PIN_AFTER), its first large copies through small windows (HALF_FIRST).  A
 * first-hit probe and a normal map at 1080p (41 MB) 3.9 -> 1.8 ms, a 2.8 MB
 * image's call 0.68 -> 0.50 ms, 2 x 7 MB 3.6 -> 2.7 ms.  With one helper the
 * probe takes 2.2 ms, with seven 1.8; windows of 4 MB 2.0, of 2 MB 2.3.
 */
class CopyOut {
 public:
  ~CopyOut();
  /* Queues the copies on `st` behind the work there, waits for them, and reads
   * the 8 words at `stats` (may be null) with them.  The stream is idle after
   * any return. */
  hipError_t run(hipStream_t st, const std::vector<CopyArray> &arrays, const std::vector<CopySeg> &segs,
                 const uint64_t *stats, uint64_t stats_out[8]);

 private:
  struct Window {
    uint32_t array;
    size_t off, bytes;
    uint32_t stamp;
    std::atomic<uint32_t> left{0}; /* parts of it that are not copied yet */
  };
  struct Part { /* within one window */
    uint32_t window;
    size_t off, bytes; /* in the window */
    char *dst;
  };
  void plan(const std::vector<CopySeg> &segs, size_t total);
  bool reserve(size_t total);
  void map_pages(const std::vector<CopySeg> &segs);
  void start_helpers();
  void helper();
  void work(bool caller);
  bool landed(size_t window, size_t off, size_t bytes, bool caller);
  bool pump();
  bool alive(size_t window, const uint32_t *flag);
  uint32_t *flags(size_t window) const;
  char *half(size_t window) const;

  char *pin_ = nullptr; /* the stats, the flags of both halves, the halves */
  size_t cap_ = 0;      /* bytes of a half */
  size_t half_ = 0;     /* largest window of the current run */
  size_t touched_[2] = {0, 0}; /* bytes of the halves whose pages the caller has touched ahead */
  size_t direct_ = 0; /* bytes sent the runtime's way for want of pinned memory */
  size_t sent_ = 0;   /* bytes sent through the windows */
  uint32_t stamp_ = 0;
  /* the current run */
  hipStream_t st_ = nullptr;
  const std::vector<CopyArray> *arrays_ = nullptr;
  const uint64_t *stats_ = nullptr;
  std::vector<Window> windows_;
  std::vector<Part> parts_;
  size_t launched_ = 0;
  std::atomic<uint32_t> next_{0};
  std::atomic<int> failed_{0};
  /* helpers sleep until a run wakes them and join only while it lasts */
  std::mutex m_;
  std::condition_variable cv_;
  std::vector<std::thread> helpers_;
  bool tried_ = false, stop_ = false, open_ = false;
  uint64_t run_ = 0;
  uint32_t inside_ = 0;
};

}  // namespace clv

// eph_stage.hpp -- host side of the host-array hooks: copies between the
// caller's (pageable) arrays and device buffers through pinned staging
// chunks.  The host copy of a chunk is split over a few worker threads and
// overlaps the DMA of the neighbouring chunk; pageable memory would otherwise
// be copied by the runtime at about half the link rate (one host thread).
#pragma once

#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstddef>
#include <mutex>
#include <thread>
#include <vector>

namespace eph {

// Pinned host memory for the arrays of small calls.  The kernels read and
// write it in place, so that a call with several arrays takes one memcpy per
// array, one launch and one wait instead of a copy operation with a wait of
// its own per array (15 to 25 us each).  A call holds the arena from use() until
// its Use goes, so calls of several threads on one context or grid (a monitor
// that reads values while another thread steps) take turns: without that, one
// call's copy in would land in another's arrays.
class PinnedArena {
 public:
  // Beyond this many bytes a call takes the runtime's or the stager's copies.
  // That bounds the memory each context pins; it is not where the copies become
  // the faster: the four hooks of a step (us) with 1 / 2 / 4 / 8 MB here take
  // 200 / 200 / 200 / 204 for 4000 atoms, 505 / 308 / 311 / 309 for 10,976,
  // 890 / 847 / 722 / 624 for 32,000 and 1460 / 1430 / 1330 / 1109 for 55,296.
  static constexpr size_t kMax = size_t(1) << 20;
  // memory for one call, free to be written; empty when bytes > kMax or no
  // pinned memory is to be had
  class Use {
   public:
    Use() = default;
    double* get() const { return p_; }
    explicit operator bool() const { return p_ != nullptr; }

   private:
    friend class PinnedArena;
    std::unique_lock<std::mutex> lock_;
    double* p_ = nullptr;
  };
  PinnedArena() = default;
  PinnedArena(const PinnedArena&) = delete;
  PinnedArena& operator=(const PinnedArena&) = delete;
  ~PinnedArena();
  Use use(size_t bytes);
  // the work queued on s so far still reads the memory in use after it is given back
  hipError_t mark(const Use&, hipStream_t s);

 private:
  std::mutex m_;
  char* p_ = nullptr;
  size_t n_ = 0;
  hipEvent_t ev_ = nullptr;
  bool busy_ = false, failed_ = false;
};

class HostStager {
 public:
  HostStager() = default;
  HostStager(const HostStager&) = delete;
  HostStager& operator=(const HostStager&) = delete;
  ~HostStager();

  // pinned chunks of chunk_bytes and threads - 1 workers (threads >= 1)
  hipError_t init(int threads, size_t chunk_bytes);
  bool ready() const { return pin_[0] != nullptr; }

  // n bytes host -> device on stream s; returns once src may be reused (the
  // last chunk's DMA may still be in flight, ordered before later work on s)
  hipError_t to_device(void* dst, const void* src, size_t n, hipStream_t s);
  // n bytes device -> host after the work already enqueued on s; returns once
  // dst holds them
  hipError_t to_host(void* dst, const void* src, size_t n, hipStream_t s);

  // threads from EPH_HOST_THREADS (default 4, at most the hardware threads)
  static int default_threads();

 private:
  void copy(void* dst, const void* src, size_t n);  // split over the workers
  void work(int id);

  char* pin_[2] = {nullptr, nullptr};
  hipEvent_t ev_[2] = {nullptr, nullptr};
  size_t chunk_ = 0;
  int threads_ = 1;
  // worker pool: one job at a time, split into threads_ ranges
  std::vector<std::thread> pool_;
  std::mutex m_;
  std::condition_variable go_, done_;
  unsigned long gen_ = 0;
  int pending_ = 0;
  bool stop_ = false;
  char* job_dst_ = nullptr;
  const char* job_src_ = nullptr;
  size_t job_n_ = 0;
};

}  // namespace eph

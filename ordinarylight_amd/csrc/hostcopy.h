// Downloads of results into pageable host memory.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <memory>
#include <mutex>
#include <vector>

// A download runs in pieces: the copy engine brings one into a slot of a
// pinned ring while the caller copies the one before into the user's memory.
//
// The copy engine and not a kernel: a kernel fills the link better (33 MB into
// mapped pages in 1.0-1.2 ms, the copy engine in 1.4, a pageable hipMemcpy in
// 1.8), but its blocks wait for room beside a worker's traversal waves, which
// live as long as their launch: a 1 MB image fetched beside a rendering worker
// took 0.7 ms at the median and 11 ms at worst, here 0.1 and 0.2.
// Pieces are awaited by synchronising their stream, which follows the copy
// itself.  An event would go through the stream's hardware queue, which
// may be the one that a worker's steps use (there are four per process): each
// piece then waited for a step, 33 MB for 130 ms.
// Two pieces of 768 KB: 5 MB in 0.17 ms, 33 MB in 1.40 ms into mapped pages
// and 1.94 into fresh ones; 256 KB 0.26, 1.66 and 2.54, 1 MB 0.21, 1.29 and 2.39.
// The driver wipes freed device memory with the same engine: for some tens of
// milliseconds after 1 GB has been freed a piece takes 145 us instead of 22.
// Where a piece is that late and the device is idle, a kernel brings the rest
// (26 us a piece; 33 MB in 2.2 ms instead of 4.7).
// Pages of a fresh destination are populated by one call per part (27-66 us per
// MB, page faults take 100-220), or beforehand where the caller knows its
// destination while the device still works (Prefault).
//
// The contexts of a device share one HostCopier, freed with the last of them: a
// context made beside others finds a ring ready.  (With 8 MB of its own, made
// in its first frame, that frame took 1 to 4 ms longer; the first touch of
// pinned pages is the dearest, 0.34 ms per MB.)  A second ring is made when the
// first is in use, up to kRings; further downloads wait for one.
class HostCopier {
 public:
  static std::shared_ptr<HostCopier> of(int device);
  explicit HostCopier(int device) : device_(device) { idle_.reserve(kRings); }
  ~HostCopier() { (void)hipSetDevice(device_); }
  HostCopier(const HostCopier&) = delete;
  HostCopier& operator=(const HostCopier&) = delete;
  // Work that writes `dev` must have completed.  From any thread.  `idle`: a
  // stream that nothing else uses meanwhile, on a device with nothing else to
  // do; without one the copy runs on a stream of the ring's, made when it is
  // first needed (0.25 ms, 3.5 ms while the process has hardware queues left
  // to open).
  void download(void* dst, const void* dev, size_t bytes, hipStream_t idle);
  // Steps that the device's engines have queued, and their running workers.
  // Beside either a download keeps off its context's stream, where each piece
  // would wait for a step, and off the compute units.
  std::atomic<uint32_t> steps_queued{0}, workers{0};
  bool device_busy() const { return steps_queued != 0 || workers != 0; }
  // Maps the pages of [dst, dst + bytes) without changing their contents.
  // A hint: what cannot be mapped this way faults page by page when written.
  static void prefault(void* dst, size_t bytes);

 private:
  static constexpr size_t kPiece = size_t(768) << 10, kRings = 4;
  struct Ring {
    char* slots = nullptr;  // two pieces
    hipStream_t stream = nullptr;
    Ring();
    ~Ring();
  };
  std::unique_ptr<Ring> take();
  void give_back(std::unique_ptr<Ring> ring);
  static void through(char* slots, hipStream_t stream, bool idle, char* dst, const char* dev, size_t bytes);

  int device_;
  std::mutex mu_;
  std::condition_variable returned_;
  std::vector<std::unique_ptr<Ring>> idle_;
  size_t made_ = 0;  // idle and in use
};

// Populates destinations piece by piece while their data is being computed.
class Prefault {
 public:
  void add(void* dst, size_t bytes) {
    if (dst && bytes) ranges_.push_back({static_cast<char*>(dst), bytes});
  }
  // The next piece: 2 MB take 50-130 us, less than a step of a large frame.
  void advance() {
    if (ranges_.empty()) return;
    Range& r = ranges_.back();
    const size_t piece = size_t(2) << 20, n = r.bytes < piece ? r.bytes : piece;
    HostCopier::prefault(r.at, n);
    r.at += n;
    r.bytes -= n;
    if (r.bytes == 0) ranges_.pop_back();
  }

 private:
  struct Range {
    char* at;
    size_t bytes;
  };
  std::vector<Range> ranges_;
};

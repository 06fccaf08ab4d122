// Downloads of results into pageable host memory.
#pragma once

#include <hip/hip_runtime.h>

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
// Pieces are awaited by synchronising the ring's stream, which follows the
// copy itself.  An event would go through the stream's hardware queue, which
// may be the one that a worker's steps use (there are four per process): each
// piece then waited for a step, 33 MB for 130 ms.
// Two pieces of 768 KB: 5 MB in 0.17 ms, 33 MB in 1.40 ms into mapped pages
// and 1.94 into fresh ones; 256 KB 0.26, 1.66 and 2.54, 1 MB 0.21, 1.29 and 2.39.
// Pages of a fresh destination are populated by one call per part (27-66 us per
// MB, page faults take 100-220), or beforehand where the caller knows its
// destination while the device still works (Prefault).
//
// The contexts of a device share one HostCopier, freed with the last of them.
// Its ring costs what it saves over some 40 MB (a stream 0.2 ms, the
// allocation 0.1, the first touch of its pages 0.34 per MB; it saves 20 us per
// MB), so the first kPlain bytes are copied plainly, and a context made beside
// others finds the ring ready: with a ring of 8 MB per context, made in its
// first frame, that frame took 1 to 4 ms longer.  One download uses the ring at
// a time; one that finds it in use is copied plainly beside it.
class HostCopier {
 public:
  static std::shared_ptr<HostCopier> of(int device);
  explicit HostCopier(int device) : device_(device) {}
  ~HostCopier();
  HostCopier(const HostCopier&) = delete;
  HostCopier& operator=(const HostCopier&) = delete;
  // Work that writes `dev` must have completed.  From any thread.
  void download(void* dst, const void* dev, size_t bytes);
  // Maps the pages of [dst, dst + bytes) without changing their contents.
  // A hint: what cannot be mapped this way faults page by page when written.
  static void prefault(void* dst, size_t bytes);

 private:
  static constexpr size_t kPiece = size_t(768) << 10, kPlain = size_t(32) << 20;
  bool ring_for(size_t bytes);
  void through_ring(char* dst, const char* dev, size_t bytes);

  int device_;
  std::mutex use_;  // the ring, and the words below
  size_t plain_ = 0;  // bytes copied plainly before the ring was made
  hipStream_t stream_ = nullptr;
  char* ring_ = nullptr;  // two pieces
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

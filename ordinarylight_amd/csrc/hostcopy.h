// Downloads of results into pageable host memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <mutex>
#include <vector>

// A download runs in pieces: a kernel writes a piece into a slot of a pinned
// ring and raises a flag per 256 KB, and the caller copies each flagged part
// into the user's memory while the rest is on its way.  The link takes 54 GB/s
// from the kernel (33 MB in 0.62 ms), one host thread copies 50-80 GB/s
// between mapped pages.  Copies by the copy engine with an event each took
// 35 us per MB in pieces of 1 MB, a pageable hipMemcpy 55 us per MB warm; with
// the page faults of a fresh destination it took 100-220 us per MB, 2.7 ms of
// a 9.1 ms frame.  Pages are therefore populated by one call per part (27-66
// us per MB), or beforehand where the caller knows its destination while the
// device still works (Prefault).
// Downloads of one HostCopier run one after the other; it holds kRing bytes of
// pinned memory, made at its first download.
class HostCopier {
 public:
  explicit HostCopier(int device) : device_(device) {}
  ~HostCopier();
  HostCopier(const HostCopier&) = delete;
  HostCopier& operator=(const HostCopier&) = delete;
  // Work that writes `dev` must have completed.
  void download(void* dst, const void* dev, size_t bytes);
  // Maps the pages of [dst, dst + bytes) without changing their contents.
  // A hint: what cannot be mapped this way faults page by page when written.
  static void prefault(void* dst, size_t bytes);

 private:
  void prepare();
  void await(const uint32_t* flag, uint32_t value);

  int device_;
  std::mutex use_;  // one download at a time
  hipStream_t stream_ = nullptr;
  char* ring_ = nullptr;               // kSlots pieces
  uint32_t* flags_ = nullptr;          // pinned: per slot and part, the number of the piece that filled it
  uint32_t* arrived_ = nullptr;        // device: per slot and part, blocks done
  uint32_t piece_ = 0;                 // pieces issued so far (never 0 in a flag)
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

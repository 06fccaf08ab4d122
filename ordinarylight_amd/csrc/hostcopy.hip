// HostCopier: device results into pageable host memory.

#include "hostcopy.h"

#include <sys/mman.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <map>

#include "internal.h"

HostCopier::~HostCopier() {
  (void)hipSetDevice(device_);
  if (stream_) (void)hipStreamSynchronize(stream_);
  if (ring_) (void)hipHostFree(ring_);
  if (stream_) (void)hipStreamDestroy(stream_);
}

std::shared_ptr<HostCopier> HostCopier::of(int device) {
  static std::mutex mu;
  static auto& copiers = *new std::map<int, std::weak_ptr<HostCopier>>;
  std::lock_guard<std::mutex> g(mu);
  std::shared_ptr<HostCopier> c = copiers[device].lock();
  if (!c) copiers[device] = c = std::make_shared<HostCopier>(device);
  return c;
}

// Whether the ring serves this download, with `use_` held.  Without pinned
// memory for it the plain copies go on.
bool HostCopier::ring_for(size_t bytes) {
  if (ring_) return true;
  if (plain_ < kPlain) {
    plain_ += bytes;
    return false;
  }
  plain_ = 0;
  if (!stream_) OL_HIP_CHECK(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
  if (hipHostMalloc(reinterpret_cast<void**>(&ring_), 2 * kPiece, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    ring_ = nullptr;
  }
  return ring_ != nullptr;
}

void HostCopier::prefault(void* dst, size_t bytes) {
#if !defined(MADV_POPULATE_WRITE)
  constexpr int MADV_POPULATE_WRITE = 23;
#endif
  constexpr uintptr_t page = 4096;
  const uintptr_t first = reinterpret_cast<uintptr_t>(dst) & ~(page - 1);
  const uintptr_t last = (reinterpret_cast<uintptr_t>(dst) + bytes + page - 1) & ~(page - 1);
  if (bytes >= 4 * page) (void)madvise(reinterpret_cast<void*>(first), last - first, MADV_POPULATE_WRITE);
}

void HostCopier::download(void* dst, const void* dev, size_t bytes) {
  if (bytes == 0) return;
  OL_HIP_CHECK(hipSetDevice(device_));
  {
    std::unique_lock<std::mutex> use(use_, std::try_to_lock);
    if (use.owns_lock() && ring_for(bytes)) return through_ring(static_cast<char*>(dst), static_cast<const char*>(dev), bytes);
  }
  prefault(dst, bytes);
  OL_HIP_CHECK(hipMemcpy(dst, dev, bytes, hipMemcpyDeviceToHost));
}

void HostCopier::through_ring(char* dst, const char* dev, size_t bytes) {
  const size_t pieces = (bytes + kPiece - 1) / kPiece;
  auto length = [&](size_t k) { return std::min(kPiece, bytes - k * kPiece); };
  auto slot = [&](size_t k) { return ring_ + (k & 1u) * kPiece; };
  auto issue = [&](size_t k) {
    OL_HIP_CHECK(hipMemcpyAsync(slot(k), dev + k * kPiece, length(k), hipMemcpyDeviceToHost, stream_));
  };
  issue(0);
  for (size_t k = 0; k < pieces; ++k) {
    char* to = dst + k * kPiece;
    constexpr size_t part = size_t(256) << 10;
    for (size_t at = 0; at < length(k); at += part) prefault(to + at, std::min(part, length(k) - at));
    OL_HIP_CHECK(hipStreamSynchronize(stream_));
    if (k + 1 < pieces) issue(k + 1);
    std::memcpy(to, slot(k), length(k));
  }
}

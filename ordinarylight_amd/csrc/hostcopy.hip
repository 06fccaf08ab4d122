// HostCopier: device results into pageable host memory.

#include "hostcopy.h"

#include <sys/mman.h>

#include <algorithm>
#include <cstdint>
#include <cstring>

#include "internal.h"

HostCopier::~HostCopier() {
  (void)hipSetDevice(device_);
  if (stream_) (void)hipStreamSynchronize(stream_);
  if (ring_) (void)hipHostFree(ring_);
  if (stream_) (void)hipStreamDestroy(stream_);
}

void HostCopier::prepare() {
  OL_HIP_CHECK(hipSetDevice(device_));
  if (!stream_) OL_HIP_CHECK(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
  if (!ring_) OL_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&ring_), 2 * kPiece, hipHostMallocDefault));
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
  std::lock_guard<std::mutex> use(use_);
  prepare();
  const size_t pieces = (bytes + kPiece - 1) / kPiece;
  auto length = [&](size_t k) { return std::min(kPiece, bytes - k * kPiece); };
  auto slot = [&](size_t k) { return ring_ + (k & 1u) * kPiece; };
  auto issue = [&](size_t k) {
    OL_HIP_CHECK(hipMemcpyAsync(slot(k), static_cast<const char*>(dev) + k * kPiece, length(k), hipMemcpyDeviceToHost,
                                stream_));
  };
  issue(0);
  for (size_t k = 0; k < pieces; ++k) {
    char* to = static_cast<char*>(dst) + k * kPiece;
    constexpr size_t part = size_t(256) << 10;
    for (size_t at = 0; at < length(k); at += part) prefault(to + at, std::min(part, length(k) - at));
    OL_HIP_CHECK(hipStreamSynchronize(stream_));
    if (k + 1 < pieces) issue(k + 1);
    std::memcpy(to, slot(k), length(k));
  }
}

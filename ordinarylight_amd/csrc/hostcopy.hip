// HostCopier: device results into pageable host memory.

#include "hostcopy.h"

#include <sys/mman.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <map>

#include "internal.h"

std::shared_ptr<HostCopier> HostCopier::of(int device) {
  static std::mutex mu;
  static auto& copiers = *new std::map<int, std::weak_ptr<HostCopier>>;
  std::lock_guard<std::mutex> g(mu);
  std::shared_ptr<HostCopier> c = copiers[device].lock();
  if (!c) copiers[device] = c = std::make_shared<HostCopier>(device);
  return c;
}

HostCopier::Ring::Ring() {
  OL_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&slots), 2 * kPiece, hipHostMallocDefault));
}

HostCopier::Ring::~Ring() {
  (void)hipHostFree(slots);
  if (stream) (void)hipStreamDestroy(stream);
}

std::unique_ptr<HostCopier::Ring> HostCopier::take() {
  {
    std::unique_lock<std::mutex> g(mu_);
    returned_.wait(g, [&] { return !idle_.empty() || made_ < kRings; });
    if (!idle_.empty()) {
      std::unique_ptr<Ring> ring = std::move(idle_.back());
      idle_.pop_back();
      return ring;
    }
    ++made_;
  }
  try {
    return std::make_unique<Ring>();
  } catch (...) {
    {
      std::lock_guard<std::mutex> g(mu_);
      --made_;
    }
    returned_.notify_one();
    throw;
  }
}

void HostCopier::give_back(std::unique_ptr<Ring> ring) {
  {
    std::lock_guard<std::mutex> g(mu_);
    idle_.push_back(std::move(ring));
  }
  returned_.notify_one();
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

void HostCopier::download(void* dst, const void* dev, size_t bytes, hipStream_t idle) {
  if (bytes == 0) return;
  OL_HIP_CHECK(hipSetDevice(device_));
  struct Lease {
    HostCopier& copier;
    std::unique_ptr<Ring> ring;
    ~Lease() { copier.give_back(std::move(ring)); }
  } lease{*this, take()};
  Ring& ring = *lease.ring;
  if (!idle && !ring.stream) OL_HIP_CHECK(hipStreamCreateWithFlags(&ring.stream, hipStreamNonBlocking));
  const hipStream_t stream = idle ? idle : ring.stream;
  try {
    through(ring.slots, stream, static_cast<char*>(dst), static_cast<const char*>(dev), bytes);
  } catch (...) {
    (void)hipStreamSynchronize(stream);  // a piece may still be on its way into the ring
    throw;
  }
}

void HostCopier::through(char* slots, hipStream_t stream, char* dst, const char* dev, size_t bytes) {
  const size_t pieces = (bytes + kPiece - 1) / kPiece;
  auto length = [&](size_t k) { return std::min(kPiece, bytes - k * kPiece); };
  auto slot = [&](size_t k) { return slots + (k & 1u) * kPiece; };
  auto issue = [&](size_t k) {
    OL_HIP_CHECK(hipMemcpyAsync(slot(k), dev + k * kPiece, length(k), hipMemcpyDeviceToHost, stream));
  };
  issue(0);
  for (size_t k = 0; k < pieces; ++k) {
    char* to = dst + k * kPiece;
    constexpr size_t part = size_t(256) << 10;
    for (size_t at = 0; at < length(k); at += part) prefault(to + at, std::min(part, length(k) - at));
    OL_HIP_CHECK(hipStreamSynchronize(stream));
    if (k + 1 < pieces) issue(k + 1);
    std::memcpy(to, slot(k), length(k));
  }
}

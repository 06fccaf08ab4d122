// HostCopier: device results into pageable host memory.

#include "hostcopy.h"

#include <sys/mman.h>

#include <algorithm>
#include <chrono>
#include <cstdint>
#include <cstring>
#include <map>

#include "internal.h"

namespace {

constexpr uint32_t kBlock = 256, kBlockBytes = 16384;  // threads, and bytes copied by them

// One piece into pinned memory: 16 bytes a thread, bound by the link.
__global__ void __launch_bounds__(kBlock) k_piece(const char* __restrict__ src, char* __restrict__ dst, uint32_t bytes) {
  const uint32_t first = blockIdx.x * kBlockBytes, last = min(bytes, first + kBlockBytes);
  const uint32_t whole = max(last & ~15u, first);
#pragma unroll
  for (uint32_t k = 0; k < kBlockBytes; k += 16u * kBlock) {
    const uint32_t at = first + k + 16u * threadIdx.x;
    if (at < whole) *reinterpret_cast<float4*>(dst + at) = *reinterpret_cast<const float4*>(src + at);
  }
  if (threadIdx.x < last - whole) dst[whole + threadIdx.x] = src[whole + threadIdx.x];
}

}  // namespace

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
    through(ring.slots, stream, idle != nullptr, static_cast<char*>(dst), static_cast<const char*>(dev), bytes);
  } catch (...) {
    (void)hipStreamSynchronize(stream);  // a piece may still be on its way into the ring
    throw;
  }
}

void HostCopier::through(char* slots, hipStream_t stream, bool idle, char* dst, const char* dev, size_t bytes) {
  const size_t pieces = (bytes + kPiece - 1) / kPiece;
  auto length = [&](size_t k) { return std::min(kPiece, bytes - k * kPiece); };
  auto slot = [&](size_t k) { return slots + (k & 1u) * kPiece; };
  bool kernel = false;
  auto issue = [&](size_t k) {
    if (!kernel) {
      OL_HIP_CHECK(hipMemcpyAsync(slot(k), dev + k * kPiece, length(k), hipMemcpyDeviceToHost, stream));
      return;
    }
    hipLaunchKernelGGL(k_piece, dim3((unsigned)((length(k) + kBlockBytes - 1) / kBlockBytes)), dim3(kBlock), 0, stream,
                       dev + k * kPiece, slot(k), (uint32_t)length(k));
    OL_HIP_CHECK(hipGetLastError());
  };
  const bool may_launch = idle && (reinterpret_cast<uintptr_t>(dev) & 15u) == 0;
  issue(0);
  for (size_t k = 0; k < pieces; ++k) {
    char* to = dst + k * kPiece;
    constexpr size_t part = size_t(256) << 10;
    for (size_t at = 0; at < length(k); at += part) prefault(to + at, std::min(part, length(k) - at));
    const auto begin = std::chrono::steady_clock::now();
    OL_HIP_CHECK(hipStreamSynchronize(stream));
    kernel = kernel || (may_launch && std::chrono::steady_clock::now() - begin > std::chrono::microseconds(60));
    if (k + 1 < pieces) issue(k + 1);
    std::memcpy(to, slot(k), length(k));
  }
}

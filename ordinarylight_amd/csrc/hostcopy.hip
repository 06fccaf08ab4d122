// HostCopier: device results into pageable host memory.

#include "hostcopy.h"

#include <sys/mman.h>

#include <algorithm>
#include <cstring>

#include "internal.h"

namespace {

constexpr uint32_t kBlock = 256;                    // threads
constexpr uint32_t kBlockBytes = 32u << 10;         // copied per block: 8 x 16 bytes a thread
constexpr uint32_t kPart = 256u << 10;              // bytes per flag
constexpr uint32_t kPiece = 2u << 20;               // bytes per launch and slot
constexpr uint32_t kSlots = 4, kParts = kPiece / kPart;

// Copies `bytes` (at most a piece) into pinned memory and flags every part
// once all its blocks' stores have reached the host.  Bound by the link; 32 KB
// per block leave 30 blocks for 1 MB, enough to fill it.
__global__ void __launch_bounds__(kBlock) k_download(const char* __restrict__ src, char* __restrict__ dst,
                                                     uint32_t bytes, uint32_t* arrived, uint32_t* flags,
                                                     uint32_t number) {
  const uint32_t first = blockIdx.x * kBlockBytes, last = min(bytes, first + kBlockBytes);
  const uint32_t whole = last & ~15u;
#pragma unroll 8
  for (uint32_t at = first + 16u * threadIdx.x; at < whole; at += 16u * kBlock)
    *reinterpret_cast<float4*>(dst + at) = *reinterpret_cast<const float4*>(src + at);
  if (threadIdx.x < last - max(whole, first)) dst[max(whole, first) + threadIdx.x] = src[max(whole, first) + threadIdx.x];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x != 0) return;
  const uint32_t part = first / kPart;
  const uint32_t in_part = min(kPart, bytes - part * kPart);
  const uint32_t blocks = (in_part + kBlockBytes - 1u) / kBlockBytes;
  if (__hip_atomic_fetch_add(&arrived[part], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1u == blocks) {
    __hip_atomic_store(&arrived[part], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&flags[part], number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

}  // namespace

HostCopier::~HostCopier() {
  (void)hipSetDevice(device_);
  if (stream_) (void)hipStreamSynchronize(stream_);
  if (ring_) (void)hipHostFree(ring_);
  if (flags_) (void)hipHostFree(flags_);
  if (arrived_) (void)hipFree(arrived_);
  if (stream_) (void)hipStreamDestroy(stream_);
}

void HostCopier::prepare() {
  OL_HIP_CHECK(hipSetDevice(device_));
  if (!stream_) OL_HIP_CHECK(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
  if (!ring_) OL_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&ring_), size_t(kSlots) * kPiece, hipHostMallocDefault));
  if (!flags_) {
    OL_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&flags_), 4u * kSlots * kParts, hipHostMallocDefault));
    std::memset(flags_, 0, 4u * kSlots * kParts);
  }
  if (!arrived_) {
    void* p = nullptr;
    OL_HIP_CHECK(hipMalloc(&p, 4u * kSlots * kParts));
    arrived_ = static_cast<uint32_t*>(p);
    OL_HIP_CHECK(hipMemsetAsync(arrived_, 0, 4u * kSlots * kParts, stream_));
  }
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

// Spins until the device has raised the flag, or has stopped without it.
void HostCopier::await(const uint32_t* flag, uint32_t value) {
  for (uint32_t spin = 1;; ++spin) {
    if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == value) return;
    if (spin % 4096u == 0u) {
      const hipError_t e = hipStreamQuery(stream_);
      if (e == hipErrorNotReady) continue;
      if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == value) return;
      OL_HIP_CHECK(e);
      throw OlError{-4, "download: the device finished without delivering the data"};
    }
  }
}

void HostCopier::download(void* dst, const void* dev, size_t bytes) {
  if (bytes == 0) return;
  std::lock_guard<std::mutex> use(use_);
  prepare();
  if (reinterpret_cast<uintptr_t>(dev) & 15u) {  // not an allocation of its own; k_download reads 16 bytes at once
    OL_HIP_CHECK(hipMemcpy(dst, dev, bytes, hipMemcpyDeviceToHost));
    return;
  }
  const size_t pieces = (bytes + kPiece - 1) / kPiece;
  auto length = [&](size_t k) { return (uint32_t)std::min<size_t>(kPiece, bytes - k * kPiece); };
  size_t issued = 0;
  uint32_t numbers[kSlots] = {};
  for (size_t k = 0; k < pieces; ++k) {
    // Slots are taken in turn by this download: piece k - kSlots has been
    // copied out when piece k is issued.
    for (; issued < std::min(pieces, k + kSlots); ++issued) {
      const size_t slot = issued % kSlots;
      if (++piece_ == 0u) ++piece_;
      numbers[slot] = piece_;
      hipLaunchKernelGGL(k_download, dim3((length(issued) + kBlockBytes - 1) / kBlockBytes), dim3(kBlock), 0, stream_,
                         static_cast<const char*>(dev) + issued * kPiece, ring_ + slot * kPiece, length(issued),
                         arrived_ + slot * kParts, flags_ + slot * kParts, piece_);
      OL_HIP_CHECK(hipGetLastError());
    }
    const size_t slot = k % kSlots;
    char* to = static_cast<char*>(dst) + k * kPiece;
    for (uint32_t part = 0; part * kPart < length(k); ++part) {
      const uint32_t at = part * kPart, n = std::min(kPart, length(k) - at);
      prefault(to + at, n);
      await(flags_ + slot * kParts + part, numbers[slot]);
      std::memcpy(to + at, ring_ + slot * kPiece + at, n);
    }
  }
}

// Device scratch of one call whose caller brings none (qk_matmul, the FFN
// entry points at M > 8), from a small cache of blocks.
//
// A hipMallocAsync / hipFreeAsync pair costs 15 us of host time when every
// call asks for one size and 35-50 us when sizes alternate (200 us with a
// device synchronisation between the calls), so a layer's seven projections
// at M = 200 spent 1.0 of their 1.3 ms in allocation. A cached block costs an
// event record and a wait, about 2 us each (a layer's calls at M = 200: 1203 ->
// 289 us; at M = 23: 387 -> 150).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace qk {

// At most kScratchBlocks blocks per device, of 16 or 64 MiB; larger requests,
// requests while a block cannot be had, calls on the per-thread default stream
// and calls under stream capture (whose graph may be replayed beside later
// calls) are stream-ordered allocations.
constexpr int kScratchBlocks = 8;
constexpr size_t kScratchSmall = size_t{16} << 20;
constexpr size_t kScratchLarge = size_t{64} << 20;

// Bytes of the block that serves a request (0: not served from the cache).
constexpr size_t scratch_class(size_t bytes) {
  return bytes <= kScratchSmall ? kScratchSmall : bytes <= kScratchLarge ? kScratchLarge : 0;
}

// Owns the scratch of one call on one stream: nothing enqueued before get()
// or after the destructor may use it.
class Scratch {
 public:
  explicit Scratch(hipStream_t stream) : stream_(stream) {}
  ~Scratch();
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
  // Sets ptr to `bytes` of device memory (256-byte aligned).
  hipError_t get(size_t bytes, void*& ptr);

 private:
  hipStream_t stream_;
  void* ptr_ = nullptr;
  int device_ = -1, block_ = -1;  // block_ < 0: an allocation of this call alone
};

// Waits for the current device and frees its cached blocks (those not held
// by a call that another thread is making).
hipError_t release_scratch();

}  // namespace qk

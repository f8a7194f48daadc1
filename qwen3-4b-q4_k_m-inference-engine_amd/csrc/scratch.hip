// The scratch cache (scratch.hpp). A block belongs to the stream that used it
// last and goes to that stream's next call; another stream gets it only once
// its event has completed, so calls on different streams never wait for each
// other. The stream waits for the block's event even when the handle is the
// one that recorded it: a destroyed stream's handle may name a new stream.
// (hipStreamPerThread is one handle for a stream of each thread, which would
// wait for each other so: its calls allocate stream-ordered.)
// A block is held by one call at a time (busy), so threads that share a
// stream, and calls that make another call, take different blocks.
#include "scratch.hpp"

#include <mutex>

namespace qk {
namespace {

struct Block {
  void* ptr = nullptr;
  size_t bytes = 0;
  hipEvent_t event = nullptr;   // recorded when the last call's work was enqueued
  hipStream_t stream = nullptr;  // that call's stream
  bool busy = false;
};

constexpr int kMaxDevices = 64;
std::mutex g_mutex;
Block g_blocks[kMaxDevices][kScratchBlocks];

// Drops the error that a failed call of this file left, unless one of the
// caller's was pending already.
struct OwnErrors {
  const bool clean = hipPeekAtLastError() == hipSuccess;
  void drop() const {
    if (clean) (void)hipGetLastError();
  }
};

// hipEventQuery, allowed while another stream is being captured: in any
// capture mode but the relaxed one a query ends that capture with an error,
// whichever event it asks about.
hipError_t query(hipEvent_t event) {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  const bool exchanged = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
  const hipError_t status = hipEventQuery(event);
  if (exchanged) (void)hipThreadExchangeStreamCaptureMode(&mode);
  return status;
}

// An idle block for `stream`: its own of the right size or any of its own,
// an unused one, one whose work is done; else -1. Called with the lock held.
int choose(Block (&blocks)[kScratchBlocks], hipStream_t stream, size_t bytes) {
  int own = -1, unused = -1;
  for (int i = 0; i < kScratchBlocks; ++i) {
    const Block& b = blocks[i];
    if (b.busy) continue;
    if (b.ptr && b.stream == stream) {
      if (b.bytes >= bytes) return i;
      own = i;
    } else if (!b.ptr && unused < 0) {
      unused = i;
    }
  }
  if (own >= 0) return own;
  if (unused >= 0) return unused;
  const OwnErrors errors;
  for (int i = 0; i < kScratchBlocks; ++i)
    if (!blocks[i].busy && query(blocks[i].event) == hipSuccess) return i;
  errors.drop();  // "not ready"
  return -1;
}

}  // namespace

hipError_t Scratch::get(size_t bytes, void*& ptr) {
  const size_t size = scratch_class(bytes);
  hipStreamCaptureStatus capture = hipStreamCaptureStatusActive;
  int device = -1;
  const OwnErrors errors;
  if (size != 0 && stream_ != hipStreamPerThread && hipStreamIsCapturing(stream_, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone &&
      hipGetDevice(&device) == hipSuccess && device >= 0 && device < kMaxDevices) {
    std::lock_guard<std::mutex> lock(g_mutex);
    Block(&blocks)[kScratchBlocks] = g_blocks[device];
    const int i = choose(blocks, stream_, size);
    if (i >= 0) {
      Block& b = blocks[i];
      hipError_t error = hipSuccess;
      if (!b.event) error = hipEventCreateWithFlags(&b.event, hipEventDisableTiming);
      if (error == hipSuccess && b.ptr) error = hipStreamWaitEvent(stream_, b.event, 0);
      if (error == hipSuccess && b.bytes < size) {
        if (b.ptr) error = hipFreeAsync(b.ptr, stream_);
        b.ptr = nullptr;
        b.bytes = 0;
        if (error == hipSuccess) error = hipMallocAsync(&b.ptr, size, stream_);
        if (error == hipSuccess)
          b.bytes = size;
        else
          b.ptr = nullptr;
      }
      if (error == hipSuccess) {
        b.busy = true;
        b.stream = stream_;
        device_ = device;
        block_ = i;
        ptr = ptr_ = b.ptr;
        return hipSuccess;
      }
    }
  }
  errors.drop();
  const hipError_t error = hipMallocAsync(&ptr_, bytes, stream_);
  if (error != hipSuccess) ptr_ = nullptr;
  ptr = ptr_;
  return error;
}

Scratch::~Scratch() {
  if (!ptr_) return;
  if (block_ < 0) {
    (void)hipFreeAsync(ptr_, stream_);
    return;
  }
  std::lock_guard<std::mutex> lock(g_mutex);
  Block& b = g_blocks[device_][block_];
  const OwnErrors errors;
  if (hipEventRecord(b.event, stream_) != hipSuccess) {  // not orderable: give it back instead
    errors.drop();
    (void)hipFreeAsync(b.ptr, stream_);
    b.ptr = nullptr;
    b.bytes = 0;
  }
  b.busy = false;
}

hipError_t release_scratch() {
  int device = -1;
  hipError_t error = hipGetDevice(&device);
  if (error != hipSuccess || device < 0 || device >= kMaxDevices) return error;
  std::lock_guard<std::mutex> lock(g_mutex);
  error = hipDeviceSynchronize();
  for (Block& b : g_blocks[device]) {
    if (error != hipSuccess || b.busy || !b.ptr) continue;
    error = hipFreeAsync(b.ptr, nullptr);
    if (error != hipSuccess) break;
    b.ptr = nullptr;
    b.bytes = 0;
  }
  // (a stream-ordered free returns the memory to the pool; the pool gives it
  // back when its stream is next synchronised)
  if (error == hipSuccess) error = hipStreamSynchronize(nullptr);
  return error;
}

}  // namespace qk

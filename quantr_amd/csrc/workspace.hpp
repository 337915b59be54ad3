// workspace.hpp — device and pinned host memory of the entry points: buffers that grow, blocks
// kept between calls, and uploads that are not waited for.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <string>

#include "engine.hpp"

namespace qr {

inline void hip_check(hipError_t e, const char* what) {
  if (e == hipSuccess) return;
  if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation)
    throw Error{QR_ERR_OOM, std::string(what) + ": " + hipGetErrorString(e)};
  throw Error{QR_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e)};
}

// Device memory with what the library keeps for later calls given back before it fails.
hipError_t device_malloc(void** p, size_t bytes);

// A block of device memory held for one call without a state of its own. Blocks are kept for later
// calls (allocating and freeing them took longer than the call's kernels): at most 8 of them and
// 256 MB, or kDeviceIdleBytes while no state or batch lives, and all are given back when an
// allocation would fail. Larger ones are not kept. The holder's work on the block is done before it
// lets go. 500 re-simulated shots of 12 qubits, whose own states take 33 MB, while no other lives: 2.27 ms with
// 64 MB kept, 2.34 with 4, 2.44 with none.
constexpr size_t kDeviceIdleBytes = 4ull << 20;
class DeviceLease {
 public:
  DeviceLease() = default;
  ~DeviceLease();
  DeviceLease(const DeviceLease&) = delete;
  DeviceLease& operator=(const DeviceLease&) = delete;
  void reserve(size_t bytes);  // at least this size; what it held is lost
  void* p = nullptr;

 private:
  void release();
  size_t cap_ = 0;
  int device_ = 0;
};

// Device buffer that grows on demand.
struct DevBuf {
  void* p = nullptr;
  size_t cap = 0;
  void reserve(size_t bytes) {
    if (bytes <= cap) return;
    if (p) hip_check(hipFree(p), "hipFree");
    p = nullptr;
    cap = 0;
    size_t want = std::max<size_t>(bytes, 1 << 16);
    hip_check(device_malloc(&p, want), "hipMalloc (workspace)");
    cap = want;
  }
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
};

// A block of pinned host memory, which kernels and copies reach directly, held for one call.
// Blocks are kept for later calls (pinning a new one takes longer than a small call): at most 8 of
// them and kPinnedBytes, or kPinnedIdleBytes while no state or batch lives: programs that make a state for
// each circuit would else pin and free its blocks every time (create, apply, 500 draws, destroy,
// complex128, 10 / 16 / 20 qubits: 147 / 412 / 510 us without them, 112 / 256 / 355 with; an
// expectation in place of the draws, 12 qubits: 360 and 256).
// Nor is more pinned for a call's data: draws are taken in slices, and blocks that only copies reach
// are ordinary memory beyond kPinnedBytes.
constexpr size_t kPinnedBytes = 64ull << 20, kPinnedIdleBytes = 4ull << 20;
class PinnedLease {
 public:
  PinnedLease() = default;
  explicit PinnedLease(size_t bytes) { reserve(bytes); }
  ~PinnedLease() { release(); }
  PinnedLease(const PinnedLease&) = delete;
  PinnedLease& operator=(const PinnedLease&) = delete;
  void reserve(size_t bytes);  // at least this size; what it held is lost
  // The same for a block that only copies reach: ordinary memory beyond kPinnedBytes, and where no
  // more can be pinned.
  void reserve_for_copies(size_t bytes);
  void release();  // back to the kept blocks
  uint8_t* data() const { return (uint8_t*)p_; }

 private:
  void* p_ = nullptr;
  size_t cap_ = 0;
  bool plain_ = false;  // ordinary memory
};
void pinned_state_created();    // one more state or batch lives
void pinned_state_destroyed();  // one less; the last one, its own blocks let go of, leaves the idle bounds

// Uploads of host data onto a stream without waiting for it: two blocks in turn, each reused once its
// last copy is done. The owner's stream is idle before it is destroyed.
class Uploader {
 public:
  ~Uploader();
  // A block of `bytes` to fill, then send() it to dst on stream s.
  uint8_t* begin(size_t bytes);
  void send(void* dst, size_t bytes, hipStream_t s);
  // Lets go of both blocks; their copies are done.
  void release() {
    for (PinnedLease& b : buf_) b.release();
    busy_[0] = busy_[1] = false;
  }

 private:
  PinnedLease buf_[2];
  hipEvent_t ev_[2] = {nullptr, nullptr};
  bool busy_[2] = {false, false};
  int at_ = 0;
};

}  // namespace qr

// workspace.cpp — the blocks of device and pinned host memory kept between calls.
#include "workspace.hpp"

#include <algorithm>
#include <cstdlib>
#include <exception>
#include <mutex>
#include <new>

namespace qr {

// ---- pinned host memory -------------------------------------------------------------------
namespace {
constexpr size_t kKeep = 8;
struct PinnedBlock {
  void* p;
  size_t cap;
};
std::mutex g_pin_mu;
uint64_t g_pin_states = 0;

// Blocks nobody holds, at most kKeep of them between calls. Nothing here allocates: blocks come back
// in destructors.
template <class Block>
struct Kept {
  Block block[kKeep + 1];
  size_t count = 0, held = 0;
  void take_out(size_t i) {
    held -= block[i].cap;
    block[i] = block[--count];
  }
  void add(const Block& b) {  // count <= kKeep
    block[count++] = b;
    held += b.cap;
  }
  // Takes out blocks until no more than kKeep of at most `bytes` are left, the smallest first (a large
  // block is the one that costs most to make again), or the largest first where little may stay
  // (one of them would push out all that small calls use). drop[kKeep + 1] receives them.
  size_t trim(size_t bytes, bool largest_first, Block* drop) {
    size_t n = 0;
    while (count > kKeep || held > bytes) {
      size_t out = 0;
      for (size_t i = 1; i < count; ++i)
        if (largest_first ? block[i].cap > block[out].cap : block[i].cap < block[out].cap) out = i;
      drop[n++] = block[out];
      take_out(out);
    }
    return n;
  }
};
Kept<PinnedBlock> g_pinned;

void pinned_give_back(void* p, size_t cap) {
  PinnedBlock drop[kKeep + 1] = {{p, cap}};
  size_t n = 1;
  {
    std::lock_guard<std::mutex> lk(g_pin_mu);
    const bool idle = g_pin_states == 0;
    const size_t most = idle ? kPinnedIdleBytes : kPinnedBytes;
    if (cap <= most) {
      g_pinned.add(drop[0]);
      n = g_pinned.trim(most, idle, drop);
    }
  }
  for (size_t i = 0; i < n; ++i) (void)hipHostFree(drop[i].p);
}
}  // namespace

void pinned_state_created() {
  std::lock_guard<std::mutex> lk(g_pin_mu);
  ++g_pin_states;
}

void PinnedLease::reserve(size_t bytes) {
  if (bytes <= cap_ && !plain_) return;
  release();
  {
    std::lock_guard<std::mutex> lk(g_pin_mu);
    size_t best = g_pinned.count;
    for (size_t i = 0; i < g_pinned.count; ++i)
      if (g_pinned.block[i].cap >= bytes && (best == g_pinned.count || g_pinned.block[i].cap < g_pinned.block[best].cap))
        best = i;
    if (best < g_pinned.count) {
      p_ = g_pinned.block[best].p;
      cap_ = g_pinned.block[best].cap;
      g_pinned.take_out(best);
      return;
    }
  }
  // rounded, so that calls of about one size share a block: to a power of two, from 4 MB on to whole MB
  constexpr size_t MB = 1 << 20;
  size_t want = 1 << 16;
  while (want < bytes && want < 4 * MB) want *= 2;
  if (want < bytes) want = (bytes + MB - 1) / MB * MB;
  hipError_t e = hipHostMalloc(&p_, want, hipHostMallocPortable | hipHostMallocCoherent);
  if (e != hipSuccess) {  // without the blocks nobody holds, and no more than is asked for
    (void)hipGetLastError();
    PinnedBlock drop[kKeep + 1];
    size_t n = 0;
    {
      std::lock_guard<std::mutex> lk(g_pin_mu);
      n = g_pinned.trim(0, true, drop);
    }
    for (size_t i = 0; i < n; ++i) (void)hipHostFree(drop[i].p);
    want = bytes;
    e = hipHostMalloc(&p_, want, hipHostMallocPortable | hipHostMallocCoherent);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      p_ = nullptr;
    }
  }
  hip_check(e, "hipHostMalloc");
  cap_ = want;
}

void PinnedLease::reserve_for_copies(size_t bytes) {
  if (bytes <= cap_) return;
  if (bytes <= kPinnedBytes) {
    try {
      reserve(bytes);
      return;
    } catch (const Error&) {  // pinned memory is short: copies take other memory too
    }
  }
  release();
  p_ = std::malloc(bytes);
  if (!p_) throw std::bad_alloc();
  cap_ = bytes;
  plain_ = true;
}

void PinnedLease::release() {
  if (!p_) return;
  // a call that ends in an error may leave work in flight on the block: hipHostFree waits for it
  if (plain_) {
    if (std::uncaught_exceptions()) (void)hipDeviceSynchronize();
    std::free(p_);
  } else if (std::uncaught_exceptions())
    (void)hipHostFree(p_);
  else
    pinned_give_back(p_, cap_);
  p_ = nullptr;
  cap_ = 0;
  plain_ = false;
}

// ---- device memory kept between calls -----------------------------------------------------
namespace {
constexpr size_t kDeviceBytes = 256ull << 20;
struct DeviceBlock {
  void* p;
  size_t cap;
  int device;
};
std::mutex g_dev_mu;
Kept<DeviceBlock> g_device_blocks;
}  // namespace

void pinned_state_destroyed() {
  PinnedBlock drop[kKeep + 1];
  DeviceBlock drop_dev[kKeep + 1];
  size_t n = 0, nd = 0;
  {
    std::scoped_lock lk(g_pin_mu, g_dev_mu);
    if (--g_pin_states == 0) {
      n = g_pinned.trim(kPinnedIdleBytes, true, drop);
      nd = g_device_blocks.trim(kDeviceIdleBytes, true, drop_dev);
    }
  }
  for (size_t i = 0; i < n; ++i) (void)hipHostFree(drop[i].p);
  for (size_t i = 0; i < nd; ++i) (void)hipFree(drop_dev[i].p);
}

hipError_t device_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory && e != hipErrorMemoryAllocation) return e;
  DeviceBlock drop[kKeep + 1];
  size_t n = 0;
  {
    std::lock_guard<std::mutex> lk(g_dev_mu);
    n = g_device_blocks.trim(0, true, drop);
  }
  (void)hipGetLastError();  // it is returned, not left for the check of the next launch
  if (n == 0) return e;
  for (size_t i = 0; i < n; ++i) (void)hipFree(drop[i].p);
  e = hipMalloc(p, bytes);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

void DeviceLease::reserve(size_t bytes) {
  if (bytes <= cap_) return;
  release();
  hip_check(hipGetDevice(&device_), "hipGetDevice");
  {
    std::lock_guard<std::mutex> lk(g_dev_mu);
    size_t best = g_device_blocks.count;
    for (size_t i = 0; i < g_device_blocks.count; ++i) {
      const DeviceBlock& b = g_device_blocks.block[i];
      if (b.device == device_ && b.cap >= bytes &&
          (best == g_device_blocks.count || b.cap < g_device_blocks.block[best].cap))
        best = i;
    }
    if (best < g_device_blocks.count) {
      p = g_device_blocks.block[best].p;
      cap_ = g_device_blocks.block[best].cap;
      g_device_blocks.take_out(best);
      return;
    }
  }
  size_t want = 1 << 16;
  while (want < bytes && want < kDeviceBytes) want *= 2;
  want = std::max(want, bytes);
  hipError_t e = device_malloc(&p, want);
  if (e != hipSuccess && want > bytes) {  // short of memory: no room for later calls then
    want = bytes;
    e = device_malloc(&p, want);
  }
  if (e != hipSuccess) p = nullptr;
  hip_check(e, "hipMalloc (workspace)");
  cap_ = want;
}

void DeviceLease::release() {
  if (!p) return;
  DeviceBlock drop[kKeep + 1] = {{p, cap_, device_}};
  size_t n = 1;
  if (!std::uncaught_exceptions()) {  // after an error, hipFree waits for what may still run
    std::scoped_lock lk(g_pin_mu, g_dev_mu);
    const bool idle = g_pin_states == 0;
    const size_t most = idle ? kDeviceIdleBytes : kDeviceBytes;
    if (cap_ <= most) {
      g_device_blocks.add(drop[0]);
      n = g_device_blocks.trim(most, idle, drop);
    }
  }
  for (size_t i = 0; i < n; ++i) (void)hipFree(drop[i].p);
  p = nullptr;
  cap_ = 0;
}

DeviceLease::~DeviceLease() { release(); }

Uploader::~Uploader() {
  for (hipEvent_t e : ev_)
    if (e) (void)hipEventDestroy(e);
}

uint8_t* Uploader::begin(size_t bytes) {
  at_ ^= 1;
  if (busy_[at_]) hip_check(hipEventSynchronize(ev_[at_]), "hipEventSynchronize");
  busy_[at_] = false;
  buf_[at_].reserve_for_copies(std::max<size_t>(bytes, 1));
  return buf_[at_].data();
}

void Uploader::send(void* dst, size_t bytes, hipStream_t s) {
  if (!ev_[at_]) hip_check(hipEventCreateWithFlags(&ev_[at_], hipEventDisableTiming), "hipEventCreate");
  hip_check(hipMemcpyAsync(dst, buf_[at_].data(), bytes, hipMemcpyHostToDevice, s), "hipMemcpyAsync H2D");
  hip_check(hipEventRecord(ev_[at_], s), "hipEventRecord");
  busy_[at_] = true;
}

}  // namespace qr

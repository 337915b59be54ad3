// workspace.cpp — the blocks of device and pinned host memory kept between calls.
#include "workspace.hpp"

#include <algorithm>
#include <exception>
#include <mutex>
#include <vector>

namespace qr {

// ---- pinned host memory -------------------------------------------------------------------
namespace {
constexpr size_t kPinnedKeep = 8, kPinnedBytes = 64ull << 20;
struct PinnedBlock {
  void* p;
  size_t cap;
};
std::mutex g_pin_mu;
std::vector<PinnedBlock> g_pinned;  // kept blocks, none in use
uint64_t g_pin_states = 0;

// Adds a block to the kept ones and takes out the smallest until no more than `keep` of at most
// `bytes` are left (a large block is the one that costs most to make again); returns those.
template <class Block>
std::vector<Block> keep_block(std::vector<Block>& kept, const Block& b, size_t keep, size_t bytes) {
  std::vector<Block> drop;
  if (b.cap > bytes) {
    drop.push_back(b);
    return drop;
  }
  kept.push_back(b);
  size_t held = 0;
  for (const Block& x : kept) held += x.cap;
  while (kept.size() > keep || held > bytes) {
    auto least = std::min_element(kept.begin(), kept.end(), [](const Block& x, const Block& y) { return x.cap < y.cap; });
    held -= least->cap;
    drop.push_back(*least);
    kept.erase(least);
  }
  return drop;
}

void pinned_give_back(void* p, size_t cap) {
  std::vector<PinnedBlock> drop;
  {
    std::lock_guard<std::mutex> lk(g_pin_mu);
    drop = keep_block(g_pinned, PinnedBlock{p, cap}, kPinnedKeep, kPinnedBytes);
  }
  for (const PinnedBlock& b : drop) (void)hipHostFree(b.p);
}
}  // namespace

void pinned_state_created() {
  std::lock_guard<std::mutex> lk(g_pin_mu);
  ++g_pin_states;
}

void PinnedLease::reserve(size_t bytes) {
  if (bytes <= cap_) return;
  if (p_) pinned_give_back(p_, cap_);
  p_ = nullptr;
  cap_ = 0;
  {
    std::lock_guard<std::mutex> lk(g_pin_mu);
    size_t best = g_pinned.size();
    for (size_t i = 0; i < g_pinned.size(); ++i)
      if (g_pinned[i].cap >= bytes && (best == g_pinned.size() || g_pinned[i].cap < g_pinned[best].cap)) best = i;
    if (best < g_pinned.size()) {
      p_ = g_pinned[best].p;
      cap_ = g_pinned[best].cap;
      g_pinned.erase(g_pinned.begin() + best);
      return;
    }
  }
  size_t want = 1 << 16;
  while (want < bytes) want *= 2;
  hip_check(hipHostMalloc(&p_, want, hipHostMallocPortable | hipHostMallocCoherent), "hipHostMalloc");
  cap_ = want;
}

void PinnedLease::release() {
  if (!p_) return;
  // a call that ends in an error may leave work in flight on the block: hipHostFree waits for it
  if (std::uncaught_exceptions()) (void)hipHostFree(p_);
  else pinned_give_back(p_, cap_);
  p_ = nullptr;
  cap_ = 0;
}

// ---- device memory kept between calls -----------------------------------------------------
namespace {
constexpr size_t kDeviceKeep = 8, kDeviceBytes = 256ull << 20;
struct DeviceBlock {
  void* p;
  size_t cap;
  int device;
};
std::mutex g_dev_mu;
std::vector<DeviceBlock> g_device_blocks;  // kept blocks, none in use
}  // namespace

void pinned_state_destroyed() {
  std::vector<PinnedBlock> drop;
  std::vector<DeviceBlock> drop_dev;
  {
    std::scoped_lock lk(g_pin_mu, g_dev_mu);
    if (--g_pin_states == 0) {
      drop.swap(g_pinned);
      drop_dev.swap(g_device_blocks);
    }
  }
  for (const PinnedBlock& b : drop) (void)hipHostFree(b.p);
  for (const DeviceBlock& b : drop_dev) (void)hipFree(b.p);
}

hipError_t device_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory && e != hipErrorMemoryAllocation) return e;
  std::vector<DeviceBlock> drop;
  {
    std::lock_guard<std::mutex> lk(g_dev_mu);
    drop.swap(g_device_blocks);
  }
  if (drop.empty()) return e;
  (void)hipGetLastError();
  for (const DeviceBlock& b : drop) (void)hipFree(b.p);
  return hipMalloc(p, bytes);
}

void DeviceLease::reserve(size_t bytes) {
  if (bytes <= cap_) return;
  release();
  hip_check(hipGetDevice(&device_), "hipGetDevice");
  {
    std::lock_guard<std::mutex> lk(g_dev_mu);
    size_t best = g_device_blocks.size();
    for (size_t i = 0; i < g_device_blocks.size(); ++i) {
      const DeviceBlock& b = g_device_blocks[i];
      if (b.device == device_ && b.cap >= bytes && (best == g_device_blocks.size() || b.cap < g_device_blocks[best].cap))
        best = i;
    }
    if (best < g_device_blocks.size()) {
      p = g_device_blocks[best].p;
      cap_ = g_device_blocks[best].cap;
      g_device_blocks.erase(g_device_blocks.begin() + best);
      return;
    }
  }
  size_t want = 1 << 16;
  while (want < bytes && want < kDeviceBytes) want *= 2;
  want = std::max(want, bytes);
  hip_check(device_malloc(&p, want), "hipMalloc (workspace)");
  cap_ = want;
}

void DeviceLease::release() {
  if (!p) return;
  std::vector<DeviceBlock> drop(1, DeviceBlock{p, cap_, device_});
  if (!std::uncaught_exceptions()) {  // after an error, hipFree waits for what may still run
    std::lock_guard<std::mutex> lk(g_dev_mu);
    drop = keep_block(g_device_blocks, drop[0], kDeviceKeep, kDeviceBytes);
  }
  for (const DeviceBlock& b : drop) (void)hipFree(b.p);
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
  buf_[at_].reserve(std::max<size_t>(bytes, 1));
  return buf_[at_].data();
}

void Uploader::send(void* dst, size_t bytes, hipStream_t s) {
  if (!ev_[at_]) hip_check(hipEventCreateWithFlags(&ev_[at_], hipEventDisableTiming), "hipEventCreate");
  hip_check(hipMemcpyAsync(dst, buf_[at_].data(), bytes, hipMemcpyHostToDevice, s), "hipMemcpyAsync H2D");
  hip_check(hipEventRecord(ev_[at_], s), "hipEventRecord");
  busy_[at_] = true;
}

}  // namespace qr

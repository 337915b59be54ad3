// workspace_check.cpp — the blocks kept between calls (workspace.cpp) over a HIP runtime of stubs
// that counts what is allocated; no GPU is used. The argument names the check.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

#include "workspace.hpp"

using namespace qr;

namespace {

hipError_t last_error = hipSuccess;

struct Memory {
  std::map<void*, size_t> live;
  size_t held = 0, calls = 0;
  size_t limit = ~size_t(0);
  hipError_t get(void** p, size_t bytes) {
    ++calls;
    if (bytes > limit - held) return last_error = hipErrorOutOfMemory;
    *p = std::malloc(bytes);
    live[*p] = bytes;
    held += bytes;
    return hipSuccess;
  }
  hipError_t put(void* p) {
    if (!live.count(p)) return hipErrorInvalidValue;
    held -= live[p];
    live.erase(p);
    std::free(p);
    return hipSuccess;
  }
} pinned, device;

int failures = 0;
void expect(bool ok, const char* what) {
  if (ok) return;
  std::printf("FAIL: %s (pinned %zu bytes, device %zu bytes)\n", what, pinned.held, device.held);
  ++failures;
}

// One circuit on a state of its own: an upload block and a call's workspaces.
void circuit(size_t upload, size_t work) {
  pinned_state_created();
  {
    PinnedLease up(upload);
    PinnedLease a(work), b(2 * work);
    a.data()[work - 1] = 1;
  }
  pinned_state_destroyed();
}

// A program that makes and drops a state for every circuit pins its blocks once.
void state_per_circuit() {
  circuit(1000, 100000);
  const size_t calls = pinned.calls;
  for (int i = 0; i < 20; ++i) circuit(1000, 100000);
  expect(pinned.calls == calls, "blocks pinned anew for each circuit");
  circuit(1000, 3u << 20);
  expect(pinned.held <= kPinnedIdleBytes, "more than the allowance stays past the last state");
  const size_t after = pinned.calls;
  circuit(1000, 100000);
  expect(pinned.calls == after, "a large call pushed out the blocks of small ones");
}

// A call without a state (re-simulated shots) keeps no more than the idle bounds, also where the
// last state went while it ran, and with a state alive its blocks are still there.
void call_without_a_state() {
  auto call = [] {
    PinnedLease host(20u << 20), small(1000);
    DeviceLease states, tables;
    states.reserve(100u << 20);
    tables.reserve(100000);
  };
  call();
  expect(pinned.held <= kPinnedIdleBytes, "pinned blocks stay without a state");
  expect(device.held <= kDeviceIdleBytes, "device blocks stay without a state");
  pinned_state_created();
  call();
  const size_t calls = pinned.calls + device.calls;
  call();
  expect(pinned.calls + device.calls == calls, "blocks allocated anew while a state lives");
  {
    DeviceLease d;
    d.reserve(100u << 20);
    PinnedLease p(20u << 20);
    pinned_state_destroyed();
  }
  expect(pinned.held <= kPinnedIdleBytes, "pinned blocks stay after the last state");
  expect(device.held <= kDeviceIdleBytes, "device blocks stay after the last state");
}

// A workspace that fits is had, also where its rounded size doesn't fit.
void short_of_device_memory() {
  device.limit = 100u << 20;
  {
    DeviceLease a;
    a.reserve(70u << 20);
    expect(a.p != nullptr && device.held >= (70u << 20), "no workspace");
    std::memset(a.p, 1, 70u << 20);
  }
  DeviceLease b;
  bool refused = false;
  try {
    b.reserve(101u << 20);
  } catch (const Error& e) {
    refused = e.status == QR_ERR_OOM;
  }
  expect(refused, "a workspace beyond the device");
  expect(last_error == hipSuccess, "the error is left for the next launch");
  b.reserve(1000);
  expect(b.p != nullptr, "no workspace after a refused one");
}

}  // namespace

extern "C" {
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned int) { return pinned.get(p, bytes); }
hipError_t hipHostFree(void* p) { return pinned.put(p); }
hipError_t hipMalloc(void** p, size_t bytes) { return device.get(p, bytes); }
hipError_t hipFree(void* p) { return device.put(p); }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipEventCreateWithFlags(hipEvent_t*, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t bytes, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, bytes);
  return hipSuccess;
}
}

int main(int argc, char** argv) {
  struct {
    const char* name;
    void (*run)();
  } const checks[] = {{"state_per_circuit", state_per_circuit}, {"call_without_a_state", call_without_a_state},
                {"short_of_device_memory", short_of_device_memory}};
  for (const auto& c : checks)
    if (argc == 2 && std::strcmp(argv[1], c.name) == 0) {
      c.run();
      if (!failures) std::printf("ok\n");
      return failures ? 1 : 0;
    }
  return 2;
}

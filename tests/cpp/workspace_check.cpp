// workspace_check.cpp — the blocks kept between calls (workspace.cpp) over a HIP runtime of stubs
// that counts what is allocated; no GPU is used. The argument names the check.
#include <cstdio>
#include <cstring>

#include "hip_stubs.hpp"
#include "workspace.hpp"

using namespace qr;
using stub::device;
using stub::last_error;
using stub::pinned;

namespace {

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

// Uploads beyond the pinned bound, or where nothing can be pinned, take ordinary memory.
void large_uploads() {
  char* dst = (char*)std::malloc(200u << 20);
  auto send = [&](Uploader& up, size_t bytes) {
    uint8_t* h = up.begin(bytes);
    std::memset(h, 7, bytes);
    dst[bytes - 1] = 0;
    up.send(dst, bytes, nullptr);
    expect(dst[bytes - 1] == 7, "the upload's data");
  };
  {
    Uploader up;
    for (size_t bytes : {100u, 200u << 20, 200u << 20, 3u << 20, 200u << 20}) send(up, bytes);
    expect(pinned.largest <= kPinnedBytes, "more than the bound is pinned");
  }
  pinned.limit = pinned.held;
  {
    Uploader up;
    send(up, 50u << 20);
    send(up, 10);
  }
  PinnedLease kernel;
  bool refused = false;
  try {
    kernel.reserve(50u << 20);
  } catch (const Error&) {
    refused = true;
  }
  expect(refused && last_error == hipSuccess, "what kernels write must be pinned");
  pinned.limit = ~size_t(0);
  std::free(dst);
}

}  // namespace

int main(int argc, char** argv) {
  struct {
    const char* name;
    void (*run)();
  } const checks[] = {{"state_per_circuit", state_per_circuit}, {"call_without_a_state", call_without_a_state},
                {"short_of_device_memory", short_of_device_memory},
                {"large_uploads", large_uploads}};
  for (const auto& c : checks)
    if (argc == 2 && std::strcmp(argv[1], c.name) == 0) {
      c.run();
      if (!failures) std::printf("ok\n");
      return failures ? 1 : 0;
    }
  return 2;
}

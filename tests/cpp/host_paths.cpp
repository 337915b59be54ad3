// host_paths.cpp — the host code between a caller's program and the kernels (lower.cpp,
// planner.cpp, plan_image.cpp), built with sanitizers; no GPU is used. The argument names the check.
#include <cstdio>
#include <cstring>
#include <random>

#include "engine.hpp"
#include "kernels.hpp"

using namespace qr;

namespace {

int failures = 0;
void expect(bool ok, const char* what) {
  if (ok) return;
  std::printf("FAIL: %s\n", what);
  ++failures;
}

struct Prog {
  std::vector<qr_op> ops;
  std::vector<uint32_t> ctl;
  std::vector<double> img;
  std::vector<uint8_t> some;
  qr_program view() const {
    return qr_program{ops.data(), ops.size(), ctl.data(), ctl.size(), img.data(), img.size(), some.data(), some.size()};
  }
  // A custom gate on the wires (the last one its position), dense or diagonal.
  void custom(const std::vector<uint32_t>& wires, bool dense, std::mt19937_64& rng) {
    qr_op op{};
    op.kind = QR_GATE_CUSTOM;
    op.position = wires.back();
    op.ncontrols = (uint32_t)wires.size() - 1;
    op.controls_offset = ctl.size();
    ctl.insert(ctl.end(), wires.begin(), wires.end() - 1);
    op.image_offset = img.size();
    op.some_offset = some.size();
    const uint64_t dim = 1ull << wires.size();
    some.resize(some.size() + dim, 1);
    img.resize(img.size() + 2 * dim * dim, 0.0);
    std::normal_distribution<double> g;
    for (uint64_t j = 0; j < dim; ++j)
      for (uint64_t r = 0; r < dim; ++r)
        if (dense || r == j) {
          img[op.image_offset + 2 * (j * dim + r)] = g(rng);
          img[op.image_offset + 2 * (j * dim + r) + 1] = g(rng);
        }
    ops.push_back(op);
  }
};

std::vector<uint64_t> key_of(const std::vector<FastOp>& ops) {
  std::vector<uint64_t> k;
  for (const FastOp& op : ops) plan_key_append(op, k);
  return k;
}

// Custom gates on more than eight wires: all of their wires reach the op and the plan's key.
void wide_customs() {
  std::mt19937_64 rng(7);
  const uint32_t n = 12;
  for (int k : {8, 9, 10})
    for (bool dense : {false, true}) {
      std::vector<uint32_t> wires;
      for (int q = 0; q < k; ++q) wires.push_back((uint32_t)(q * 5 % 11));
      Prog p, other;
      p.custom(wires, dense, rng);
      wires.back() = 11;
      other.custom(wires, dense, rng);
      const qr_program v = p.view(), w = other.view();
      validate_program(n, &v);
      const std::vector<FastOp> ops = lower_program(n, &v, false), ops2 = lower_program(n, &w, false);
      expect(ops.size() == 1 && ops[0].k == k && ops[0].cmask == 0, "the op of a wide custom gate");
      expect(ops[0].kind == (dense ? FK_DENSEK : FK_DIAGK), "its kind");
      for (int q = 0; q < k; ++q) expect(ops[0].bits[q] == (int)(n - 1 - (uint32_t)(q * 5 % 11)), "its wires");
      const uint64_t dim = 1ull << k;
      for (uint64_t j = 0; j < dim; ++j) {
        const cd want(p.img[2 * (j * dim + j)], p.img[2 * (j * dim + j) + 1]);
        expect(ops[0].m[dense ? j * dim + j : j] == want, "its table");
      }
      expect(key_of(ops) != key_of(ops2), "gates on other wires share a plan");
    }
}

}  // namespace

int main(int argc, char** argv) {
  struct {
    const char* name;
    void (*run)();
  } const checks[] = {{"wide_customs", wide_customs}};
  for (const auto& c : checks)
    if (argc == 2 && std::strcmp(argv[1], c.name) == 0) {
      c.run();
      if (!failures) std::printf("ok\n");
      return failures ? 1 : 0;
    }
  return 2;
}

// lower_compare.cpp — the direct lowering of a program against the general one (test
// infrastructure only): random programs of every gate kind, custom tables included, must give
// identical ops, numbers compared bit for bit.
#include <cstdio>
#include <cstring>
#include <random>

#include "engine.hpp"

using namespace qr;

namespace {

bool same(const FastOp& a, const FastOp& b) {
  return a.kind == b.kind && a.k == b.k && std::memcmp(a.bits, b.bits, sizeof a.bits) == 0 && a.cmask == b.cmask &&
         a.m.size() == b.m.size() &&
         (a.m.empty() || std::memcmp(a.m.data(), b.m.data(), a.m.size() * sizeof(cd)) == 0) && a.form == b.form &&
         a.sub == b.sub && a.param == b.param && a.gen == b.gen && a.gate_index == b.gate_index &&
         a.f_touch == b.f_touch;
}

}  // namespace

int main() {
  std::mt19937_64 rng(20);
  const double angles[] = {0.0, 3.141592653589793, -3.141592653589793, 6.283185307179586, 1e-9, 0.7, -2.1};
  for (int trial = 0; trial < 400; ++trial) {
    const uint32_t n = 3 + (uint32_t)(rng() % 8);
    std::vector<qr_op> ops;
    std::vector<uint32_t> controls;
    std::vector<double> images;
    std::vector<uint8_t> some;
    for (int g = 0; g < 60; ++g) {
      qr_op op{};
      op.kind = (uint32_t)(rng() % QR_GATE_KIND_COUNT);
      std::vector<uint32_t> w(n);
      for (uint32_t i = 0; i < n; ++i) w[i] = i;
      std::shuffle(w.begin(), w.end(), rng);
      op.position = w[0];
      op.arg = rng() % 2 ? angles[rng() % 7] : (double)(int64_t)rng() * 1e-18;
      op.arg_int = (int32_t)(rng() % 7) - 2;
      uint32_t nc = 0;
      switch (op.kind) {
        case QR_GATE_CR: case QR_GATE_CRK: case QR_GATE_CZ: case QR_GATE_CY: case QR_GATE_CNOT: case QR_GATE_SWAP: nc = 1; break;
        case QR_GATE_TOFFOLI: nc = 2; break;
        case QR_GATE_CUSTOM: nc = (uint32_t)(rng() % 3); break;
        default: break;
      }
      op.ncontrols = nc;
      op.controls_offset = controls.size();
      for (uint32_t i = 0; i < nc; ++i) controls.push_back(w[1 + i]);
      if (op.kind == QR_GATE_CUSTOM) {
        const uint64_t dim = 2ull << nc;
        op.image_offset = images.size();
        op.some_offset = some.size();
        const int shape = (int)(rng() % 3);  // dense, diagonal, identity with a controlled block
        for (uint64_t j = 0; j < dim; ++j) some.push_back(rng() % 8 != 0);
        for (uint64_t j = 0; j < dim; ++j)
          for (uint64_t r = 0; r < dim; ++r) {
            const bool on = shape == 0 || (shape == 1 && r == j) || (shape == 2 && (j >= dim / 2 ? r >= dim / 2 : r == j));
            const bool one = shape == 2 && j < dim / 2;
            images.push_back(on ? (one ? 1.0 : (double)(int64_t)rng() * 1e-19) : 0.0);
            images.push_back(on && !one ? (double)(int64_t)rng() * 1e-19 : 0.0);
          }
      }
      ops.push_back(op);
    }
    qr_program p{ops.data(), ops.size(), controls.data(), controls.size(), images.data(), images.size(), some.data(), some.size()};
    for (int params = 0; params < 2; ++params) {
      const std::vector<FastOp> want = lower_fast(n, lower_exact(n, &p), params != 0);
      const std::vector<FastOp> got = lower_program(n, &p, params != 0);
      if (got.size() != want.size()) {
        std::printf("FAIL: %zu ops, want %zu\n", got.size(), want.size());
        return 1;
      }
      for (size_t i = 0; i < got.size(); ++i)
        if (!same(got[i], want[i])) {
          std::printf("FAIL: trial %d op %zu (params %d)\n", trial, i, params);
          return 1;
        }
    }
  }
  std::printf("ok\n");
  return 0;
}

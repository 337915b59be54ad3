// plan_rules.cpp — the rules that choose tile shapes (planner.cpp); no GPU is used.
#include <cstdio>

#include "engine.hpp"

using namespace qr;

int main() {
  int failures = 0;
  auto expect = [&](bool ok, const char* what, uint32_t n, int prec, int tile, uint64_t simds) {
    if (ok) return;
    std::printf("FAIL: %s (n %u, prec %d, tile %d, simds %llu)\n", what, n, prec, tile, (unsigned long long)simds);
    ++failures;
  };
  for (uint64_t simds : {0ull, 128ull, 1024ull, 1216ull})
    for (int prec : {0, 1})
      for (uint32_t n = 1; n <= 34; ++n)
        for (int tile = 0; tile <= 13; ++tile) {
          const PlanParams p = dual_plan_params(n, prec, tile, simds);
          expect(p.tile_bits >= 1 && p.tile_bits <= (int)n && (!tile || p.tile_bits == std::min(tile, (int)n)),
                 "tile width", n, prec, tile, simds);
          expect(p.reg_bits >= 1 && p.reg_bits <= 4 && p.reg_bits <= p.tile_bits, "register bits", n, prec, tile, simds);
          expect(p.tile_bits < 7 || p.tile_bits - p.reg_bits >= 6, "less than a wavefront", n, prec, tile, simds);
          if (tile) {  // an instance of a batch and a gradient alone differ in the one-wavefront rule only
            const PlanParams q = dual_plan_params(n, prec, tile, 0);
            const bool one_wave = prec == 0 && (1ull << n) == simds * 64 * 16 && p.tile_bits >= 10;
            expect(one_wave ? p.reg_bits == 4 : p.reg_bits == q.reg_bits, "batch and gradient differ", n, prec, tile, simds);
          }
        }
  if (!failures) std::printf("ok\n");
  return failures ? 1 : 0;
}

// host_paths.cpp — the host code between a caller's program and the kernels (lower.cpp,
// planner.cpp, plan_image.cpp), built with sanitizers; no GPU is used. The argument names the check.
#include <algorithm>
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

// Random gates of every kind but Custom on n >= 3 wires, the same gates for the same seed, angles apart.
Prog random_program(uint32_t n, int count, uint64_t seed, uint64_t angles) {
  std::mt19937_64 rng(seed), ang(angles);
  Prog p;
  for (int g = 0; g < count; ++g) {
    qr_op op{};
    op.kind = (uint32_t)(rng() % QR_GATE_CUSTOM);
    std::vector<uint32_t> w(n);
    for (uint32_t i = 0; i < n; ++i) w[i] = i;
    std::shuffle(w.begin(), w.end(), rng);
    op.position = w[0];
    op.arg = 0.1 + (double)(ang() % 1000) / 400.0;
    op.arg_int = 1 + (int)(rng() % 5);
    switch (op.kind) {
      case QR_GATE_CR: case QR_GATE_CRK: case QR_GATE_CZ: case QR_GATE_CY: case QR_GATE_CNOT: case QR_GATE_SWAP:
        op.ncontrols = 1; break;
      case QR_GATE_TOFFOLI: op.ncontrols = 2; break;
      default: break;
    }
    op.controls_offset = p.ctl.size();
    for (uint32_t i = 0; i < op.ncontrols; ++i) p.ctl.push_back(w[1 + i]);
    p.ops.push_back(op);
  }
  return p;
}

// A plan's blob: its values are those of the program at hand, its standalone offsets those of the
// wires, nothing of it is left unwritten, and the plan keeps no table of its own.
void plan_images() {
  std::mt19937_64 rng(11);
  for (int trial = 0; trial < 24; ++trial) {
    const uint32_t n = 4 + (uint32_t)(trial % 9);
    Prog a = random_program(n, 80, 100 + trial, 1), b = random_program(n, 80, 100 + trial, 2);
    std::vector<std::vector<uint32_t>> wires = {{2, 0}, {1, 3, 0}, {3, 2, 1, 0}};
    if (n >= 10) wires.push_back({9, 8, 7, 6, 5, 4, 3, 2, 1});
    for (const auto& w : wires)
      for (bool dense : {true, false}) {
        std::mt19937_64 ra(rng()), rb(rng());
        a.custom(w, dense, ra);
        b.custom(w, dense, rb);
      }
    const qr_program va = a.view(), vb = b.view();
    const bool dual = trial % 2 == 1;
    std::vector<FastOp> opa = lower_program(n, &va, dual), opb = lower_program(n, &vb, dual);
    if (dual) {
      opa = adjoint_sweep_ops(opa);
      opb = adjoint_sweep_ops(opb);
    }
    expect(key_of(opa) == key_of(opb), "programs that differ in values have one structure");
    PlanParams pp;
    pp.tile_bits = std::min<int>(trial % 3 ? 10 : 5, (int)n);
    pp.reg_bits = std::min(4, pp.tile_bits);
    pp.low_bits = 3;
    const std::vector<Stage> stages = plan_fused(n, opa, pp, 16, dual);
    const PlanImage im = plan_image(opa, stages);
    std::vector<uint8_t> x(im.size() + 16, 0x11), y(im.size() + 16, 0x77);
    for (std::vector<uint8_t>* blob : {&x, &y}) {
      im.write_fixed(blob->data(), im.size());
      write_values(opb, stages, im.loc, blob->data());
    }
    expect(std::equal(x.begin(), x.begin() + im.size(), y.begin()), "part of the blob is left unwritten");
    expect(x[im.size()] == 0x11, "written behind the blob");
    std::vector<uint8_t> live(im.live + 16, 0x33);
    im.write_fixed(live.data(), im.live);
    write_values(opb, stages, im.loc, live.data());
    expect(std::equal(x.begin(), x.begin() + im.live, live.begin()) && live[im.live] == 0x33, "the live part");
    size_t tables = 0, offsets = 0;
    for (size_t si = 0; si < stages.size(); ++si) {
      const Stage& s = stages[si];
      const cd* c = (const cd*)(x.data() + im.loc[si].coefs);
      if (s.tile) {
        std::vector<cd> want;
        stage_coefficients(s, opb, want);
        expect(want.empty() || std::memcmp(c, want.data(), want.size() * sizeof(cd)) == 0, "a stage's coefficients");
        expect(im.loc[si].ops >= im.live && im.loc[si].ops % 64 == 0, "a stage's ops");
        const TileOpDev* d = (const TileOpDev*)(x.data() + im.loc[si].ops);
        for (size_t i = 0; i < s.ops.size(); ++i) expect((d[i].w0 & 0xFF) == (uint32_t)s.ops[i].code, "an op's code");
        continue;
      }
      const FastOp& op = opb[s.standalone];
      if (op.kind != FK_DENSEK && op.kind != FK_DIAGK) continue;
      tables += op.m.size() * sizeof(cd);
      offsets += sizeof(uint64_t) << op.k;
      expect(std::equal(op.m.begin(), op.m.end(), c), "a table");
      const uint64_t* off = (const uint64_t*)(x.data() + im.loc[si].off);
      for (uint64_t j = 0; j < 1ull << op.k; ++j) {
        uint64_t want = 0;
        for (int q = 0; q < op.k; ++q)
          if ((j >> (op.k - 1 - q)) & 1) want |= 1ull << op.bits[q];
        expect(off[j] == want, "an offset");
      }
    }
    expect(im.values >= tables && im.live - im.values == offsets, "the plan keeps values");
  }
}

// ---- expectation records, read as k_pauli_expect_tiles reads them -----------------------------

uint64_t deposit(uint64_t x, uint64_t mask) {
  uint64_t out = 0;
  for (int b = 0; mask; ++b) {
    const uint64_t low = mask & (0ull - mask);
    mask ^= low;
    if ((x >> b) & 1u) out |= low;
  }
  return out;
}
double sign(uint64_t x) { return __builtin_popcountll(x) & 1 ? -1.0 : 1.0; }

double replay(int prec, uint32_t n, const std::vector<cd>& psi, const uint8_t* group_records, const uint8_t* term_records,
              const std::vector<PauliTilePass>& passes, const uint32_t* diag_count) {
  const int K = pauli_tile_bits(prec);
  const PauliTileGroup* groups = (const PauliTileGroup*)group_records;
  const PauliTileTerm* terms = (const PauliTileTerm*)term_records;
  double total = 0.0;
  for (const PauliTilePass& ps : passes) {
    if (ps.tmask == 0) {
      for (uint32_t i = 0; i < ps.cnt[0]; ++i) {
        const PauliGroup& g = ((const PauliGroup*)group_records)[ps.first + i];
        for (uint32_t t = 0; t < g.count; ++t) {
          const PauliZTerm& z = ((const PauliZTerm*)term_records)[g.first + t];
          for (uint64_t o = 0; o < psi.size(); ++o)
            total += (std::conj(psi[o]) * cd(z.cr, z.ci) * sign((o ^ g.xm) & z.zm) * psi[o ^ g.xm]).real();
        }
      }
      continue;
    }
    expect(__builtin_popcountll(ps.tmask) == K, "a pass's tile");
    const uint64_t nontile = (psi.size() - 1) & ~ps.tmask;
    std::vector<uint64_t> at(1u << K);
    for (uint64_t p = 0; p < at.size(); ++p) at[p] = deposit(p, ps.tmask);
    for (uint64_t tile = 0; tile < psi.size() >> K; ++tile) {
      const uint64_t base = deposit(tile, nontile);
      for (uint32_t lane = 0; lane < 1u << (K - 4); ++lane) {
        const PauliTileGroup* gp = groups + ps.first;
        const PauliTileTerm* tp = terms + ps.term0;
        for (int arr = 0; arr < kPauliArrangements; ++arr) {
          if (!((ps.arrs >> arr) & 1u)) continue;
          const int nb = pauli_arrangement_bit(K, arr);
          const uint32_t pt = (lane & ((1u << nb) - 1u)) | ((lane >> nb) << (nb + 4));
          auto amp = [&](uint32_t r, uint32_t lx = 0) { return psi[base | at[(pt | (r << nb)) ^ lx]]; };
          auto coef = [&](const PauliTileTerm& t) { return t.c * sign(pt & t.lz) * sign(base & t.zout); };
          if (arr == 0 && ps.diag)
            for (uint32_t p = 0; p < 16; ++p)
              for (uint32_t c = diag_count[p]; c; --c, ++tp) {
                expect(tp->pat == p, "the order of Z strings");
                for (uint32_t r = 0; r < 16; ++r) total += coef(*tp) * sign(r & p) * std::norm(amp(r));
              }
          for (uint32_t m = 1; m < 16; ++m)
            if ((ps.plain[arr] >> m) & 1u) {
              const uint32_t top = 31 - __builtin_clz(m);
              for (uint32_t r = 0; r < 16; ++r)
                if (!((r >> top) & 1u)) total += coef(*tp) * (std::conj(amp(r)) * amp(r ^ m)).real();
              ++tp;
            }
          for (uint32_t g = 0; g < ps.cnt[arr]; ++g, ++gp) {
            const uint32_t top = gp->op >= PAULI_LDS ? gp->op - PAULI_LDS : 31 - (uint32_t)__builtin_clz(gp->op);
            expect(gp->op >= PAULI_LDS ? ((gp->lx >> nb) & 15u) >> top == 1u : gp->lx == gp->op << nb, "a group's pairs");
            for (uint32_t q = 0; q < gp->nre + gp->nim; ++q, ++tp)
              for (uint32_t r = 0; r < 16; ++r) {
                if ((r >> top) & 1u) continue;
                const uint32_t i = (r & ((1u << top) - 1u)) | ((r >> (top + 1)) << top);
                const cd v = std::conj(amp(r)) * amp(r, gp->lx);
                total += coef(*tp) * sign(i & tp->pat) * (q < gp->nre ? v.real() : v.imag());
              }
          }
        }
      }
    }
  }
  return total;
}

// The records of observables that use every arrangement, masks that cross them, both parities of Y,
// more passes than one launch takes and masks too wide for a tile, against the plain sum. Both are
// sums of products of modulus at most 1 in binary64.
void expectation_records() {
  struct Shape {
    int prec;
    uint32_t n;
    int kind;
  };
  for (const Shape sh : {Shape{0, 15, 0}, Shape{0, 15, 1}, Shape{0, 16, 2}, Shape{0, 10, 0}, Shape{1, 16, 0},
                         Shape{1, 16, 1}, Shape{1, 17, 2}}) {
    std::mt19937_64 rng(500 + sh.n + (uint64_t)sh.kind);
    std::normal_distribution<double> g;
    const uint32_t n = sh.n;
    std::vector<cd> psi(1ull << n);
    for (cd& a : psi) a = cd(g(rng), g(rng)) * std::ldexp(1.0, -(int)n / 2);
    std::vector<PauliMasks> obs;
    auto term = [&](uint64_t xm, uint64_t zm) { obs.push_back(PauliMasks{g(rng), xm, zm, __builtin_popcountll(xm & zm)}); };
    const uint64_t all = (1ull << n) - 1;
    const int tile = pauli_tile_bits(sh.prec), low = pauli_low_bits(sh.prec);
    if (sh.kind < 2)
      for (uint32_t b = 0; b < n; ++b) {
        term(1ull << b, 0);
        term(0, (1ull << b) | (1ull << ((b + 5) % n)));
        if (sh.kind == 1) continue;
        term(1ull << b, 1ull << b);
        term(3ull << (b % (n - 1)), rng() & all);
        term(15ull << (b % (n - 3)), rng() & all);
        term((1ull << b) | (1ull << (rng() % n)), rng() & all);
      }
    if (sh.kind == 2)
      for (int t = 0; t < 60; ++t) {  // as many high bits as a tile holds beside the low ones, and all
        uint64_t xm = rng() & ((1ull << low) - 1);
        while (__builtin_popcountll(xm >> low) < tile - low) xm |= 1ull << (low + (int)(rng() % (n - (uint32_t)low)));
        term(t % 20 == 19 ? all : xm, rng() & all);
      }
    std::vector<PauliGroup> groups;
    std::vector<PauliZTerm> flat;
    pauli_tables(obs, groups, flat);
    const int G = (int)groups.size();
    std::vector<PauliPass> passes(G + 1);
    std::vector<uint32_t> lxm(G);
    const int np = pauli_passes(n, sh.prec, groups.data(), G, passes.data(), lxm.data());
    if (sh.kind == 2) expect(np > (int)kPauliPassesPerLaunch, "more passes than one launch takes");
    std::vector<PauliTilePass> tp(np);
    uint32_t diag_count[16];
    std::vector<uint8_t> gr((G + 1) * sizeof(PauliGroup)), tr((flat.size() + 1) * sizeof(PauliZTerm));
    pauli_tile_tables(sh.prec, groups.data(), lxm.data(), passes.data(), np, flat.data(), gr.data(), tr.data(), tp.data(),
                      diag_count);
    const double got = replay(sh.prec, n, psi, gr.data(), tr.data(), tp, diag_count);
    double want = 0.0, weight = 0.0;
    for (const PauliMasks& t : obs) {
      cd f = t.coeff;
      for (int q = 0; q < t.ny; ++q) f *= cd(0, 1);
      weight += std::fabs(t.coeff);
      for (uint64_t j = 0; j < psi.size(); ++j) want += (std::conj(psi[j ^ t.xm]) * f * sign(j & t.zm) * psi[j]).real();
    }
    expect(std::fabs(got - want) < 64 * n * 2.3e-16 * weight * 2.0, "the value of an observable");
  }
}

}  // namespace

int main(int argc, char** argv) {
  struct {
    const char* name;
    void (*run)();
  } const checks[] = {{"wide_customs", wide_customs}, {"plan_images", plan_images},
                {"expectation_records", expectation_records}};
  for (const auto& c : checks)
    if (argc == 2 && std::strcmp(argv[1], c.name) == 0) {
      c.run();
      if (!failures) std::printf("ok\n");
      return failures ? 1 : 0;
    }
  return 2;
}

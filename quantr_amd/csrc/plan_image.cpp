// plan_image.cpp — the layout of a plan's device blob and what fills it.
#include <cstring>

#include "engine.hpp"
#include "kernels.hpp"

namespace qr {

static bool has_table(const FastOp& op) { return op.kind == FK_DENSEK || op.kind == FK_DIAGK; }

PlanImage plan_image(const std::vector<FastOp>& ops, const std::vector<Stage>& stages) {
  PlanImage im;
  im.loc.assign(stages.size(), Loc{});
  // ---- coefficients and standalone tables: their places only
  for (size_t si = 0; si < stages.size(); ++si) {
    const Stage& s = stages[si];
    if (!s.tile && !has_table(ops[s.standalone])) continue;
    im.loc[si].coefs = im.values;
    im.values += (s.tile ? s.ops.size() * 4 : ops[s.standalone].m.size()) * sizeof(double2);
  }
  std::vector<uint8_t>& blob = im.fixed;
  auto align = [&](size_t a) {
    while (im.size() % a) blob.push_back(0);
  };
  auto append = [&](const void* p, size_t bytes) {
    const size_t at = blob.size();
    blob.resize(at + bytes);
    if (bytes) std::memcpy(blob.data() + at, p, bytes);
    return im.values + at;
  };
  for (size_t si = 0; si < stages.size(); ++si) {
    const Stage& s = stages[si];
    if (s.tile || !has_table(ops[s.standalone])) continue;
    const FastOp& op = ops[s.standalone];
    const int dim = 1 << op.k;
    std::vector<uint64_t> off(dim, 0);
    for (int j = 0; j < dim; ++j)
      for (int q = 0; q < op.k; ++q)
        if ((j >> (op.k - 1 - q)) & 1) off[j] |= 1ull << op.bits[q];
    im.loc[si].off = append(off.data(), off.size() * sizeof(uint64_t));
  }
  im.live = im.size();
  // ---- what interpreted stages read
  for (size_t si = 0; si < stages.size(); ++si) {
    const Stage& s = stages[si];
    if (!s.tile) continue;
    align(64);
    std::vector<TileOpDev> d(s.ops.size());
    for (size_t i = 0; i < s.ops.size(); ++i) {
      const TileOpHost& h = s.ops[i];
      TileOpDev t{};
      const bool maps_op = h.code == TC_REMAP || h.code == TC_SWAPSLOTS;
      t.w0 = (h.code & 0xFF) | ((maps_op ? 0u : (h.a & 0xFF)) << 8) | ((h.b & 0xFF) << 16) | ((h.flags & 0xFF) << 24);
      t.ns = h.ns;
      t.lane_cmask = h.lane_cmask;
      t.map = maps_op ? h.a : 0;
      t.swz = h.swz;
      d[i] = t;
    }
    im.loc[si].ops = append(d.data(), d.size() * sizeof(TileOpDev));
    align(4);
    std::vector<uint32_t> m(s.maps.size());
    for (size_t i = 0; i < m.size(); ++i)  // physical bit | tile position << 8
      m[i] = (uint32_t)s.phys_bit((int)(i / s.k), s.maps[i]) | ((uint32_t)s.maps[i] << 8);
    im.loc[si].maps = append(m.data(), m.size() * sizeof(uint32_t));
    std::vector<uint32_t> z(s.swz.begin(), s.swz.end());
    if (z.empty()) z.push_back(0);
    im.loc[si].off = append(z.data(), z.size() * sizeof(uint32_t));
  }
  return im;
}

void write_values(const std::vector<FastOp>& ops, const std::vector<Stage>& stages, const std::vector<Loc>& loc,
                  uint8_t* blob) {
  static_assert(sizeof(cd) == sizeof(double2), "coefficients are stored as pairs of doubles");
  for (size_t si = 0; si < stages.size(); ++si) {
    const Stage& s = stages[si];
    cd* c = reinterpret_cast<cd*>(blob + loc[si].coefs);
    if (s.tile) {
      // the program's own coefficients (plans are shared by structure), folded scalars applied;
      // gradient taps carry their parameter row
      stage_coefficients(s, ops, c);
      continue;
    }
    const FastOp& op = ops[s.standalone];
    if (has_table(op)) std::copy(op.m.begin(), op.m.end(), c);
  }
}

}  // namespace qr

// sampler_check.cpp — the samplers of one state (sampler.cpp) and of re-simulated programs
// (shots.cpp) over a HIP runtime of stubs and kernels written for the host: what they pin and
// launch, and the bins against the left fold. No GPU is used. The argument names the check.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

#include "hip_stubs.hpp"
#include "runtime.hpp"

using namespace qr;

namespace {

int failures = 0;
void expect(bool ok, const char* what) {
  if (ok) return;
  std::printf("FAIL: %s (largest pinned block %zu bytes)\n", what, stub::pinned.largest);
  ++failures;
}

size_t gathers = 0, placings = 0, folds = 0;

template <class R>
double prob(const void* psi, uint64_t i) {
  const double re = (double)((const R*)psi)[2 * i], im = (double)((const R*)psi)[2 * i + 1];
  return re * re + im * im;
}
double prob(int prec, const void* psi, uint64_t i) { return prec == 0 ? prob<double>(psi, i) : prob<float>(psi, i); }

// The bins of ascending draws by the left fold.
std::vector<uint64_t> left_fold(int prec, const void* psi, uint64_t dim, const std::vector<double>& us) {
  std::vector<uint64_t> out(us.size(), ~0ull);
  double s = 0.0;
  size_t d = 0;
  for (uint64_t i = 0; i < dim && d < us.size(); ++i) {
    s = s + prob(prec, psi, i);
    while (d < us.size() && us[d] < s) out[d++] = i;
  }
  return out;
}

// A normalised random state of n qubits in the state's own memory.
void random_state(qr_state& st, uint32_t n, int prec, uint64_t seed) {
  st.n = n;
  st.prec = prec;
  st.dim = 1ull << n;
  (void)hipMalloc(&st.amp, st.dim * st.bytes_per_amp());
  std::mt19937_64 rng(seed);
  std::normal_distribution<double> g;
  const double f = std::ldexp(1.0, -(int)n / 2) / std::sqrt(2.0);
  for (uint64_t i = 0; i < 2 * st.dim; ++i) {
    if (prec == 0) ((double*)st.amp)[i] = f * g(rng);
    else ((float*)st.amp)[i] = (float)(f * g(rng));
  }
}

std::vector<double> draws(size_t count, uint64_t seed) {
  std::mt19937_64 rng(seed);
  std::uniform_real_distribution<double> u;
  std::vector<double> v(count);
  for (double& x : v) x = u(rng);
  return v;
}

// Many draws are placed in slices: a bounded block is pinned whatever their number.
void many_draws() {
  const size_t count = 5 * kDrawSlice + 12345;
  std::vector<double> us;
  std::vector<uint64_t> perm, res;
  sort_draws(draws(count, 3).data(), count, us, perm);
  {
    qr_state st;
    random_state(st, 16, 0, 1);
    sample_exact_parallel(&st, us, res);
    expect(res == left_fold(0, st.amp, st.dim, us), "bins of many draws");
  }
  expect(placings >= 5, "draws were not sliced");
  expect(stub::pinned.largest <= 24 * kDrawSlice, "pinned memory grows with the draws");
}

// The same for the draws of re-simulated programs; the states of this check are |0...0>.
void many_draws_of_programs() {
  const uint64_t per[] = {3, kDrawSlice + 7, 0, kDrawSlice + 5, 2};
  uint64_t total = 0;
  for (uint64_t p : per) total += p;
  std::vector<double> u = draws(total, 5);
  u[total - 1] = 1.5;  // beyond the total: none
  std::vector<uint64_t> out(total, 7);
  qr_program none{};
  const qr_program programs[5] = {none, none, none, none, none};
  sample_programs(4, 0, programs, 5, per, u.data(), out.data());
  for (uint64_t d = 0; d < total; ++d)
    if (out[d] != (u[d] < 1.0 ? 0 : ~0ull)) {
      expect(false, "bins of many programs' draws");
      break;
    }
  expect(folds == 3, "draws were not sliced");
  expect(stub::pinned.largest <= 24 * kDrawSlice, "pinned memory grows with the draws");
}

// Blocks that the host folds arrive together, however many have a halfway case.
void halfway_blocks() {
  const std::vector<double> u = draws(1000, 9);
  std::vector<double> us;
  std::vector<uint64_t> perm, res;
  sort_draws(u.data(), u.size(), us, perm);
  for (int prec : {0, 1})
    for (uint32_t n : {16u, 20u, 22u}) {
      qr_state st;
      random_state(st, n, prec, n);
      if (prec == 0 && n == 22)  // short mantissas: hundreds of blocks
        for (uint64_t i = 0; i < 2 * st.dim; ++i) {
          double& x = ((double*)st.amp)[i];
          x = std::ldexp(std::rint(std::ldexp(x, 34)), -34);
        }
      gathers = 0;
      sample_exact_parallel(&st, us, res);
      expect(res == left_fold(prec, st.amp, st.dim, us), "bins of a state with halfway cases");
      if (gathers > 2) std::printf("%zu launches, %u qubits, precision %d\n", gathers, n, prec);
      expect(gathers <= 2, "blocks fetched one by one");
    }
}

}  // namespace

namespace qr {

// ---- kernels, on the host
hipError_t launch_gather_probs(int prec, const void* psi, int bb, const uint64_t* list, uint32_t count, double* out,
                               hipStream_t) {
  if (count) ++gathers;
  for (uint64_t y = 0; y < count; ++y)
    for (uint64_t q = 0; q < 1ull << bb; ++q)
      out[(y << bb) + q] = prob(prec, psi, ((list ? list[y] : y) << bb) + q);
  return hipSuccess;
}

hipError_t launch_block_mass(int prec, const void* psi, uint64_t dim, int bb, double* mass, hipStream_t) {
  for (uint64_t b = 0; b < dim >> bb; ++b) {
    mass[b] = 0.0;
    for (uint64_t q = 0; q < 1ull << bb; ++q) mass[b] += prob(prec, psi, (b << bb) + q);
  }
  return hipSuccess;
}

hipError_t launch_block_exact_sums(int prec, const void* psi, uint64_t dim, int bb, const int32_t* ebase, double* sums,
                                   uint32_t* flags, const TieBlocks& tie, hipStream_t) {
  for (uint64_t b = 0; b < dim >> bb; ++b) {
    flags[b] = 0;
    for (int c = 0; c < 3; ++c) {
      const int e = ebase[b] + c;
      double sum = 0.0;
      if (e < -960 || e > 52) flags[b] |= 1u << c;
      else
        for (uint64_t q = 0; q < 1ull << bb; ++q) {
          const double x = prob(prec, psi, (b << bb) + q) * std::ldexp(1.0, 52 - e), r = std::rint(x);
          if (std::fabs(x - std::trunc(x)) == 0.5) flags[b] |= 1u << c;
          sum += r;
        }
      sums[3 * b + c] = sum;
    }
    if (!(flags[b] & 2u) || ebase[b] + 1 < -960 || ebase[b] + 1 > 52) continue;
    const uint32_t place = (*tie.count)++;
    if (place >= tie.most) continue;
    tie.block[place] = b;
    for (uint64_t q = 0; q < 1ull << bb; ++q) tie.probs[((uint64_t)place << bb) + q] = prob(prec, psi, (b << bb) + q);
  }
  return hipSuccess;
}

hipError_t launch_sample_exact_blocks(int prec, const void* psi, uint64_t, int bb, const ExactJob* jobs, uint64_t njobs,
                                      const double* u, uint64_t* out, hipStream_t) {
  ++placings;
  for (uint64_t j = 0; j < njobs; ++j) {
    const ExactJob& job = jobs[j];
    double run = job.m_start;
    uint64_t d = job.first;
    for (uint64_t q = 0; q < 1ull << bb && d < job.last; ++q) {
      const uint64_t i = (job.block << bb) + q;
      run += std::rint(prob(prec, psi, i) * job.scale);
      while (d < job.last && u[d] < run * job.unit) out[d++] = i;
    }
  }
  return hipSuccess;
}

hipError_t launch_init_instances(int prec, void* psi, uint64_t dim, uint64_t count, hipStream_t) {
  std::memset(psi, 0, dim * count * (prec == 0 ? 16 : 8));
  for (uint64_t y = 0; y < count; ++y) {
    if (prec == 0) ((double*)psi)[2 * dim * y] = 1.0;
    else ((float*)psi)[2 * dim * y] = 1.0f;
  }
  return hipSuccess;
}

hipError_t launch_sample_fold_instances(int prec, const void* psi, uint64_t dim, uint64_t count, const double* u,
                                        const uint64_t* off, uint64_t* out, hipStream_t) {
  ++folds;
  for (uint64_t y = 0; y < count; ++y) {
    double s = 0.0;
    uint64_t d = off[y];
    for (uint64_t i = 0; i < dim; ++i) {
      s = s + prob(prec, psi, y * dim + i);
      while (d < off[y + 1] && u[d] < s) out[d++] = i;
    }
    while (d < off[y + 1]) out[d++] = ~0ull;
  }
  return hipSuccess;
}

// ---- plans: programs without gates
PlanParams plan_params(uint32_t, int, const qr_options&) { return PlanParams{}; }
std::shared_ptr<CachedPlan> get_plan_for(uint32_t, int, const std::vector<FastOp>&, const PlanParams&, bool, bool, bool) {
  return std::make_shared<CachedPlan>();
}
void prepare_compiled(CachedPlan&, int, int, bool, bool) {}
void write_values(const std::vector<FastOp>&, const std::vector<Stage>&, const std::vector<Loc>&, uint8_t*) {}
TileArgs tile_args_at(uint32_t, const Stage&, const uint8_t*, const Loc&) { return TileArgs{}; }
void launch_standalone_raw(int, uint64_t, void*, DevBuf&, const FastOp&, const uint8_t*, const Loc&, hipStream_t) {}
bool launch_standalone_instances(int, uint64_t, void*, const FastOp&, const uint8_t*, const Loc&, hipStream_t,
                                 const Instances&) {
  return true;
}
hipError_t jit_launch(hipFunction_t, int, int, bool, void*, const double2*, uint64_t, uint64_t, hipStream_t, uint32_t,
                      uint32_t, uint64_t, uint64_t) {
  return hipSuccess;
}

}  // namespace qr

int main(int argc, char** argv) {
  struct {
    const char* name;
    void (*run)();
  } const checks[] = {{"many_draws", many_draws}, {"many_draws_of_programs", many_draws_of_programs},
                {"halfway_blocks", halfway_blocks}};
  for (const auto& c : checks)
    if (argc == 2 && std::strcmp(argv[1], c.name) == 0) {
      c.run();
      if (!failures) std::printf("ok\n");
      return failures ? 1 : 0;
    }
  return 2;
}

// sampler.cpp — measure_all's sampling step: SuperPosition::measure (super_positions.rs:332-342)
// for a batch of injected draws, reproducing the reference's sequential left fold bit for bit.
//
// The reference draws u and returns the first index i with u < S_i, where
// S_i = fl(S_{i-1} + (re_i * re_i + im_i * im_i)) is folded in index order (no fused
// operations), or None when u >= S_last. The fold is rebuilt exactly in parallel:
//  1. block masses (any order) give approximate block starts and so the binade e in which each
//     block's fold most likely runs, and which blocks cross into the next one;
//  2. per block, exact integer sums of rint(p_i / 2^(e-52)) for e and its two neighbours; the
//     probabilities of the crossing blocks and of those with a halfway case go to the host in
//     the same step;
//  3. on the host, the exact start of every block, in order: while a block's fold stays in the
//     binade of its start, fl(S + p) = S + rint(p / U) * U exactly (U = 2^(e-52)), so its end is
//     its start plus the integer sum. Blocks that cross into the next binade, hold a halfway
//     case, or start at 0 are folded sequentially on the host from their exact start;
//  4. each draw goes to the block whose exact fold range holds it; blocks of the integer kind
//     resolve their draws on the device from an exact in-block prefix sum, the others on the
//     host by the sequential fold.
// Two reads of the state bound large states (4.9 ms at 30 qubits, complex128); small ones are
// bound by the host's fold (about 1 ns per amplitude) and the waits for the device. So everything
// the host reads is written by the kernels straight into pinned memory, once per step.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "engine.hpp"
#include "kernels.hpp"
#include "runtime.hpp"

namespace qr {

namespace {

constexpr double kTwo53 = 9007199254740992.0;

// Folds the probabilities p of a block in index order from `s`, exactly as the reference does
// (binary64, no contraction). Assigns each u[d] (sorted, d in [first, last)) the first index,
// counted from b0, whose fold value exceeds it, and stops there if `place` alone is asked for.
// Returns the fold's end value.
double fold(const double* p, uint64_t len, double s, const double* u, uint64_t& first, uint64_t last, uint64_t* out,
            uint64_t b0, bool place) {
#pragma clang fp contract(off)
  uint64_t d = first;
  for (uint64_t i = 0; i < len; ++i) {
    if (d == last) {
      if (place) break;
      for (; i < len; ++i) s = s + p[i];
      break;
    }
    s = s + p[i];
    while (d < last && u[d] < s) out[d++] = b0 + i;
  }
  first = d;
  return s;
}

// States of up to 2^kHostFoldBits amplitudes are folded on the host as a whole: one launch and one
// wait (13 qubits, 500 shots: 136 -> 24 us); from 2^16 on the fold takes longer than the
// parallel steps.
constexpr uint32_t kHostFoldBits = 15;

// Amplitudes per block, as a power of two: the crossing blocks (about one per binade of the total,
// up to 30) are folded at 1 ns per amplitude, while every block costs the host a few ns and the
// device a workgroup. 2^12, the least the device resolves draws in, up to 2^27 amplitudes; wider
// above, so that there are 2^16 blocks at 30 qubits.
int block_bits(uint32_t n) { return std::min(14, std::max(12, (int)n - 15)); }

// Places for the probabilities of blocks with a halfway case. A complex128 state of full mantissas
// has about one such case per binade of its total (5 to 9 blocks at 20 to 24 qubits); a complex64
// state, whose probabilities have 48 bits, about 32 (44 / 66 / 80 blocks at 20 / 22 / 24 qubits).
// 1000 draws on such states of 22 / 24 / 26 qubits, 0.40 / 0.45 / 0.84 ms; with 48 places and the
// other blocks fetched one by one 1.14 / 1.14 / 1.80.
uint32_t tie_places(int prec) { return prec == 0 ? 48 : 96; }

struct BlockFold {
  double start = 0.0;
  int e = 0;         // binade of the integer fold
  bool exact = false;  // integer fold on the device (else sequential on the host)
};

}  // namespace

// A stable counting sort by leading digits, then by value inside each of the buckets: for draws
// spread over [0, 1) a few ns each (measure_all with 1e5 draws on 2^25 amplitudes 8.6 -> 1.6 ms,
// most of it std::stable_sort before).
void sort_draws(const double* u, uint64_t shots, std::vector<double>& us, std::vector<uint64_t>& perm) {
  us.resize(shots);
  perm.resize(shots);
  uint64_t B = 1;
  while (B < shots && B < (1u << 16)) B *= 2;
  std::vector<uint64_t> at(B + 1, 0);
  auto bucket = [&](double x) -> uint64_t {  // monotone in x; anything outside [0, 1) is clamped
    if (!(x > 0.0)) return 0;
    if (!(x < 1.0)) return B - 1;
    return (uint64_t)(x * (double)B);
  };
  for (uint64_t s = 0; s < shots; ++s) at[bucket(u[s]) + 1]++;
  for (uint64_t b = 0; b < B; ++b) at[b + 1] += at[b];
  std::vector<uint64_t> next(at.begin(), at.end() - 1);
  for (uint64_t s = 0; s < shots; ++s) {
    const uint64_t q = next[bucket(u[s])]++;
    perm[q] = s;
    us[q] = u[s];
  }
  for (uint64_t b = 0; b < B; ++b) {
    const uint64_t f = at[b], l = at[b + 1];
    if (l - f > 32) {
      std::stable_sort(perm.begin() + f, perm.begin() + l, [&](uint64_t x, uint64_t y) { return u[x] < u[y]; });
      for (uint64_t q = f; q < l; ++q) us[q] = u[perm[q]];
      continue;
    }
    for (uint64_t q = f + 1; q < l; ++q) {  // insertion: the few draws of a bucket
      const double x = us[q];
      const uint64_t px = perm[q];
      uint64_t r = q;
      for (; r > f && x < us[r - 1]; --r) {
        us[r] = us[r - 1];
        perm[r] = perm[r - 1];
      }
      us[r] = x;
      perm[r] = px;
    }
  }
}

// us: draws in ascending order (no NaN); res: shots slots, UINT64_MAX = None.
void sample_exact_parallel(qr_state* st, const std::vector<double>& us, std::vector<uint64_t>& res) {
  const uint64_t shots = us.size();
  res.assign(shots, ~0ull);
  if (shots == 0) return;
  if (st->n <= kHostFoldBits) {
    PinnedLease pin(st->dim * 8);
    double* p = (double*)pin.data();
    hip_check(launch_gather_probs(st->prec, st->amp, (int)st->n, nullptr, 1, p, st->stream), "probabilities");
    hip_check(hipStreamSynchronize(st->stream), "sync");
    uint64_t d = 0;
    fold(p, st->dim, 0.0, us.data(), d, shots, res.data(), 0, true);
    return;
  }
  const int bb = block_bits(st->n);
  const uint64_t nblk = st->dim >> bb, len = 1ull << bb;
  // ---- 1. block masses
  PinnedLease pin_mass(nblk * 8);
  const double* mass = (const double*)pin_mass.data();
  {
    ProfScope ps_(st, "block_mass", (double)st->dim * st->bytes_per_amp());
    hip_check(launch_block_mass(st->prec, st->amp, st->dim, bb, (double*)pin_mass.data(), st->stream), "block mass");
  }
  hip_check(hipStreamSynchronize(st->stream), "sync");
  // ---- 2. candidate binades from the approximate (compensated) prefix, and the blocks whose fold
  // leaves its binade, give or take the masses' rounding; then exact unit sums and these blocks'
  // probabilities
  constexpr uint64_t kMostFolds = 128;  // far above one per binade; further ones are fetched singly
  PinnedLease pin(nblk * (4 + 3 * 8 + 4) + 64 + kMostFolds * 8 + 4);
  double* sums = (double*)pin.data();
  uint64_t* list = (uint64_t*)(sums + 3 * nblk);
  uint32_t* flags = (uint32_t*)(list + kMostFolds);
  int32_t* ebase = (int32_t*)(flags + nblk);
  uint64_t folds = 0;
  {
    double acc = 0.0, comp = 0.0;
    double low = 0.0, high = 0.0;  // [low, high): the binade e of the last start
    int e = 0;
    for (uint64_t b = 0; b < nblk; ++b) {
      const double a = acc + comp;
      const bool ok = a > 0.0 && std::isfinite(a);
      if (ok && !(a >= low && a < high)) {
        e = std::ilogb(a);
        low = std::ldexp(1.0, e);
        high = 2.0 * low;
      }
      ebase[b] = ok ? e - 1 : -2000;
      const double t = acc + mass[b];
      comp += std::fabs(acc) >= std::fabs(mass[b]) ? (acc - t) + mass[b] : (mass[b] - t) + acc;
      acc = t;
      const double end = acc + comp;
      constexpr double kSlack = 1e-10;
      const bool inside = ok && a * (1.0 - kSlack) >= low && end * (1.0 + kSlack) < high;
      if (mass[b] != 0.0 && !inside && folds < kMostFolds) list[folds++] = b;
    }
  }
  // blocks with a halfway case: their number isn't known before the kernel runs
  const uint32_t most_ties = (uint32_t)std::min<uint64_t>(nblk, tie_places(st->prec));
  PinnedLease pin_probs((folds + most_ties) * len * 8 + most_ties * 8);
  const double* probs = (const double*)pin_probs.data();
  const double* tie_probs = probs + folds * len;
  uint64_t* tie_block = (uint64_t*)(tie_probs + most_ties * len);
  std::fill(tie_block, tie_block + most_ties, ~0ull);
  ebase[nblk] = 0;  // their counter travels behind the binades
  st->aux.reserve((nblk + 1) * 4);
  hip_check(hipMemcpyAsync(st->aux.p, ebase, (nblk + 1) * 4, hipMemcpyHostToDevice, st->stream), "H2D");
  const TieBlocks tie{(uint32_t*)st->aux.p + nblk, most_ties, tie_block, (double*)tie_probs};
  {
    ProfScope ps_(st, "block_exact_sums", (double)st->dim * st->bytes_per_amp());
    hip_check(launch_block_exact_sums(st->prec, st->amp, st->dim, bb, (const int32_t*)st->aux.p, sums, flags,
                                      tie, st->stream),
              "block exact sums");
  }
  hip_check(launch_gather_probs(st->prec, st->amp, bb, list, (uint32_t)folds, (double*)pin_probs.data(), st->stream),
            "probabilities");
  hip_check(hipStreamSynchronize(st->stream), "sync");
  // what is in hand of block b, or null
  auto fetched = [&](uint64_t b) -> const double* {
    const uint64_t* at = std::lower_bound(list, list + folds, b);
    if (at != list + folds && *at == b) return probs + (at - list) * len;
    const uint64_t* t = std::find(tie_block, tie_block + most_ties, b);
    return t != tie_block + most_ties ? tie_probs + (t - tie_block) * len : nullptr;
  };
  // the blocks with a halfway case that found no place, in one more launch (as many as 16 MB hold)
  std::vector<uint64_t> rest;
  if (tie_block[most_ties - 1] != ~0ull)
    for (uint64_t b = 0; b < nblk && rest.size() < (2ull << 20) / len; ++b)
      if ((flags[b] & 2u) && mass[b] != 0.0 && !fetched(b)) rest.push_back(b);
  PinnedLease pin_rest;
  if (!rest.empty()) {
    pin_rest.reserve(rest.size() * (len + 1) * 8);
    uint64_t* rest_list = (uint64_t*)(pin_rest.data() + rest.size() * len * 8);
    std::copy(rest.begin(), rest.end(), rest_list);
    hip_check(launch_gather_probs(st->prec, st->amp, bb, rest_list, (uint32_t)rest.size(), (double*)pin_rest.data(),
                                  st->stream),
              "probabilities");
    hip_check(hipStreamSynchronize(st->stream), "sync");
  }
  // ---- 3. exact block starts, in order
  std::vector<BlockFold> bf(nblk);
  std::vector<double> ends(nblk);
  PinnedLease pin_one;
  // the probabilities of block b: fetched ahead, else now
  auto probs_of = [&](uint64_t b) -> const double* {
    if (const double* p = fetched(b)) return p;
    const auto r = std::lower_bound(rest.begin(), rest.end(), b);
    if (r != rest.end() && *r == b) return (const double*)pin_rest.data() + (r - rest.begin()) * len;
    pin_one.reserve(len * 8 + 8);
    uint64_t* one = (uint64_t*)(pin_one.data() + len * 8);
    *one = b;
    hip_check(launch_gather_probs(st->prec, st->amp, bb, one, 1, (double*)pin_one.data(), st->stream), "probabilities");
    hip_check(hipStreamSynchronize(st->stream), "sync");
    return (const double*)pin_one.data();
  };
  double s = 0.0;
  int e = 0;
  double low = 0.0, high = 0.0, unit = 0.0, scale = 0.0;  // of the binade [low, high) = 2^e [1, 2)
  for (uint64_t b = 0; b < nblk; ++b) {
    BlockFold& f = bf[b];
    f.start = s;
    if (mass[b] == 0.0) {  // every p is +0: the fold does not move
      ends[b] = s;
      continue;
    }
    if (s > 0.0 && std::isfinite(s)) {
      if (!(s >= low && s < high)) {
        e = std::ilogb(s);
        low = std::ldexp(1.0, e);
        high = 2.0 * low;
        unit = std::ldexp(1.0, e - 52);
        scale = std::ldexp(1.0, 52 - e);
      }
      const int c = e - ebase[b];
      if (c >= 0 && c <= 2 && !((flags[b] >> c) & 1u)) {
        const double m = s * scale;  // integer in [2^52, 2^53), exact (e is in [-960, 52] here)
        const double tot = sums[3 * b + c];
        if (std::isfinite(tot) && m + tot < kTwo53) {
          f.exact = true;
          f.e = e;
          s = (m + tot) * unit;
          ends[b] = s;
          continue;
        }
      }
    }
    uint64_t none = 0;
    s = fold(probs_of(b), len, s, nullptr, none, 0, nullptr, 0, false);
    ends[b] = s;
  }
  // ---- 4. draws to blocks: block b holds the draws with start_b <= u < end_b (the first block
  // whose end exceeds u); draws at or above the total are None. A job takes at most kJobDraws.
  constexpr uint64_t kJobDraws = 2048;
  std::vector<ExactJob> jobs;
  jobs.reserve(std::min(shots, nblk) + shots / kJobDraws);
  const double* const u = us.data();
  uint64_t d = 0;
  while (d < shots) {
    const uint64_t b = (uint64_t)(std::upper_bound(ends.begin(), ends.end(), u[d]) - ends.begin());
    if (b >= nblk) break;
    const double end = ends[b];
    uint64_t last = d;
    while (last < shots && u[last] < end) ++last;
    const BlockFold& f = bf[b];
    if (f.exact) {
      const double un = std::ldexp(1.0, f.e - 52);
      for (uint64_t j = d; j < last; j += kJobDraws)
        jobs.push_back(ExactJob{b, f.start / un, un, std::ldexp(1.0, 52 - f.e), j, std::min(last, j + kJobDraws)});
    } else {
      uint64_t at = d;
      fold(probs_of(b), len, f.start, u, at, last, res.data(), b << bb, true);
    }
    d = last;
  }
  // a slice of the jobs at a time: their draws (and those between them) and bins are pinned
  for (size_t j0 = 0, j1; j0 < jobs.size(); j0 = j1) {
    const uint64_t d0 = jobs[j0].first;
    for (j1 = j0 + 1; j1 < jobs.size() && jobs[j1].last - d0 <= kDrawSlice && j1 - j0 < kDrawSlice / 8;) ++j1;
    const uint64_t count = jobs[j1 - 1].last - d0;
    const size_t ub = count * 8, jb = (j1 - j0) * sizeof(ExactJob);
    PinnedLease pin_jobs(2 * ub + jb);
    uint64_t* got = (uint64_t*)(pin_jobs.data() + ub + jb);
    std::memcpy(pin_jobs.data(), us.data() + d0, ub);
    ExactJob* up = (ExactJob*)(pin_jobs.data() + ub);
    for (size_t j = j0; j < j1; ++j) {
      up[j - j0] = jobs[j];
      up[j - j0].first -= d0;
      up[j - j0].last -= d0;
    }
    st->aux.reserve(ub + jb);
    const uint8_t* dblob = (const uint8_t*)st->aux.p;
    hip_check(hipMemcpyAsync(st->aux.p, pin_jobs.data(), ub + jb, hipMemcpyHostToDevice, st->stream), "H2D");
    {
      ProfScope ps_(st, "sample_exact_blocks", (double)(j1 - j0) * (double)len * st->bytes_per_amp());
      hip_check(launch_sample_exact_blocks(st->prec, st->amp, st->dim, bb, (const ExactJob*)(dblob + ub), j1 - j0,
                                           (const double*)dblob, got, st->stream),
                "sample exact blocks");
    }
    hip_check(hipStreamSynchronize(st->stream), "sync");
    for (size_t j = j0; j < j1; ++j)
      std::copy(got + (jobs[j].first - d0), got + (jobs[j].last - d0), res.begin() + jobs[j].first);
  }
}

}  // namespace qr

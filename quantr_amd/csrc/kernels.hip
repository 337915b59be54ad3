// kernels.hip — gfx950 kernels of the state-vector engine (wave64, CDNA4).
//
// State layout: 2^n amplitudes, interleaved (re, im), index i = sum_w bit_w * 2^(n-1-w)
// (wire 0 = most significant bit, product_states.rs:191-215). complex128 amplitudes are
// loaded as one 16-byte dwordx4, complex64 as one 8-byte dwordx2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "kernels.hpp"
#include "tile_ops.hpp"

namespace qr {
namespace dev {

// Inserts a zero bit at each position of `sorted_bits` (ascending) into x.
__device__ __forceinline__ uint64_t insert_zero_bits(uint64_t x, const uint8_t* sorted_bits, int nb) {
  for (int q = 0; q < nb; ++q) {
    const uint64_t b = sorted_bits[q];
    const uint64_t lo = x & ((1ull << b) - 1);
    x = ((x >> b) << (b + 1)) | lo;
  }
  return x;
}

// =====================================================================================
// |0...0> (SuperPosition::new_unchecked, super_positions_unchecked.rs:39-46)
// =====================================================================================
template <typename R>
__global__ void k_init_basis(typename CT<R>::T* __restrict__ psi, uint64_t dim, uint64_t one_at, int nt) {
  using C = typename CT<R>::T;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += stride) {
    C v;
    v.x = (i == one_at) ? R(1) : R(0);
    v.y = R(0);
    if (nt) store_nt(&psi[i], v);
    else psi[i] = v;
  }
}

// =====================================================================================
// Exact per-gate sweep: new[r] = sum over inputs j in ascending global index order of
// M[r][j] * a[j], the first product taken as is and the rest added, complex products in
// the textbook form with no fused multiply-add (Circuit::apply_gate, simulation.rs:64-180).
// Inputs whose custom image is None keep their amplitude (simulation.rs:120-133).
// One thread per group of 2^K amplitudes that differ only in the acting bits.
// =====================================================================================
template <typename R, int KR>
__global__ void k_exact(typename CT<R>::T* __restrict__ psi, uint64_t ngroups, ExactArgs a,
                        const double2* __restrict__ M) {
#pragma clang fp contract(off)
  using C = typename CT<R>::T;
  const int K = a.K;
  const int dim = 1 << K;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < ngroups; g += stride) {
    const uint64_t base = insert_zero_bits(g, a.sorted_bits, K);
    if (KR > 0) {
      C in[1 << (KR > 0 ? KR : 1)];
#pragma unroll
      for (int j = 0; j < (1 << KR); ++j)
        if (j < dim) in[j] = psi[base + a.off[j]];
      C out[1 << (KR > 0 ? KR : 1)];
#pragma unroll
      for (int r = 0; r < (1 << KR); ++r) {
        if (r >= dim) continue;
        if ((a.keep >> r) & 1) {
          out[r] = in[r];
          continue;
        }
        R acc_re = R(0), acc_im = R(0);
        bool first = true;
#pragma unroll
        for (int oi = 0; oi < (1 << KR); ++oi) {
          if (oi >= dim) continue;
          const int j = a.order[oi];
          if (!((a.some >> j) & 1)) continue;
          const double2 m = M[r * dim + j];
          const R mr = (R)m.x, mi = (R)m.y;
          C v;
#pragma unroll
          for (int jj = 0; jj < (1 << KR); ++jj)
            if (jj == j) v = in[jj];
          const R pr = mr * v.x - mi * v.y;
          const R pi = mr * v.y + mi * v.x;
          if (first) {
            acc_re = pr;
            acc_im = pi;
            first = false;
          } else {
            acc_re = acc_re + pr;
            acc_im = acc_im + pi;
          }
        }
        out[r].x = acc_re;
        out[r].y = acc_im;
      }
#pragma unroll
      for (int j = 0; j < (1 << KR); ++j)
        if (j < dim) psi[base + a.off[j]] = out[j];
    }
  }
}

// Generic exact sweep for wide custom gates (K > 4): inputs re-read from memory.
template <typename R>
__global__ void k_exact_wide(typename CT<R>::T* __restrict__ psi, typename CT<R>::T* __restrict__ tmp,
                             uint64_t ngroups, ExactWideArgs a, const double2* __restrict__ M,
                             const uint64_t* __restrict__ off, const uint32_t* __restrict__ order,
                             const uint8_t* __restrict__ flags) {
#pragma clang fp contract(off)
  using C = typename CT<R>::T;
  const int dim = 1 << a.K;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  // flags[j] bit0 = some, bit1 = keep
  for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < ngroups; g += stride) {
    const uint64_t base = insert_zero_bits(g, a.sorted_bits, a.K);
    C* out = tmp + ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * (uint64_t)dim;
    for (int r = 0; r < dim; ++r) {
      if (flags[r] & 2) {
        out[r] = psi[base + off[r]];
        continue;
      }
      R acc_re = R(0), acc_im = R(0);
      bool first = true;
      for (int oi = 0; oi < dim; ++oi) {
        const int j = (int)order[oi];
        if (!(flags[j] & 1)) continue;
        const double2 m = M[(uint64_t)r * dim + j];
        const C v = psi[base + off[j]];
        const R mr = (R)m.x, mi = (R)m.y;
        const R pr = mr * v.x - mi * v.y;
        const R pi = mr * v.y + mi * v.x;
        if (first) {
          acc_re = pr;
          acc_im = pi;
          first = false;
        } else {
          acc_re = acc_re + pr;
          acc_im = acc_im + pi;
        }
      }
      C o;
      o.x = acc_re;
      o.y = acc_im;
      out[r] = o;
    }
    for (int r = 0; r < dim; ++r) psi[base + off[r]] = out[r];
  }
}

// =====================================================================================
// Fast standalone sweeps (fused multiply-add allowed)
// =====================================================================================

template <typename R>
__device__ __forceinline__ void cmul_acc(R& xr, R& xi, R ur, R ui, R vr, R vi) {
  xr = fma(ur, vr, fma(-ui, vi, xr));
  xi = fma(ur, vi, fma(ui, vr, xi));
}

// 2x2 on target bit t for every pair whose control bits are all 1.
template <typename R>
__global__ void k_dense1(typename CT<R>::T* __restrict__ psi, uint64_t npairs, int t, uint64_t cmask,
                         double2 u00, double2 u01, double2 u10, double2 u11) {
  using C = typename CT<R>::T;
  const uint64_t tb = 1ull << t;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const R a_r = u00.x, a_i = u00.y, b_r = u01.x, b_i = u01.y, c_r = u10.x, c_i = u10.y, d_r = u11.x,
          d_i = u11.y;
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < npairs; p += stride) {
    const uint64_t i0 = ((p >> t) << (t + 1)) | (p & (tb - 1));
    if ((i0 & cmask) != cmask) continue;
    const uint64_t i1 = i0 | tb;
    const C x = psi[i0], y = psi[i1];
    R o0r = 0, o0i = 0, o1r = 0, o1i = 0;
    cmul_acc(o0r, o0i, a_r, a_i, (R)x.x, (R)x.y);
    cmul_acc(o0r, o0i, b_r, b_i, (R)y.x, (R)y.y);
    cmul_acc(o1r, o1i, c_r, c_i, (R)x.x, (R)x.y);
    cmul_acc(o1r, o1i, d_r, d_i, (R)y.x, (R)y.y);
    C r0, r1;
    r0.x = o0r;
    r0.y = o0i;
    r1.x = o1r;
    r1.y = o1i;
    psi[i0] = r0;
    psi[i1] = r1;
  }
}

// diag(d0, d1) on bit t where the control bits are all 1.
template <typename R>
__global__ void k_diag1(typename CT<R>::T* __restrict__ psi, uint64_t dim, int t, uint64_t cmask,
                        double2 d0, double2 d1) {
  using C = typename CT<R>::T;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += stride) {
    if ((i & cmask) != cmask) continue;
    const double2 d = ((i >> t) & 1) ? d1 : d0;
    const C x = psi[i];
    C y;
    y.x = (R)d.x * x.x - (R)d.y * x.y;
    y.y = (R)d.x * x.y + (R)d.y * x.x;
    psi[i] = y;
  }
}

// Dense 2^k x 2^k on k target bits (+ controls); one thread per group.
template <typename R>
__global__ void k_densek(typename CT<R>::T* __restrict__ psi, typename CT<R>::T* __restrict__ tmp,
                         uint64_t ngroups, DenseKArgs a, const double2* __restrict__ M,
                         const uint64_t* __restrict__ off) {
  using C = typename CT<R>::T;
  const int dim = 1 << a.k;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < ngroups; g += stride) {
    const uint64_t base = insert_zero_bits(g, a.sorted_bits, a.k);
    if ((base & a.cmask) != a.cmask) continue;
    C* out = tmp + ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * (uint64_t)dim;
    for (int r = 0; r < dim; ++r) {
      R ar = 0, ai = 0;
      for (int j = 0; j < dim; ++j) {
        const double2 m = M[(uint64_t)r * dim + j];
        const C v = psi[base + off[j]];
        cmul_acc(ar, ai, (R)m.x, (R)m.y, (R)v.x, (R)v.y);
      }
      C o;
      o.x = ar;
      o.y = ai;
      out[r] = o;
    }
    for (int r = 0; r < dim; ++r) psi[base + off[r]] = out[r];
  }
}

// Dense 2^K x 2^K on K <= 4 target bits (+ controls) with the group in registers: one thread
// per group of 2^K amplitudes, which it reads once, transforms and writes back in place.
// off[j] is the offset of local basis state j (MSB-first local index). Instance blockIdx.y has its
// state and its table at fixed strides: 500 states of 2^12 amplitudes with a table each take one
// launch (1.2 ms of launches before).
template <typename R, int K>
__global__ __launch_bounds__(256) void k_densek_reg(typename CT<R>::T* __restrict__ psi, uint64_t ngroups, DenseKArgs a,
                                                    const double2* __restrict__ M, const uint64_t* __restrict__ off,
                                                    Instances in) {
  using C = typename CT<R>::T;
  constexpr int D = 1 << K;
  psi += (uint64_t)blockIdx.y * in.state_stride;
  M += (uint64_t)blockIdx.y * in.table_stride;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < ngroups; g += stride) {
    const uint64_t base = insert_zero_bits(g, a.sorted_bits, K);
    if ((base & a.cmask) != a.cmask) continue;
    C v[D];
#pragma unroll
    for (int j = 0; j < D; ++j) v[j] = psi[base + off[j]];
#pragma unroll
    for (int r = 0; r < D; ++r) {
      R ar = 0, ai = 0;
#pragma unroll
      for (int j = 0; j < D; ++j) {
        const double2 m = M[r * D + j];
        cmul_acc(ar, ai, (R)m.x, (R)m.y, (R)v[j].x, (R)v[j].y);
      }
      C o;
      o.x = ar;
      o.y = ai;
      psi[base + off[r]] = o;
    }
  }
}

// 2^k diagonal phases over k bits (+ controls).
template <typename R>
__global__ void k_diagk(typename CT<R>::T* __restrict__ psi, uint64_t dim, DiagKArgs a,
                        const double2* __restrict__ D, Instances in) {
  using C = typename CT<R>::T;
  psi += (uint64_t)blockIdx.y * in.state_stride;
  D += (uint64_t)blockIdx.y * in.table_stride;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += stride) {
    if ((i & a.cmask) != a.cmask) continue;
    int l = 0;
    for (int q = 0; q < a.k; ++q) l = (l << 1) | (int)((i >> a.bits[q]) & 1);
    const double2 d = D[l];
    const C x = psi[i];
    C y;
    y.x = (R)d.x * x.x - (R)d.y * x.y;
    y.y = (R)d.x * x.y + (R)d.y * x.x;
    psi[i] = y;
  }
}

// =====================================================================================
// Sampling (SuperPosition::measure, super_positions.rs:332-342) with injected draws.
// =====================================================================================

// Exact left fold: one workgroup streams the probabilities through LDS; thread 0 adds them
// in index order (re*re + im*im, no fused operations) and assigns the sorted draws.
template <typename R>
__global__ __launch_bounds__(1024) void k_sample_fold(const typename CT<R>::T* __restrict__ psi,
                                                      uint64_t dim, const double* __restrict__ u,
                                                      uint64_t shots, uint64_t* __restrict__ out) {
#pragma clang fp contract(off)
  constexpr int CH = 4096;
  __shared__ double p[CH];
  __shared__ int done;
  double cum = 0.0;
  uint64_t d = 0;
  double ud = shots ? u[0] : 0.0;
  if (threadIdx.x == 0) done = (shots == 0);
  __syncthreads();
  for (uint64_t base = 0; base < dim && !done; base += CH) {
    for (int q = threadIdx.x; q < CH; q += blockDim.x) {
      const uint64_t i = base + q;
      double v = 0.0;
      if (i < dim) {
        const double re = (double)psi[i].x, im = (double)psi[i].y;
        v = re * re + im * im;
      }
      p[q] = v;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      const uint64_t cnt = (dim - base < (uint64_t)CH) ? (dim - base) : (uint64_t)CH;
      for (uint64_t q = 0; q < cnt; ++q) {
        cum = cum + p[q];
        while (d < shots && ud < cum) {
          out[d] = base + q;
          ++d;
          ud = (d < shots) ? u[d] : 0.0;
        }
        if (d >= shots) break;
      }
      done = (d >= shots);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (; d < shots; ++d) out[d] = ~0ull;
}

// Parallel path, step 1: probability mass of each block of 2^bb amplitudes (f64).
template <typename R>
__global__ __launch_bounds__(256) void k_block_mass(const typename CT<R>::T* __restrict__ psi,
                                                    uint64_t dim, int bb, double* __restrict__ mass, int nt) {
  __shared__ double red[256];
  const uint64_t b0 = (uint64_t)blockIdx.x << bb;
  const uint64_t len = 1ull << bb;
  double s = 0.0;
  for (uint64_t q = threadIdx.x; q < len; q += blockDim.x) {
    const uint64_t i = b0 + q;
    if (i < dim) {
      typename CT<R>::T v;
      if (nt) load_nt(v, &psi[i]);
      else v = psi[i];
      const double re = (double)v.x, im = (double)v.y;
      s += re * re + im * im;
    }
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) mass[blockIdx.x] = red[0];
}

// ---- Block-parallel exact fold ------------------------------------------------------------
// The reference's fold S_i = fl(S_{i-1} + p_i) is sequential, but inside one binade of S it is
// integer arithmetic: while 2^e <= S < 2^(e+1), every S is a multiple of U = 2^(e-52) and
// fl(S + p) = S + rint(p / U) * U whenever p / U is not exactly halfway between integers
// (round-to-nearest-even would then look at the parity of S). Sums of those integers are exact
// in binary64 while below 2^53, in any order. A block whose whole fold stays in one binade is
// therefore folded exactly by an integer prefix sum; blocks that cross a binade (a few per
// power of two of the cumulative mass) or hold a halfway case are folded sequentially instead.

// rint(p / U) for one amplitude, with p / U = p * scale exact (scale a power of two).
__device__ __forceinline__ double units_of(double p, double scale, bool& tie) {
  const double x = p * scale;
  const double r = rint(x);
  tie = fabs(x - r) == 0.5;
  return r;
}

// Per block b of 2^bb amplitudes: for the three candidate binades e = ebase[b] + c (c = 0, 1, 2)
// the exact sum of rint(p_i * 2^(52-e)) (sums[3b + c]; exact while below 2^53, and at least
// 2^53 exactly when the true sum is) and flags[b] bit c when some p_i * 2^(52-e) is a halfway
// case or e is outside [-960, 52] (then the scaling could overflow or the binade is unusable).
// A complex128 state of full mantissas holds about one halfway case per binade, a complex64 state,
// whose probabilities have 48 bits, about 32: blocks with one in the middle candidate (the binade the
// block most likely starts in) leave their probabilities for the host's fold in the next of tie.most
// places, so that it need not ask for them one by one (complex128, 17 qubits, 1000 draws on a state of
// full mantissas: 228 -> 150 us).
template <typename R>
__global__ __launch_bounds__(256) void k_block_exact_sums(const typename CT<R>::T* __restrict__ psi, uint64_t dim,
                                                          int bb, const int32_t* __restrict__ ebase,
                                                          double* __restrict__ sums, uint32_t* __restrict__ flags,
                                                          int nt, TieBlocks tie) {
#pragma clang fp contract(off)
  __shared__ double red[3][256];
  __shared__ uint32_t fred[256];
  const uint64_t b0 = (uint64_t)blockIdx.x << bb;
  const uint64_t len = 1ull << bb;
  const int e0 = ebase[blockIdx.x];
  double sc[3];
  uint32_t fl = 0;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const int e = e0 + c;
    const bool ok = e >= -960 && e <= 52;
    sc[c] = ok ? ldexp(1.0, 52 - e) : 0.0;
    if (!ok) fl |= 1u << c;
  }
  double acc0 = 0.0, acc1 = 0.0, acc2 = 0.0;
  for (uint64_t q = threadIdx.x; q < len; q += blockDim.x) {
    const uint64_t i = b0 + q;
    if (i >= dim) break;
    typename CT<R>::T v;
    if (nt) load_nt(v, &psi[i]);
    else v = psi[i];
    const double re = (double)v.x, im = (double)v.y;
    const double p = re * re + im * im;
    bool t0, t1, t2;
    acc0 += units_of(p, sc[0], t0);
    acc1 += units_of(p, sc[1], t1);
    acc2 += units_of(p, sc[2], t2);
    fl |= (t0 ? 1u : 0u) | (t1 ? 2u : 0u) | (t2 ? 4u : 0u);
  }
  red[0][threadIdx.x] = acc0;
  red[1][threadIdx.x] = acc1;
  red[2][threadIdx.x] = acc2;
  fred[threadIdx.x] = fl;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
#pragma unroll
      for (int c = 0; c < 3; ++c) red[c][threadIdx.x] += red[c][threadIdx.x + w];
      fred[threadIdx.x] |= fred[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < 3; ++c) sums[3 * (uint64_t)blockIdx.x + c] = red[c][0];
    flags[blockIdx.x] = fred[0];
  }
  if (!(fred[0] & 2u) || e0 + 1 < -960 || e0 + 1 > 52) return;
  __shared__ uint32_t place;
  if (threadIdx.x == 0) place = atomicAdd(tie.count, 1u);
  __syncthreads();
  if (place >= tie.most) return;
  if (threadIdx.x == 0) tie.block[place] = blockIdx.x;
  for (uint64_t q = threadIdx.x; q < len && b0 + q < dim; q += blockDim.x) {
    const double re = (double)psi[b0 + q].x, im = (double)psi[b0 + q].y;
    tie.probs[((uint64_t)place << bb) + q] = re * re + im * im;
  }
}

// Probabilities of whole blocks of 2^bb amplitudes, block list[y] (y itself without a list), for the
// sequential folds on the host: out (pinned host memory) gets 8 bytes per amplitude in place of a
// copy of 16, and every block that will need one travels in one launch.
template <typename R>
__global__ __launch_bounds__(256) void k_gather_probs(const typename CT<R>::T* __restrict__ psi, int bb,
                                                      const uint64_t* __restrict__ list, double* __restrict__ out) {
#pragma clang fp contract(off)
  const uint64_t len = 1ull << bb, b0 = (list ? list[blockIdx.y] : (uint64_t)blockIdx.y) << bb;
  double* dst = out + ((uint64_t)blockIdx.y << bb);
  for (uint64_t q = (uint64_t)blockIdx.x * 256 + threadIdx.x; q < len; q += (uint64_t)gridDim.x * 256) {
    const double re = (double)psi[b0 + q].x, im = (double)psi[b0 + q].y;
    dst[q] = re * re + im * im;
  }
}

// One workgroup per job: the block's exact fold values S_i = (m_start + prefix_i) * U from an
// integer prefix sum (binary64, exact below 2^53) in LDS, 4096 amplitudes at a time; each draw u of
// the job (in [S_start, S_end)) gets the first index i with u < S_i by a search among them. A
// thread per draw keeps a block that holds most of the draws (a state near a basis state) from
// placing them one after the other (1e5 draws on 2^25 amplitudes 0.19 -> 0.06 ms).
template <typename R>
__global__ __launch_bounds__(256) void k_sample_exact_blocks(const typename CT<R>::T* __restrict__ psi, uint64_t dim,
                                                             int bb, const ExactJob* __restrict__ jobs,
                                                             const double* __restrict__ u,
                                                             uint64_t* __restrict__ out) {
#pragma clang fp contract(off)
  constexpr int CH = 4096, PER = 16;
  __shared__ double pv[CH + CH / PER];  // one pad word per 16 against bank conflicts
  __shared__ double scan[256];
  const ExactJob job = jobs[blockIdx.x];
  const uint64_t b0 = job.block << bb;
  const uint64_t len = 1ull << bb;
  const uint32_t t = threadIdx.x;
  auto at = [](uint32_t q) { return q + q / PER; };
  double carry = job.m_start;  // integer count of units before the chunk
  for (uint64_t c0 = 0; c0 < len; c0 += CH) {
    for (uint32_t q = t; q < CH; q += 256) {
      const uint64_t i = b0 + c0 + q;
      double p = 0.0;
      if (c0 + q < len && i < dim) {
        const double re = (double)psi[i].x, im = (double)psi[i].y;
        p = re * re + im * im;
      }
      pv[at(q)] = p;
    }
    __syncthreads();
    double r[PER];
    double tsum = 0.0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      bool tie;
      r[j] = units_of(pv[at(t * PER + j)], job.scale, tie);
      tsum += r[j];
    }
    // inclusive scan of the thread sums (Hillis-Steele; integer-valued, exact)
    scan[t] = tsum;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
      const double add = t >= (uint32_t)off ? scan[t - off] : 0.0;
      __syncthreads();
      scan[t] += add;
      __syncthreads();
    }
    double run = carry + (scan[t] - tsum);
    const double chunk_total = scan[255];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      run += r[j];
      pv[at(t * PER + j)] = run * job.unit;
    }
    __syncthreads();
    // the chunk's draws: those from its start on (every draw of the job is at or above the first
    // chunk's) that lie below its end
    const double s0 = carry * job.unit, s1 = pv[at(CH - 1)];
    for (uint64_t d = job.first + t; d < job.last; d += 256) {
      const double ud = u[d];
      if (!(ud < s1) || (c0 > 0 && ud < s0)) continue;
      uint32_t lo = 0, hi = CH - 1;  // S_hi > u
      while (lo < hi) {
        const uint32_t mid = (lo + hi) / 2;
        if (ud < pv[at(mid)]) hi = mid;
        else lo = mid + 1;
      }
      out[d] = b0 + c0 + lo;
    }
    carry += chunk_total;
    __syncthreads();
  }
}

// =====================================================================================
// Reductions (f64 accumulation; complex64 promoted before multiplying)
// =====================================================================================

template <typename R>
__global__ __launch_bounds__(256) void k_norm_partial(const typename CT<R>::T* __restrict__ psi,
                                                      uint64_t dim, double* __restrict__ part) {
  __shared__ double red[256];
  double s = 0.0, comp = 0.0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += stride) {
    const double re = (double)psi[i].x, im = (double)psi[i].y;
    const double v = re * re + im * im;
    const double y = v - comp;
    const double t = s + y;
    comp = (t - s) - y;
    s = t;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Gradient term of one rotation gate: sum_j conj(lam_j) (G psi)_j for G in {X, Y, Z, I} on bit t.
// Returns partial (re, im). Y: (Y psi)_j = -i (-1)^{bit_t(j)} psi_{j^t}; Z: (-1)^{bit_t(j)} psi_j.
template <typename R>
__global__ __launch_bounds__(256) void k_gen_partial(const typename CT<R>::T* __restrict__ lam,
                                                     const typename CT<R>::T* __restrict__ psi, uint64_t dim,
                                                     int t, int gen, double2* __restrict__ part) {
  __shared__ double rr[256], ri[256];
  double sr = 0.0, si = 0.0;
  const uint64_t tb = 1ull << t;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < dim; j += stride) {
    double gr, gi;
    if (gen == 1) {
      gr = (double)psi[j ^ tb].x;
      gi = (double)psi[j ^ tb].y;
    } else if (gen == 2) {
      const double s = (j & tb) ? -1.0 : 1.0;
      const double pr = (double)psi[j ^ tb].x * s, pi = (double)psi[j ^ tb].y * s;
      gr = pi;   // -i * (pr + i pi) = pi - i pr
      gi = -pr;
    } else if (gen == 3) {
      const double s = (j & tb) ? -1.0 : 1.0;
      gr = (double)psi[j].x * s;
      gi = (double)psi[j].y * s;
    } else {
      gr = (double)psi[j].x;
      gi = (double)psi[j].y;
    }
    const double lr = (double)lam[j].x, li = -(double)lam[j].y;
    sr += lr * gr - li * gi;
    si += lr * gi + li * gr;
  }
  rr[threadIdx.x] = sr;
  ri[threadIdx.x] = si;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      rr[threadIdx.x] += rr[threadIdx.x + w];
      ri[threadIdx.x] += ri[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = make_double2(rr[0], ri[0]);
}

// lam = O psi for a whole Pauli sum in one pass: each output adds one product per X-mask group
// (groups and terms read with uniform loads). The first `nplain` groups are one real term without
// signs: their partners are fetched four at a time, since small states leave a CU one wavefront
// per SIMD, which waited for each partner in turn (25 terms, 13 qubits, complex64: 9.8 -> 7.2 us; 39 terms, 20 qubits, complex128: 37 -> 24 us).
// With `part`, the workgroup's share of Re <psi|lam> goes there as well, which saves a batch a
// pass and a launch.
template <typename R>
__global__ __launch_bounds__(256) void k_pauli_sum(typename CT<R>::T* __restrict__ lam,
                                                   const typename CT<R>::T* __restrict__ psi, uint64_t dim,
                                                   const PauliGroup* __restrict__ groups, int ngroups, int nplain,
                                                   const PauliZTerm* __restrict__ terms, double* __restrict__ part) {
  using C = typename CT<R>::T;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  double dot = 0.0;
  for (uint64_t o = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; o < dim; o += stride) {
    double yr = 0.0, yi = 0.0;
    int g = 0;
    for (; g + 4 <= nplain; g += 4) {
      C v[4];
      double c[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = psi[o ^ groups[g + q].xm];
        c[q] = terms[groups[g + q].first].cr;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        yr = fma(c[q], (double)v[q].x, yr);
        yi = fma(c[q], (double)v[q].y, yi);
      }
    }
    for (; g < ngroups; ++g) {
      const uint64_t j = o ^ groups[g].xm;
      const C v = psi[j];
      double fr = 0.0, fi = 0.0;
      const uint32_t t0 = groups[g].first, t1 = t0 + groups[g].count;
      for (uint32_t t = t0; t < t1; ++t) {
        const bool neg = __popcll(j & terms[t].zm) & 1;
        fr += neg ? -terms[t].cr : terms[t].cr;
        fi += neg ? -terms[t].ci : terms[t].ci;
      }
      const double pr = (double)v.x, pi = (double)v.y;
      yr += fr * pr - fi * pi;
      yi += fr * pi + fi * pr;
    }
    C w;
    w.x = (R)yr;
    w.y = (R)yi;
    lam[o] = w;
    if (part) dot += (double)psi[o].x * yr + (double)psi[o].y * yi;
  }
  if (!part) return;
  __shared__ double red[256];
  red[threadIdx.x] = dot;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// |0...0> in the states of a batch: instance blockIdx.y's amplitudes start at byte base[y] of the
// pool and number 2^bits[y].
template <typename R>
__global__ __launch_bounds__(256) void k_init_batch(uint8_t* __restrict__ pool, const uint64_t* __restrict__ base,
                                                    const uint32_t* __restrict__ bits) {
  using C = typename CT<R>::T;
  C* psi = reinterpret_cast<C*>(pool + base[blockIdx.y]);
  const uint64_t dim = 1ull << bits[blockIdx.y];
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < dim; i += (uint64_t)gridDim.x * 256) {
    psi[i].x = (R)(i == 0 ? 1 : 0);
    psi[i].y = (R)0;
  }
}

// |0...0> in each of `count` states of dim amplitudes laid out back to back.
template <typename R>
__global__ __launch_bounds__(256) void k_init_instances(typename CT<R>::T* __restrict__ psi, uint64_t dim,
                                                        uint64_t total) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    psi[i].x = (R)((i & (dim - 1)) == 0 ? 1 : 0);
    psi[i].y = (R)0;
  }
}

// One workgroup per state (states back to back, `stride` amplitudes apart): its draws
// u[off[y] .. off[y+1]) (ascending) placed by the left fold of its probabilities in index
// order, as k_sample_fold does for one state: probabilities in parallel, the fold in one lane.
// The fold is a chain of additions: sixteen values at a time come from LDS while the sixteen
// before are added, and draws are looked at once for each sixteen (the fold does not decrease, so
// a draw below its end, or an unordered one, is found inside): 500 states of 2^12 amplitudes
// took 690 us with an LDS read and a comparison in every step of the chain.
template <typename R>
__global__ __launch_bounds__(256) void k_sample_fold_instances(const typename CT<R>::T* __restrict__ psi,
                                                               uint64_t dim, uint64_t stride,
                                                               const double* __restrict__ u,
                                                               const uint64_t* __restrict__ off,
                                                               uint64_t* __restrict__ out) {
#pragma clang fp contract(off)
  constexpr int CH = 2048, ST = 16;
  __shared__ double p[CH + ST];  // zeros behind the chunk: the last values fetched ahead
  __shared__ int done;
  const typename CT<R>::T* ps = psi + (uint64_t)blockIdx.x * stride;
  const uint64_t d1 = off[blockIdx.x + 1];
  uint64_t d = off[blockIdx.x];
  double cum = 0.0, ud = d < d1 ? u[d] : 0.0;
  if (threadIdx.x == 0) done = (d >= d1);
  if (threadIdx.x < ST) p[CH + threadIdx.x] = 0.0;
  __syncthreads();
  for (uint64_t base = 0; base < dim && !done; base += CH) {
    for (int q = threadIdx.x; q < CH; q += blockDim.x) {
      const uint64_t i = base + q;
      double v = 0.0;
      if (i < dim) {
        const double re = (double)ps[i].x, im = (double)ps[i].y;
        v = re * re + im * im;
      }
      p[q] = v;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      const int cnt = (int)((dim - base < (uint64_t)CH) ? (dim - base) : (uint64_t)CH);
      double next[ST];
#pragma unroll
      for (int j = 0; j < ST; ++j) next[j] = p[j];
      for (int q = 0; q < cnt && d < d1; q += ST) {
        double s[ST];
#pragma unroll
        for (int j = 0; j < ST; ++j) s[j] = next[j];
#pragma unroll
        for (int j = 0; j < ST; ++j) next[j] = p[q + ST + j];
        // values at and beyond dim are +0 and leave the fold where it is
#pragma unroll
        for (int j = 0; j < ST; ++j) {
          cum = cum + s[j];
          s[j] = cum;
        }
        if (!(ud >= cum)) {
#pragma unroll
          for (int j = 0; j < ST; ++j)
            while (d < d1 && ud < s[j]) {
              out[d++] = base + q + j;
              ud = d < d1 ? u[d] : 0.0;
            }
        }
      }
      done = (d >= d1);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0)
    while (d < d1) out[d++] = ~0ull;
}

// Partial sums of Re <psi|O|psi> = Re sum_o conj(psi_o) (O psi)_o in one pass, one per workgroup.
template <typename R>
__global__ __launch_bounds__(256) void k_pauli_expect(const typename CT<R>::T* __restrict__ psi, uint64_t dim,
                                                      const PauliGroup* __restrict__ groups, int ngroups,
                                                      const PauliZTerm* __restrict__ terms, double* __restrict__ part,
                                                      int accumulate) {
  __shared__ double red[256];
  double acc = 0.0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t o = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; o < dim; o += stride) {
    double yr = 0.0, yi = 0.0;
    for (int g = 0; g < ngroups; ++g) {
      const uint64_t j = o ^ groups[g].xm;
      double fr = 0.0, fi = 0.0;
      const uint32_t t0 = groups[g].first, t1 = t0 + groups[g].count;
      for (uint32_t t = t0; t < t1; ++t) {
        const bool neg = __popcll(j & terms[t].zm) & 1;
        fr += neg ? -terms[t].cr : terms[t].cr;
        fi += neg ? -terms[t].ci : terms[t].ci;
      }
      const double pr = (double)psi[j].x, pi = (double)psi[j].y;
      yr += fr * pr - fi * pi;
      yi += fr * pi + fi * pr;
    }
    acc += (double)psi[o].x * yr + (double)psi[o].y * yi;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = accumulate ? part[blockIdx.x] + red[0] : red[0];
}

// The pairs (r, r ^ M) of a thread's 16 amplitudes, r running over the 8 registers whose bit B
// (the top bit of M) is 0: conj(a_r) a_{r^M}, real and imaginary parts.
template <int B>
__device__ __forceinline__ constexpr int pair_rep(int i) {
  return ((i >> B) << (B + 1)) | (i & ((1 << B) - 1));
}
// The values as the compiler must take them here: nothing computed from them moves above.
template <typename T, int N>
__device__ __forceinline__ void pin(T (&a)[N]) {
#pragma unroll
  for (int r = 0; r < N; ++r) asm volatile("" : "+v"(a[r].x), "+v"(a[r].y));
}
// Re (or Im) of conj(x) y in binary64.
template <typename T>
__device__ __forceinline__ double pair_part(const T& x, const T& y, bool im) {
  return im ? fma((double)x.x, (double)y.y, -(double)x.y * (double)y.x)
            : fma((double)x.x, (double)y.x, (double)x.y * (double)y.y);
}
// sum over the pairs (r, r ^ M) of Re conj(a_r) a_{r^M}
template <typename T, int M>
__device__ __forceinline__ double pairs_sum(const T (&a)[16]) {
  constexpr int B = M >= 8 ? 3 : (M >= 4 ? 2 : (M >= 2 ? 1 : 0));
  double s0 = 0.0, s1 = 0.0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const T x = a[pair_rep<B>(i)], y = a[pair_rep<B>(i) ^ M];
    s0 = fma((double)x.x, (double)y.x, s0);
    s1 = fma((double)x.y, (double)y.y, s1);
  }
  return s0 + s1;
}
template <typename T, int M>
__device__ __forceinline__ void reg_pairs(const T (&a)[16], bool re, bool im, double (&qr)[8], double (&qi)[8]) {
  constexpr int B = M >= 8 ? 3 : (M >= 4 ? 2 : (M >= 2 ? 1 : 0));
  if (re) {
#pragma unroll
    for (int i = 0; i < 8; ++i) qr[i] = pair_part(a[pair_rep<B>(i)], a[pair_rep<B>(i) ^ M], false);
  }
  if (im) {
#pragma unroll
    for (int i = 0; i < 8; ++i) qi[i] = pair_part(a[pair_rep<B>(i)], a[pair_rep<B>(i) ^ M], true);
  }
}
// The same with the partners y (read from LDS) in the order of the representatives.
template <typename T, int B>
__device__ __forceinline__ void lds_pairs(const T (&a)[16], const T (&y)[8], bool re, bool im, double (&qr)[8],
                                          double (&qi)[8]) {
  if (re) {
#pragma unroll
    for (int i = 0; i < 8; ++i) qr[i] = pair_part(a[pair_rep<B>(i)], y[i], false);
  }
  if (im) {
#pragma unroll
    for (int i = 0; i < 8; ++i) qi[i] = pair_part(a[pair_rep<B>(i)], y[i], true);
  }
}

// In-place Walsh-Hadamard transform: w[p] becomes sum_i (-1)^{popcount(i & p)} w[i], the sum of
// the values under every sign pattern p at once.
// The results are opaque: the compiler would else move the last additions to each pattern's use, and
// hold (and spill) the values of every step until then.
template <int N>
__device__ __forceinline__ void walsh(double (&w)[N]) {
#pragma unroll
  for (int h = 1; h < N; h *= 2)
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (!(i & h)) {
        const double x = w[i], y = w[i | h];
        w[i] = x + y;
        w[i | h] = x - y;
      }
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(w[i]));
}
__device__ __forceinline__ double at_pattern(const double (&w)[8], uint32_t p) {
  double v;
  switch (p) {
    case 0: v = w[0]; break;
    case 1: v = w[1]; break;
    case 2: v = w[2]; break;
    case 3: v = w[3]; break;
    case 4: v = w[4]; break;
    case 5: v = w[5]; break;
    case 6: v = w[6]; break;
    default: v = w[7]; break;
  }
  return v;
}

// Records at uniform addresses, through scalar loads: the constant address space says that nothing
// writes them while the kernel runs. From plain pointers the compiler made vector loads (it takes a
// barrier for a possible write), and a wavefront waited for each record behind its tile's loads.
__device__ __forceinline__ PauliTileTerm load_term(const PauliTileTerm* p) {
  const auto q = (const __attribute__((address_space(4))) uint64_t*)p;
  return PauliTileTerm{q[0], __longlong_as_double((long long)q[1]), (uint32_t)q[2], (uint32_t)(q[2] >> 32)};
}
__device__ __forceinline__ PauliTileGroup load_group(const PauliTileGroup* p) {
  const auto q = (const __attribute__((address_space(4))) uint32_t*)p;
  return PauliTileGroup{q[0], q[1], q[2], q[3]};
}

// A term's coefficient with its sign (-1)^{parity}: the parity of the tile's bits is uniform, the
// thread's comes from its tile position pt.
__device__ __forceinline__ double signed_coeff(const PauliTileTerm& t, uint64_t base, uint32_t pt) {
  const uint32_t ones = (uint32_t)__popc(pt & t.lz) + (uint32_t)__popcll(base & t.zout);
  const uint32_t hi = (uint32_t)__double2hiint(t.c) + (ones << 31);  // an odd count flips the sign bit
  return __hiloint2double((int)hi, __double2loint(t.c));
}

// w[p] of the transform of q alone: its additions for that one pattern, in the same order.
__device__ __forceinline__ double fold_pattern(const double (&q)[8], uint32_t p) {
  double sg[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) sg[k] = __hiloint2double((int)(0x3ff00000u | ((p >> k) & 1u) << 31), 0);
  double w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = fma(sg[0], q[2 * i + 1], q[2 * i]);
  return fma(sg[2], fma(sg[1], w[3], w[2]), fma(sg[1], w[1], w[0]));
}

// sum of c (-1)^{parity} w[pattern] over `count` terms, w the transform of q, of which t is the first
// and tp points at the one behind it; on return both have moved past them (each term is fetched
// while the one before is added). With FOLD, up to three terms take fewer additions without the
// transform (7 each, not 24 in all) and no search for the pattern's value: 250 strings on 24 qubits,
// complex128, 1416 -> 1325 us. Not in complex64, whose registers then spill (60 strings on 24
// qubits 418 -> 488 us).
template <bool FOLD>
__device__ __forceinline__ double signed_terms(double (&q)[8], const PauliTileTerm* __restrict__& tp, uint32_t count,
                                               PauliTileTerm& t, uint64_t base, uint32_t pt) {
  double acc = 0.0;
  if (FOLD && count <= 3) {
    for (; count; --count) {
      const PauliTileTerm next = load_term(tp++);
      acc = fma(signed_coeff(t, base, pt), fold_pattern(q, t.pat), acc);
      t = next;
    }
    return acc;
  }
  walsh<8>(q);
  for (; count; --count) {
    const PauliTileTerm next = load_term(tp++);
    acc = fma(signed_coeff(t, base, pt), at_pattern(q, t.pat), acc);
    t = next;
  }
  return acc;
}

// The groups of an arrangement that are one real term without a sign on the register bits, their
// X masks the patterns set in `plain`: straight-line code (a dispatch on the pattern for each
// group spent more scalar instructions than the group's own arithmetic).
template <typename T, int M>
__device__ __forceinline__ void plain_groups(const T (&a)[16], uint32_t plain, const PauliTileTerm* __restrict__& tp,
                                             PauliTileTerm& t, uint64_t base, uint32_t pt, double& acc) {
  if ((plain >> M) & 1u) {
    const PauliTileTerm next = load_term(tp++);
    acc = fma(signed_coeff(t, base, pt), pairs_sum<T, M>(a), acc);
    t = next;
  }
  if constexpr (M < 15) plain_groups<T, M + 1>(a, plain, tp, t, base, pt, acc);
}

// LDS slot of a tile's element p (see k_pauli_expect_tiles).
template <int K>
__device__ __forceinline__ uint32_t pauli_slot(uint32_t p) {
  constexpr int LN = K - 12;
  return p ^ (((p >> (LN + 4)) & 15u) << LN);
}
// Tile position of a thread's register 0 in arrangement A.
template <int K, int A>
__device__ __forceinline__ uint32_t pauli_thread(uint32_t lane) {
  constexpr uint32_t nb = (uint32_t)pauli_arrangement_bit(K, A);
  return (lane & ((1u << nb) - 1u)) | ((lane >> nb) << (nb + 4));
}

// The LDS slot of a thread's register r in arrangement A. Slots are linear: the thread's part, at byte
// offset `first`, meets the register's constant one in the lowest nibble only, so an access takes at
// most one xor, and the rest is its immediate offset.
template <typename R, int K, int A>
__device__ __forceinline__ R& pauli_at(R* lds, uint32_t first, uint32_t r) {
  const uint32_t s = pauli_slot<K>(r << pauli_arrangement_bit(K, A)), low = s & (15u << (K - 12));
  return *reinterpret_cast<R*>(reinterpret_cast<char*>(lds) + ((first ^ (low * sizeof(R))) + (s - low) * sizeof(R)));
}

// A thread's 16 amplitudes from arrangement A - 1 to arrangement A, real parts and then imaginary
// parts through an LDS array of 2^K reals.
template <typename R, int K, int A, typename T>
__device__ __forceinline__ void rearrange(T (&a)[16], R* lds, uint32_t lane) {
  static_assert(K == 12, "arrangements of whole nibbles");
  // the thread's place, opaque: addresses are computed for each round, not kept in registers
  auto place = [&](auto arrangement) {
    uint32_t l = lane;
    asm volatile("" : "+v"(l));
    return pauli_slot<K>(pauli_thread<K, decltype(arrangement)::value>(l)) * (uint32_t)sizeof(R);
  };
  constexpr std::integral_constant<int, A - 1> from{};
  constexpr std::integral_constant<int, A> to{};
  __syncthreads();  // the reads before are over
  uint32_t p = place(from);
#pragma unroll
  for (uint32_t r = 0; r < 16; ++r) pauli_at<R, K, A - 1>(lds, p, r) = a[r].x;
  __syncthreads();
  p = place(to);
#pragma unroll
  for (uint32_t r = 0; r < 16; ++r) a[r].x = pauli_at<R, K, A>(lds, p, r);
  __syncthreads();
  p = place(from);
#pragma unroll
  for (uint32_t r = 0; r < 16; ++r) pauli_at<R, K, A - 1>(lds, p, r) = a[r].y;
  __syncthreads();
  p = place(to);
#pragma unroll
  for (uint32_t r = 0; r < 16; ++r) a[r].y = pauli_at<R, K, A>(lds, p, r);
}

// X mask 0 of a tile in arrangement 0: terms sorted by pattern, diag_count[p] of each.
template <typename T>
__device__ __forceinline__ void diag_group(const T (&a)[16], const uint32_t (&diag_count)[16],
                                           const PauliTileTerm* __restrict__& tp, PauliTileTerm& tm, uint64_t base,
                                           uint32_t pt, double& acc) {
  double w[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) w[r] = fma((double)a[r].x, (double)a[r].x, (double)a[r].y * (double)a[r].y);
  walsh<16>(w);
#pragma unroll
  for (int p = 0; p < 16; ++p) {
    uint32_t count = diag_count[p];
    if (count == 0) continue;
    double f = 0.0;
    for (; count; --count) {
      const PauliTileTerm tn = load_term(tp++);
      f += signed_coeff(tm, base, pt);
      tm = tn;
    }
    acc = fma(f, w[p], acc);
  }
}

// X mask 0 and the plain groups of arrangements A and up.
template <typename R, int K, int A, typename T>
__device__ __forceinline__ void plain_arrangements(T (&a)[16], R* lds, uint32_t lane, const PauliTilePass& ps,
                                                   const uint32_t (&diag_count)[16],
                                                   const PauliTileTerm* __restrict__& tp, PauliTileTerm& tm,
                                                   uint64_t base, double& acc) {
  if ((ps.arrs >> A) == 0) return;
  if constexpr (A > 0) rearrange<R, K, A>(a, lds, lane);
  const uint32_t pt = pauli_thread<K, A>(lane);
  if constexpr (A == 0) {
    if (ps.diag) diag_group(a, diag_count, tp, tm, base, pt, acc);
  }
  if (ps.plain[A]) plain_groups<T, 1>(a, ps.plain[A], tp, tm, base, pt, acc);
  if constexpr (pauli_arrangement_bit(K, A) > 0)  // the last one holds the lowest bits
    plain_arrangements<R, K, A + 1>(a, lds, lane, ps, diag_count, tp, tm, base, acc);
}

// Partial sums of Re <psi|O|psi> for groups whose X masks lie in tiles of 2^K amplitudes (tile
// bits = the set bits of a pass's tmask, the lowest first), all passes in one launch. Workgroups
// of 2^(K-4) threads walk the tiles; a thread holds 16 amplitudes, which differ in 4 tile bits.
// What bounds it: HBM when a pass holds few groups, else vector issue, then LDS (a 16-byte read
// per amplitude costs a quarter of the CU's 128 B/clk for 8 clocks). So:
//  * the tile is held in up to three arrangements (four for 2^13 tiles), each with another 4 of its bits in
//    registers: a group whose X mask lies in one of them pairs registers, with no LDS access;
//    only masks that cross them read partners from LDS;
//  * a hermitian term gives the same for (o, o ^ xm) and (o ^ xm, o): one product for each pair;
//  * signs: a Walsh-Hadamard transform of the 8 pair products (16 probabilities for X mask 0)
//    holds the sum under every pattern of register bits, so a term takes one multiply-add for
//    all of a thread's amplitudes instead of one add for each.
//  * without general groups (Ising and the like), the exchange between arrangements moves real
//    parts and then imaginary parts through half the LDS, and complex128 fits four workgroups on a
//    CU in place of two: one's loads run under the others' arithmetic. Complex64 is held to two by
//    its registers (111 at 512 threads), and keeps the exchange of whole amplitudes.
// What it measured against one LDS read and a signed add per amplitude, group and term: the Ising
// observable of 29 qubits, complex128 (57 terms, 29 X masks, 3 passes), 13.5 -> 4.1 ms = 6.3 TB/s
// (5.6 ms with vector loads of the records and two workgroups per CU); a pass of Z terms alone 6.9
// TB/s, one of twelve contiguous X masks 6.1, one of nine X masks 2^12 and up in 128-byte segments
// 5.0. Complex64, 28 qubits, 6.5 -> 1.6 ms (2.1 with vector loads); 120 strings of up to 4 factors on 22 qubits
// 520 -> 335 us (355). Fetching the next tile ahead took longer (5.9 ms: its registers spill).
// Element p of the tile sits at LDS slot p ^ (bits above the lowest arrangement's nibble, at its
// place): consecutive lanes hit distinct slots in every arrangement.
template <typename R, int K, bool NT, bool GENERAL>
__global__ __launch_bounds__(1 << (K - 4), K == 12 && GENERAL ? 2 : 4) void k_pauli_expect_tiles(
    const typename CT<R>::T* __restrict__ psi, uint64_t dim, PauliTilePasses P,
    const PauliTileGroup* __restrict__ groups, const PauliTileTerm* __restrict__ terms, double* __restrict__ part,
    int accumulate) {
  using T = typename CT<R>::T;
  constexpr int TB = K - 4;  // thread bits
  constexpr bool HALF = !GENERAL && K == 12;
  __shared__ __align__(16) R lds_reals[(HALF ? 1 : 2) << K];
  T* const lds = reinterpret_cast<T*>(lds_reals);
  const uint32_t tid = threadIdx.x;
  const uint32_t ntiles = (uint32_t)(dim >> K);  // 2^28 at most
  auto slot = [](uint32_t p) { return pauli_slot<K>(p); };
  double acc = 0.0;
  uint32_t t = blockIdx.x;  // this workgroup's next (pass, tile), counted through all passes
  for (uint32_t ip = 0; ip < P.count; ++ip) {
    const PauliTilePass& ps = P.p[ip];
    const uint64_t tmask = ps.tmask, nontile = (dim - 1) & ~tmask;
    uint64_t toff = 0, hib[4];
    {
      uint64_t m = tmask;
#pragma unroll
      for (int b = 0; b < K; ++b) {
        const uint64_t low = m & (0ull - m);
        m ^= low;
        if (b < TB) {
          if ((tid >> b) & 1u) toff |= low;
        } else {
          hib[b - TB] = low;
        }
      }
    }
    // tile t's base has t's bits on the bits outside the tile; a step adds the deposited stride
    // with the tile's bits set, so that carries run through them
    const uint64_t step = deposit_bits(gridDim.x, nontile);
    uint64_t base = deposit_bits(t, nontile);
    for (; t < ntiles; t += gridDim.x, base = ((base | tmask) + step) & nontile) {
      uint32_t lane = tid;  // opaque: LDS addresses are recomputed for each tile, not kept
      asm volatile("" : "+v"(lane));
      T a[16];
      {
        const T* src = psi + (base | toff);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          uint64_t off = 0;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if ((r >> q) & 1) off |= hib[q];
          if (NT) {
            load_nt(a[r], src + off);
          } else {
            a[r].x = src[off].x;
            a[r].y = src[off].y;
          }
        }
      }
      // records and terms in the order of their use, each fetched one ahead
      const PauliTileGroup* __restrict__ gp = groups + ps.first;
      const PauliTileTerm* __restrict__ tp = terms + ps.term0;
      PauliTileGroup gr = load_group(gp++);
      PauliTileTerm tm = load_term(tp++);
      if constexpr (HALF) {
        plain_arrangements<R, K, 0>(a, lds_reals, lane, ps, P.diag_count, tp, tm, base, acc);
        continue;
      }
      if (ps.lds) {
        __syncthreads();  // the previous tile's reads are over
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          T& d = lds[slot(lane | ((uint32_t)r << TB))];
          d.x = a[r].x;
          d.y = a[r].y;
        }
        __syncthreads();
      }
#pragma unroll 1
      for (int arr = 0; arr < kPauliArrangements; ++arr) {
        if (!((ps.arrs >> arr) & 1u)) continue;
        const uint32_t nb = (uint32_t)pauli_arrangement_bit(K, arr);  // the register bits' place in the tile
        const uint32_t pt = (lane & ((1u << nb) - 1u)) | ((lane >> nb) << (nb + 4));
        if (arr > 0) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const T& d = lds[slot(pt | ((uint32_t)r << nb))];
            a[r].x = d.x;
            a[r].y = d.y;
          }
        }
        if (arr == 0 && ps.diag) diag_group(a, P.diag_count, tp, tm, base, pt, acc);
        if (ps.plain[arr]) plain_groups<T, 1>(a, ps.plain[arr], tp, tm, base, pt, acc);
#pragma unroll 1
        for (uint32_t left = GENERAL ? ps.cnt[arr] : 0; left; --left) {
          const PauliTileGroup next = load_group(gp++);
          const uint32_t op = gr.op, nre = gr.nre, nim = gr.nim, lx = gr.lx;
          gr = next;
          // products of the loop-invariant amplitudes must not move out of the group loop: the
          // compiler would keep every mask's pairs in registers at once, and spill them
          pin(a);
          const bool re = nre != 0, im = nim != 0;
          double qr[8] = {}, qi[8] = {};
          T y[8];
          if (op >= PAULI_LDS) {
            const uint32_t b = op & 3u;  // the register bit that tells a pair's two ends apart
            const uint32_t first = slot(pt ^ lx);  // slots are linear: the register's part is uniform
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) {
              const uint32_t r = ((i >> b) << (b + 1)) | (i & ((1u << b) - 1u));
              const T& d = lds[first ^ slot(r << nb)];
              y[i].x = d.x;
              y[i].y = d.y;
            }
          }
          switch (op) {
            case 1: reg_pairs<T, 1>(a, re, im, qr, qi); break;
            case 2: reg_pairs<T, 2>(a, re, im, qr, qi); break;
            case 3: reg_pairs<T, 3>(a, re, im, qr, qi); break;
            case 4: reg_pairs<T, 4>(a, re, im, qr, qi); break;
            case 5: reg_pairs<T, 5>(a, re, im, qr, qi); break;
            case 6: reg_pairs<T, 6>(a, re, im, qr, qi); break;
            case 7: reg_pairs<T, 7>(a, re, im, qr, qi); break;
            case 8: reg_pairs<T, 8>(a, re, im, qr, qi); break;
            case 9: reg_pairs<T, 9>(a, re, im, qr, qi); break;
            case 10: reg_pairs<T, 10>(a, re, im, qr, qi); break;
            case 11: reg_pairs<T, 11>(a, re, im, qr, qi); break;
            case 12: reg_pairs<T, 12>(a, re, im, qr, qi); break;
            case 13: reg_pairs<T, 13>(a, re, im, qr, qi); break;
            case 14: reg_pairs<T, 14>(a, re, im, qr, qi); break;
            case 15: reg_pairs<T, 15>(a, re, im, qr, qi); break;
            case PAULI_LDS + 0: lds_pairs<T, 0>(a, y, re, im, qr, qi); break;
            case PAULI_LDS + 1: lds_pairs<T, 1>(a, y, re, im, qr, qi); break;
            case PAULI_LDS + 2: lds_pairs<T, 2>(a, y, re, im, qr, qi); break;
            default: lds_pairs<T, 3>(a, y, re, im, qr, qi); break;
          }
          if (re) {
            acc += signed_terms<K == 12>(qr, tp, nre, tm, base, pt);
          }
          if (im) {
            acc += signed_terms<K == 12>(qi, tp, nim, tm, base, pt);
          }
        }
      }
    }
    t -= ntiles;
  }
  __syncthreads();
  double* red = reinterpret_cast<double*>(lds_reals);
  red[tid] = acc;
  __syncthreads();
  for (uint32_t w = 1u << (TB - 1); w > 0; w >>= 1) {
    if (tid < w) red[tid] += red[tid + w];
    __syncthreads();
  }
  if (tid == 0) part[blockIdx.x] = accumulate ? part[blockIdx.x] + red[0] : red[0];
}

// The streaming ceiling of a sweep: every amplitude read, multiplied by a real factor and
// written back in place, one amplitude per thread in index order (the fastest in-place shape
// measured on MI355X).
template <typename R>
__global__ __launch_bounds__(256) void k_stream_scale(typename CT<R>::T* __restrict__ psi, uint64_t dim, R f) {
  // non-temporal, as the tile sweeps of large states access memory
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < dim) {
    typename CT<R>::T v;
    load_nt(v, &psi[i]);
    v.x *= f;
    v.y *= f;
    store_nt(&psi[i], v);
  }
}

__global__ void k_stamp(uint64_t* out) {
  if (threadIdx.x == 0 && blockIdx.x == 0) out[0] = wall_clock64();
}

__device__ __forceinline__ double row_sum(const double* __restrict__ row, uint64_t ncols) {
  __shared__ double red[256];
  double acc = 0.0;
  for (uint64_t j = threadIdx.x; j < ncols; j += 256) acc += row[j];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  return red[0];
}

// Row sums of a partial-sum table in a fixed order (one workgroup per row): each thread adds
// a strided subset, then a tree over the workgroup.
__global__ __launch_bounds__(256) void k_sum_rows(const double* __restrict__ part, uint64_t ncols,
                                                  double* __restrict__ out) {
  const double s = row_sum(part + (uint64_t)blockIdx.x * ncols, ncols);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// The end of a batch instance in one launch: workgroups 0 .. gridDim.x - 2 sum its gradient rows, the
// last its expectation partials, and the instance's time stamp is when the last of them is done
// (the clock only rises, so the maximum needs no reset between runs).
__global__ __launch_bounds__(256) void k_finish_instance(const double* __restrict__ part, uint64_t ncols,
                                                         double* __restrict__ grads, const double* __restrict__ dot,
                                                         uint64_t ndot, double* __restrict__ energy,
                                                         unsigned long long* __restrict__ stamp) {
  const bool last = blockIdx.x == gridDim.x - 1;
  const double s = last ? row_sum(dot, ndot) : row_sum(part + (uint64_t)blockIdx.x * ncols, ncols);
  if (threadIdx.x != 0) return;
  if (last) energy[0] = s;
  else grads[blockIdx.x] = s;
  atomicMax(stamp, (unsigned long long)wall_clock64());
}

// complex64 <-> binary64 conversion for state upload/download
__global__ void k_f64_to_c64(float2* __restrict__ dst, const double2* __restrict__ src, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    dst[i] = make_float2((float)src[i].x, (float)src[i].y);
}
__global__ void k_c64_to_f64(double2* __restrict__ dst, const float2* __restrict__ src, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    dst[i] = make_double2((double)src[i].x, (double)src[i].y);
}

}  // namespace dev

// =====================================================================================
// Host launchers
// =====================================================================================

namespace {
inline unsigned grid_for(uint64_t work, int block, unsigned cap = 1u << 20) {
  uint64_t g = (work + block - 1) / block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (unsigned)g;
}
}  // namespace

int tile_max_bits(int prec) { return 13; }
int tile_reg_bits(int K) { return K < 4 ? K : 4; }

// States of at least 512 MB (twice the memory-side cache) are streamed with non-temporal
// accesses: no later pass finds them in a cache anyway.
inline int streamed(int prec, uint64_t dim) { return dim * (prec == 0 ? 16u : 8u) >= (512ull << 20) ? 1 : 0; }

hipError_t launch_init_basis(int prec, void* psi, uint64_t dim, uint64_t one_at, hipStream_t s) {
  const unsigned g = grid_for(dim, 256, 1u << 16);
  const int nt = streamed(prec, dim);
  if (prec == 0)
    dev::k_init_basis<double><<<g, 256, 0, s>>>((double2*)psi, dim, one_at, nt);
  else
    dev::k_init_basis<float><<<g, 256, 0, s>>>((float2*)psi, dim, one_at, nt);
  return hipGetLastError();
}

hipError_t launch_exact(int prec, void* psi, uint64_t ngroups, const ExactArgs& a, const double2* M,
                        hipStream_t s) {
  const unsigned g = grid_for(ngroups, 256, 1u << 16);
#define QR_EXACT_CASE(KR)                                                                   \
  case KR:                                                                                  \
    if (prec == 0)                                                                          \
      dev::k_exact<double, KR><<<g, 256, 0, s>>>((double2*)psi, ngroups, a, M);             \
    else                                                                                    \
      dev::k_exact<float, KR><<<g, 256, 0, s>>>((float2*)psi, ngroups, a, M);               \
    break;
  switch (a.K) {
    QR_EXACT_CASE(1)
    QR_EXACT_CASE(2)
    QR_EXACT_CASE(3)
    QR_EXACT_CASE(4)
    default:
      return hipErrorInvalidValue;
  }
#undef QR_EXACT_CASE
  return hipGetLastError();
}

hipError_t launch_exact_wide(int prec, void* psi, void* tmp, uint64_t tmp_groups, uint64_t ngroups,
                             const ExactWideArgs& a, const double2* M, const uint64_t* off,
                             const uint32_t* order, const uint8_t* flags, hipStream_t s) {
  // one thread per tmp slot: grid * block == tmp_groups
  const int block = tmp_groups >= 256 ? 256 : (int)tmp_groups;
  const unsigned g = (unsigned)(tmp_groups / block);
  if (prec == 0)
    dev::k_exact_wide<double><<<g, block, 0, s>>>((double2*)psi, (double2*)tmp, ngroups, a, M, off, order, flags);
  else
    dev::k_exact_wide<float><<<g, block, 0, s>>>((float2*)psi, (float2*)tmp, ngroups, a, M, off, order, flags);
  return hipGetLastError();
}

hipError_t launch_dense1(int prec, void* psi, uint64_t npairs, int t, uint64_t cmask, const double2* u,
                         hipStream_t s) {
  const unsigned g = grid_for(npairs, 256, 1u << 18);
  if (prec == 0)
    dev::k_dense1<double><<<g, 256, 0, s>>>((double2*)psi, npairs, t, cmask, u[0], u[1], u[2], u[3]);
  else
    dev::k_dense1<float><<<g, 256, 0, s>>>((float2*)psi, npairs, t, cmask, u[0], u[1], u[2], u[3]);
  return hipGetLastError();
}

hipError_t launch_diag1(int prec, void* psi, uint64_t dim, int t, uint64_t cmask, double2 d0, double2 d1,
                        hipStream_t s) {
  const unsigned g = grid_for(dim, 256, 1u << 18);
  if (prec == 0)
    dev::k_diag1<double><<<g, 256, 0, s>>>((double2*)psi, dim, t, cmask, d0, d1);
  else
    dev::k_diag1<float><<<g, 256, 0, s>>>((float2*)psi, dim, t, cmask, d0, d1);
  return hipGetLastError();
}

hipError_t launch_densek_reg(int prec, void* psi, uint64_t ngroups, const DenseKArgs& a, const double2* M,
                             const uint64_t* off, hipStream_t s, const Instances& in) {
  if (in.count == 0 || in.count > 65535u) return hipErrorInvalidValue;
  const dim3 g(grid_for(ngroups, 256, 1u << 18), in.count);
#define QR_DENSEK_CASE(KK)                                                                     \
  case KK:                                                                                     \
    if (prec == 0)                                                                             \
      dev::k_densek_reg<double, KK><<<g, 256, 0, s>>>((double2*)psi, ngroups, a, M, off, in);  \
    else                                                                                       \
      dev::k_densek_reg<float, KK><<<g, 256, 0, s>>>((float2*)psi, ngroups, a, M, off, in);    \
    break;
  switch (a.k) {
    QR_DENSEK_CASE(2)
    QR_DENSEK_CASE(3)
    QR_DENSEK_CASE(4)
    default:
      return hipErrorInvalidValue;
  }
#undef QR_DENSEK_CASE
  return hipGetLastError();
}

hipError_t launch_densek(int prec, void* psi, void* tmp, uint64_t tmp_groups, uint64_t ngroups,
                         const DenseKArgs& a, const double2* M, const uint64_t* off, hipStream_t s) {
  const int block = tmp_groups >= 256 ? 256 : (int)tmp_groups;
  const unsigned g = (unsigned)(tmp_groups / block);
  if (prec == 0)
    dev::k_densek<double><<<g, block, 0, s>>>((double2*)psi, (double2*)tmp, ngroups, a, M, off);
  else
    dev::k_densek<float><<<g, block, 0, s>>>((float2*)psi, (float2*)tmp, ngroups, a, M, off);
  return hipGetLastError();
}

hipError_t launch_diagk(int prec, void* psi, uint64_t dim, const DiagKArgs& a, const double2* D,
                        hipStream_t s, const Instances& in) {
  if (in.count == 0 || in.count > 65535u) return hipErrorInvalidValue;
  const dim3 g(grid_for(dim, 256, 1u << 18), in.count);
  if (prec == 0)
    dev::k_diagk<double><<<g, 256, 0, s>>>((double2*)psi, dim, a, D, in);
  else
    dev::k_diagk<float><<<g, 256, 0, s>>>((float2*)psi, dim, a, D, in);
  return hipGetLastError();
}


hipError_t launch_sample_fold(int prec, const void* psi, uint64_t dim, const double* u, uint64_t shots,
                              uint64_t* out, hipStream_t s) {
  if (prec == 0)
    dev::k_sample_fold<double><<<1, 1024, 0, s>>>((const double2*)psi, dim, u, shots, out);
  else
    dev::k_sample_fold<float><<<1, 1024, 0, s>>>((const float2*)psi, dim, u, shots, out);
  return hipGetLastError();
}

hipError_t launch_block_mass(int prec, const void* psi, uint64_t dim, int bb, double* mass, hipStream_t s) {
  const uint64_t nb = (dim + (1ull << bb) - 1) >> bb;
  const int nt = streamed(prec, dim);
  if (prec == 0)
    dev::k_block_mass<double><<<(unsigned)nb, 256, 0, s>>>((const double2*)psi, dim, bb, mass, nt);
  else
    dev::k_block_mass<float><<<(unsigned)nb, 256, 0, s>>>((const float2*)psi, dim, bb, mass, nt);
  return hipGetLastError();
}

hipError_t launch_block_exact_sums(int prec, const void* psi, uint64_t dim, int bb, const int32_t* ebase,
                                   double* sums, uint32_t* flags, const TieBlocks& tie, hipStream_t s) {
  const uint64_t nb = (dim + (1ull << bb) - 1) >> bb;
  const int nt = streamed(prec, dim);
  if (prec == 0)
    dev::k_block_exact_sums<double>
        <<<(unsigned)nb, 256, 0, s>>>((const double2*)psi, dim, bb, ebase, sums, flags, nt, tie);
  else
    dev::k_block_exact_sums<float>
        <<<(unsigned)nb, 256, 0, s>>>((const float2*)psi, dim, bb, ebase, sums, flags, nt, tie);
  return hipGetLastError();
}

hipError_t launch_gather_probs(int prec, const void* psi, int bb, const uint64_t* list, uint32_t count, double* out,
                               hipStream_t s) {
  if (count == 0) return hipSuccess;
  if (count > 65535u) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((1u << bb) > 1024u ? (1u << bb) / 1024u : 1u), count);
  if (prec == 0)
    dev::k_gather_probs<double><<<grid, 256, 0, s>>>((const double2*)psi, bb, list, out);
  else
    dev::k_gather_probs<float><<<grid, 256, 0, s>>>((const float2*)psi, bb, list, out);
  return hipGetLastError();
}

hipError_t launch_sample_exact_blocks(int prec, const void* psi, uint64_t dim, int bb, const ExactJob* jobs,
                                      uint64_t njobs, const double* u, uint64_t* out, hipStream_t s) {
  if (njobs == 0) return hipSuccess;
  if (bb < 12) return hipErrorInvalidValue;  // blocks are whole 4096-amplitude chunks
  if (prec == 0)
    dev::k_sample_exact_blocks<double><<<(unsigned)njobs, 256, 0, s>>>((const double2*)psi, dim, bb, jobs, u, out);
  else
    dev::k_sample_exact_blocks<float><<<(unsigned)njobs, 256, 0, s>>>((const float2*)psi, dim, bb, jobs, u, out);
  return hipGetLastError();
}

hipError_t launch_norm_partial(int prec, const void* psi, uint64_t dim, double* part, int nblocks,
                               hipStream_t s) {
  if (prec == 0)
    dev::k_norm_partial<double><<<nblocks, 256, 0, s>>>((const double2*)psi, dim, part);
  else
    dev::k_norm_partial<float><<<nblocks, 256, 0, s>>>((const float2*)psi, dim, part);
  return hipGetLastError();
}

hipError_t launch_gen_partial(int prec, const void* lam, const void* psi, uint64_t dim, int t, int gen,
                              double2* part, int nblocks, hipStream_t s) {
  if (prec == 0)
    dev::k_gen_partial<double><<<nblocks, 256, 0, s>>>((const double2*)lam, (const double2*)psi, dim, t, gen, part);
  else
    dev::k_gen_partial<float><<<nblocks, 256, 0, s>>>((const float2*)lam, (const float2*)psi, dim, t, gen, part);
  return hipGetLastError();
}

hipError_t launch_pauli_sum(int prec, void* lam, const void* psi, uint64_t dim, const PauliGroup* groups, int ngroups,
                            int nplain, const PauliZTerm* terms, hipStream_t s, double* part) {
  const unsigned g = part ? pauli_sum_partials(dim) : grid_for(dim, 256, 1u << 18);
  if (prec == 0)
    dev::k_pauli_sum<double><<<g, 256, 0, s>>>((double2*)lam, (const double2*)psi, dim, groups, ngroups, nplain, terms, part);
  else
    dev::k_pauli_sum<float><<<g, 256, 0, s>>>((float2*)lam, (const float2*)psi, dim, groups, ngroups, nplain, terms, part);
  return hipGetLastError();
}

unsigned pauli_sum_partials(uint64_t dim) { return grid_for(dim, 256, 1024); }

hipError_t launch_init_batch(int prec, void* pool, const uint64_t* base, const uint32_t* bits, uint32_t count,
                             hipStream_t s) {
  if (count == 0) return hipSuccess;
  if (count > 65535u) return hipErrorInvalidValue;
  const dim3 g(64, count);
  if (prec == 0)
    dev::k_init_batch<double><<<g, 256, 0, s>>>((uint8_t*)pool, base, bits);
  else
    dev::k_init_batch<float><<<g, 256, 0, s>>>((uint8_t*)pool, base, bits);
  return hipGetLastError();
}

hipError_t launch_finish_instance(const double* part, uint64_t ncols, uint32_t nrows, double* grads, const double* dot,
                                  uint64_t ndot, double* energy, uint64_t* stamp, hipStream_t s) {
  dev::k_finish_instance<<<nrows + 1, 256, 0, s>>>(part, ncols, grads, dot, ndot, energy, (unsigned long long*)stamp);
  return hipGetLastError();
}

hipError_t launch_pauli_expect(int prec, const void* psi, uint64_t dim, const PauliGroup* groups, int ngroups,
                               const PauliZTerm* terms, double* part, int nblocks, hipStream_t s, int accumulate) {
  if (prec == 0)
    dev::k_pauli_expect<double>
        <<<nblocks, 256, 0, s>>>((const double2*)psi, dim, groups, ngroups, terms, part, accumulate);
  else
    dev::k_pauli_expect<float>
        <<<nblocks, 256, 0, s>>>((const float2*)psi, dim, groups, ngroups, terms, part, accumulate);
  return hipGetLastError();
}

hipError_t launch_init_instances(int prec, void* psi, uint64_t dim, uint64_t count, hipStream_t s) {
  const uint64_t total = dim * count;
  if (prec == 0)
    dev::k_init_instances<double><<<grid_for(total, 256, 1u << 16), 256, 0, s>>>((double2*)psi, dim, total);
  else
    dev::k_init_instances<float><<<grid_for(total, 256, 1u << 16), 256, 0, s>>>((float2*)psi, dim, total);
  return hipGetLastError();
}

hipError_t launch_sample_fold_instances(int prec, const void* psi, uint64_t dim, uint64_t count, const double* u,
                                        const uint64_t* off, uint64_t* out, hipStream_t s) {
  if (count == 0) return hipSuccess;
  if (count > 0x7fffffffull) return hipErrorInvalidValue;
  if (prec == 0)
    dev::k_sample_fold_instances<double><<<(unsigned)count, 256, 0, s>>>((const double2*)psi, dim, dim, u, off, out);
  else
    dev::k_sample_fold_instances<float><<<(unsigned)count, 256, 0, s>>>((const float2*)psi, dim, dim, u, off, out);
  return hipGetLastError();
}

int pauli_expect_partials(uint64_t dim) { return (int)std::min<uint64_t>(1024, std::max<uint64_t>(1, dim / 256)); }

hipError_t launch_pauli_expect_passes(int prec, const void* psi, uint64_t dim, const void* groups, const void* terms,
                                      const PauliTilePass* passes, int npasses, const uint32_t* diag_count,
                                      double* part, hipStream_t s) {
  const int nb = pauli_expect_partials(dim), K = pauli_tile_bits(prec), nt = streamed(prec, dim);
  int acc = 0;
  for (int i = 0; i < npasses;) {
    if (passes[i].tmask == 0) {
      const PauliTilePass& ps = passes[i++];
      const hipError_t e = launch_pauli_expect(prec, psi, dim, (const PauliGroup*)groups + ps.first, (int)ps.cnt[0],
                                               (const PauliZTerm*)terms, part, nb, s, acc);
      if (e != hipSuccess) return e;
      acc = 1;
      continue;
    }
    PauliTilePasses P{};
    for (int p = 0; p < 16; ++p) P.diag_count[p] = diag_count[p];
    for (; i < npasses && passes[i].tmask != 0 && P.count < kPauliPassesPerLaunch; ++i) {
      if (__builtin_popcountll(passes[i].tmask) != K || (dim >> K) == 0) return hipErrorInvalidValue;
      P.p[P.count++] = passes[i];
    }
    const PauliTileGroup* tg = (const PauliTileGroup*)groups;
    const PauliTileTerm* tt = (const PauliTileTerm*)terms;
    // observables without general groups (Ising and the like) run a variant without their code,
    // whose registers cost the others their occupancy
    bool general = false;
    for (uint32_t p = 0; p < P.count; ++p)
      for (int a = 0; a < kPauliArrangements; ++a) general = general || P.p[p].cnt[a] != 0;
    auto run = [&](auto kernel, auto* amp, unsigned threads) { kernel<<<nb, threads, 0, s>>>(amp, dim, P, tg, tt, part, acc); };
    if (prec == 0) {
      const double2* amp = (const double2*)psi;
      if (nt) general ? run(dev::k_pauli_expect_tiles<double, 12, true, true>, amp, 256)
                      : run(dev::k_pauli_expect_tiles<double, 12, true, false>, amp, 256);
      else general ? run(dev::k_pauli_expect_tiles<double, 12, false, true>, amp, 256)
                   : run(dev::k_pauli_expect_tiles<double, 12, false, false>, amp, 256);
    } else {
      const float2* amp = (const float2*)psi;
      if (nt) general ? run(dev::k_pauli_expect_tiles<float, 13, true, true>, amp, 512)
                      : run(dev::k_pauli_expect_tiles<float, 13, true, false>, amp, 512);
      else general ? run(dev::k_pauli_expect_tiles<float, 13, false, true>, amp, 512)
                   : run(dev::k_pauli_expect_tiles<float, 13, false, false>, amp, 512);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    acc = 1;
  }
  return hipSuccess;
}

hipError_t launch_stream_scale(int prec, void* psi, uint64_t dim, double f, hipStream_t s) {
  const uint64_t g = (dim + 255) / 256;
  if (g > 0x7fffffffull) return hipErrorInvalidValue;
  if (prec == 0)
    dev::k_stream_scale<double><<<(unsigned)g, 256, 0, s>>>((double2*)psi, dim, f);
  else
    dev::k_stream_scale<float><<<(unsigned)g, 256, 0, s>>>((float2*)psi, dim, (float)f);
  return hipGetLastError();
}

hipError_t launch_stamp(uint64_t* out, hipStream_t s) {
  dev::k_stamp<<<1, 64, 0, s>>>(out);
  return hipGetLastError();
}

hipError_t launch_sum_rows(const double* part, uint64_t ncols, uint32_t nrows, double* out, hipStream_t s) {
  if (nrows == 0) return hipSuccess;
  dev::k_sum_rows<<<nrows, 256, 0, s>>>(part, ncols, out);
  return hipGetLastError();
}

hipError_t launch_f64_to_c64(float2* dst, const double2* src, uint64_t n, hipStream_t s) {
  dev::k_f64_to_c64<<<grid_for(n, 256, 1u << 16), 256, 0, s>>>(dst, src, n);
  return hipGetLastError();
}

hipError_t launch_c64_to_f64(double2* dst, const float2* src, uint64_t n, hipStream_t s) {
  dev::k_c64_to_f64<<<grid_for(n, 256, 1u << 16), 256, 0, s>>>(dst, src, n);
  return hipGetLastError();
}

}  // namespace qr

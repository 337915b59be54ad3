// kernels.hpp — argument blocks and host launchers of the gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace qr {

// Exact per-gate sweep (K <= 4 acting wires, amplitudes held in registers).
struct ExactArgs {
  int K;
  uint8_t sorted_bits[8];  // acting bits ascending
  uint64_t off[16];        // offset of local basis state j (MSB-first local index)
  uint8_t order[16];       // local states in ascending global offset order
  uint32_t some;           // bit j: input j contributes
  uint32_t keep;           // bit r: output r keeps its input (custom None)
};

struct ExactWideArgs {
  int K;
  uint8_t sorted_bits[20];
};

struct DenseKArgs {
  int k;
  uint8_t sorted_bits[20];
  uint64_t cmask;
};

// Several states of one shape in a launch: instance y's state is y * state_stride amplitudes and its
// table y * table_stride double2 behind the first one's (at most 65535).
struct Instances {
  uint32_t count = 1;
  uint64_t state_stride = 0, table_stride = 0;
};

struct DiagKArgs {
  int k;
  uint8_t bits[20];  // local MSB first
  uint64_t cmask;
};

// Tile op codes (device interpreter).
enum TileCode : uint32_t {
  TC_END = 0,
  TC_REMAP = 1,      // a = index of the new slot map (data moves through LDS)
  TC_U1 = 2,         // a = register slot, coef -> 4 complex, b = form
  TC_D1 = 3,         // a = global bit, b = register slot or 0xFF, coef -> 2 complex, c = only |1>
  TC_SWAPSLOTS = 4,  // a = index of the new slot map (relabel, no data movement)
  TC_GRAD = 5,       // compiled dual-state stages only: gradient partial of one parameter
  TC_SCALE = 6,      // every amplitude times coef 0 (the stage's folded scalars)
};

// One interpreted op of a tile program (32 bytes, read with scalar loads).
struct TileOpDev {
  uint32_t w0;          // code | a << 8 | b << 16 | flags << 24
  uint32_t ns;          // register slots that must be 1
  uint64_t lane_cmask;  // control bits on thread slots / outside the tile
  uint32_t map;         // REMAP / SWAPSLOTS: new map index
  uint32_t swz;         // REMAP: swizzle table index
  uint32_t pad[2];
};
static_assert(sizeof(TileOpDev) == 32, "TileOpDev layout");

struct TileArgs {
  const TileOpDev* ops;
  const double2* coefs;   // 4 per op, op o at coefs[4 o]
  const uint32_t* maps;   // per map, K words: global bit | tile position << 8
  const uint32_t* swz;    // per remap, 2K words: LDS pattern of each slot, old map then new map
  uint64_t ntiles;
  uint64_t nontile_mask;  // index bits outside the tile; tile number bits are deposited there
  uint32_t nops;
  uint32_t pad;
};

// A block of the exact block-parallel sampler whose fold stays in one binade: its draws are
// u[first .. last), its fold starts at m_start units of `unit` = 2^(e-52), scale = 1 / unit.
struct ExactJob {
  uint64_t block;
  double m_start;
  double unit, scale;
  uint64_t first, last;
};

// Tile kernel variants available: tile bits K and register bits RB per precision.
int tile_max_bits(int prec);  // widest tile variant compiled (13)
int tile_reg_bits(int K);

// ---- launchers (prec: 0 = complex128, 1 = complex64) ----
hipError_t launch_init_basis(int prec, void* psi, uint64_t dim, uint64_t one_at, hipStream_t s);
hipError_t launch_exact(int prec, void* psi, uint64_t ngroups, const ExactArgs& a, const double2* M,
                        hipStream_t s);
hipError_t launch_exact_wide(int prec, void* psi, void* tmp, uint64_t tmp_groups, uint64_t ngroups,
                             const ExactWideArgs& a, const double2* M, const uint64_t* off,
                             const uint32_t* order, const uint8_t* flags, hipStream_t s);
hipError_t launch_dense1(int prec, void* psi, uint64_t npairs, int t, uint64_t cmask, const double2* u,
                         hipStream_t s);
hipError_t launch_diag1(int prec, void* psi, uint64_t dim, int t, uint64_t cmask, double2 d0, double2 d1,
                        hipStream_t s);
hipError_t launch_densek(int prec, void* psi, void* tmp, uint64_t tmp_groups, uint64_t ngroups,
                         const DenseKArgs& a, const double2* M, const uint64_t* off, hipStream_t s);
// Dense 2^k x 2^k, 2 <= k <= 4, each group of amplitudes in registers (no staging).
hipError_t launch_densek_reg(int prec, void* psi, uint64_t ngroups, const DenseKArgs& a, const double2* M,
                             const uint64_t* off, hipStream_t s, const Instances& in = Instances());
hipError_t launch_diagk(int prec, void* psi, uint64_t dim, const DiagKArgs& a, const double2* D,
                        hipStream_t s, const Instances& in = Instances());
hipError_t launch_tile(int prec, int K, int RB, bool prefetch, void* psi, const TileArgs& a, hipStream_t s);
hipError_t launch_sample_fold(int prec, const void* psi, uint64_t dim, const double* u, uint64_t shots,
                              uint64_t* out, hipStream_t s);
hipError_t launch_block_mass(int prec, const void* psi, uint64_t dim, int bb, double* mass, hipStream_t s);
// Where blocks with a halfway case leave their probabilities: place p holds block[p]'s 2^bb from
// probs[p * 2^bb] on. *count (device memory, zero at the start) may end above `most`.
struct TieBlocks {
  uint32_t* count;
  uint32_t most;
  uint64_t* block;
  double* probs;
};
// Exact sums of rint(p_i * 2^(52-e)) per block for e = ebase[b] + 0..2, and halfway flags.
hipError_t launch_block_exact_sums(int prec, const void* psi, uint64_t dim, int bb, const int32_t* ebase,
                                   double* sums, uint32_t* flags, const TieBlocks& tie, hipStream_t s);
// out[y * 2^bb + q] = re^2 + im^2 (no fused operations) of amplitude q of block list[y] (block y if
// list is null), y < count; out and list may be pinned host memory.
hipError_t launch_gather_probs(int prec, const void* psi, int bb, const uint64_t* list, uint32_t count, double* out,
                               hipStream_t s);
// Resolves each job's draws with its block's exact fold values (bb >= 12).
hipError_t launch_sample_exact_blocks(int prec, const void* psi, uint64_t dim, int bb, const ExactJob* jobs,
                                      uint64_t njobs, const double* u, uint64_t* out, hipStream_t s);
hipError_t launch_norm_partial(int prec, const void* psi, uint64_t dim, double* part, int nblocks,
                               hipStream_t s);
hipError_t launch_gen_partial(int prec, const void* lam, const void* psi, uint64_t dim, int t, int gen,
                              double2* part, int nblocks, hipStream_t s);
// One Pauli-sum term of an X-mask group: coefficient (with i^ny folded in) times
// (-1)^{popcount(j & zm)}.
struct PauliZTerm {
  uint64_t zm;
  double cr, ci;
};
// An X-mask group of a Pauli sum: terms[first .. first + count) share X mask xm.
struct PauliGroup {
  uint64_t xm;
  uint32_t first, count;
};
// lam[o] = sum over groups g, terms t of g: c_t (-1)^{popcount(j & zm_t)} psi[j], j = o ^ xm_g
// (the whole observable in one pass). The first nplain groups have one term, with zm = 0 and ci = 0.
// With `part`, part[0 .. pauli_sum_partials(dim)) = partial sums of Re <psi|lam>.
hipError_t launch_pauli_sum(int prec, void* lam, const void* psi, uint64_t dim, const PauliGroup* groups, int ngroups,
                            int nplain, const PauliZTerm* terms, hipStream_t s, double* part = nullptr);
unsigned pauli_sum_partials(uint64_t dim);
// |0...0> in `count` states of a pool: state y starts at byte base[y] and has 2^bits[y] amplitudes.
hipError_t launch_init_batch(int prec, void* pool, const uint64_t* base, const uint32_t* bits, uint32_t count,
                             hipStream_t s);
// grads[r] = sum of part[r * ncols ..], r < nrows; energy[0] = sum of dot[0 .. ndot); stamp[0] = the
// device clock when both are done.
hipError_t launch_finish_instance(const double* part, uint64_t ncols, uint32_t nrows, double* grads, const double* dot,
                                  uint64_t ndot, double* energy, uint64_t* stamp, hipStream_t s);
// |0...0> in each of `count` states of dim amplitudes stored back to back.
hipError_t launch_init_instances(int prec, void* psi, uint64_t dim, uint64_t count, hipStream_t s);
// For each of `count` states stored back to back: its draws u[off[y] .. off[y+1]) (ascending)
// placed by the left fold of its probabilities in index order (out = first index whose
// cumulative probability exceeds the draw, UINT64_MAX if none).
hipError_t launch_sample_fold_instances(int prec, const void* psi, uint64_t dim, uint64_t count, const double* u,
                                        const uint64_t* off, uint64_t* out, hipStream_t s);
// part[b] = partial sums of Re <psi| O |psi> over nblocks blocks, O as in launch_pauli_sum
// (added to part[b] with `accumulate`). Every group costs a read of the state.
hipError_t launch_pauli_expect(int prec, const void* psi, uint64_t dim, const PauliGroup* groups, int ngroups,
                               const PauliZTerm* terms, double* part, int nblocks, hipStream_t s,
                               int accumulate = 0);
// Groups of an observable evaluated together in one read of the state: groups[first ..
// first + count) whose X masks lie in the tile bits tmask (pauli_tile_bits of them), or with
// tmask == 0 groups read directly (X masks too wide for a tile).
struct PauliPass {
  uint64_t tmask;
  uint32_t first, count;
};
// Tile width of the grouped expectation passes: 2^12 complex128 / 2^13 complex64 amplitudes
// (64 KB of LDS, two workgroups per CU), of which the lowest 3 / 4 bits (128-byte segments) are always tile bits.
inline int pauli_tile_bits(int prec) { return prec == 0 ? 12 : 13; }
inline int pauli_low_bits(int prec) { return prec == 0 ? 3 : 4; }
// Device records of the tiled passes (pauli_tile_tables). A pass holds each tile in up to four
// arrangements; arrangement a keeps the tile bits pauli_arrangement_bit(K, a) + 0..3 in a thread's
// 16 registers (the last one only serves the lowest bits of 2^13 tiles).
constexpr int kPauliArrangements = 4;
__host__ __device__ constexpr int pauli_arrangement_bit(int K, int a) { return K - 4 - 4 * a > 0 ? K - 4 - 4 * a : 0; }
// Group ops. 1..15: the X mask is this pattern of the register bits; PAULI_LDS + b: partners read
// from LDS, b = the highest of its register bits.
enum PauliOp : uint32_t { PAULI_DIAG = 0, PAULI_LDS = 16 };
// nre terms with an even number of Y factors, then nim with an odd one; lx = X mask in the tile
// (whole words: the record is read with scalar loads).
struct PauliTileGroup {
  uint32_t op, lx, nre, nim;
};
// One term: its Z mask outside the tile, on the thread's tile bits (lz), and on the register bits
// as a sign pattern (pat); c = its real coefficient, doubled where each pair is taken once.
struct PauliTileTerm {
  uint64_t zout;
  double c;
  uint32_t lz, pat;
};
static_assert(sizeof(PauliTileGroup) == sizeof(PauliGroup) && sizeof(PauliTileTerm) == sizeof(PauliZTerm),
              "tiled and direct passes share one table");
// One pass over the state, its groups by arrangement: with `diag`, X mask 0 (in arrangement 0);
// the register patterns plain[a] whose group is one real term of pattern 0; then cnt[a] other
// groups, whose records lie from `first` on. Terms lie in this order from `term0` on. arrs: the
// arrangements in use; lds: the tile goes through LDS. A direct pass has tmask 0 and cnt[0] groups.
struct PauliTilePass {
  uint64_t tmask;
  uint32_t first, term0, lds, diag, arrs;
  uint32_t cnt[kPauliArrangements], plain[kPauliArrangements];
};
constexpr uint32_t kPauliPassesPerLaunch = 16;  // passes travel as a kernel argument
struct PauliTilePasses {
  uint32_t count;
  uint32_t diag_count[16];  // X mask 0: its terms are sorted by pattern; how many each has
  PauliTilePass p[kPauliPassesPerLaunch];
};
// Partial sums (workgroups) of every expectation pass over a state of dim amplitudes.
int pauli_expect_partials(uint64_t dim);
// part[0 .. pauli_expect_partials(dim)) = partial sums of Re <psi|O|psi>, pass after pass, from
// the records of pauli_tile_tables.
hipError_t launch_pauli_expect_passes(int prec, const void* psi, uint64_t dim, const void* groups, const void* terms,
                                      const PauliTilePass* passes, int npasses, const uint32_t* diag_count,
                                      double* part, hipStream_t s);
// psi[i] *= f for every amplitude, in place (the streaming ceiling of a sweep).
hipError_t launch_stream_scale(int prec, void* psi, uint64_t dim, double f, hipStream_t s);
// out[0] = the device wall clock (constant-rate counter).
hipError_t launch_stamp(uint64_t* out, hipStream_t s);
// out[r] = sum of part[r * ncols + 0 .. ncols-1] (fixed order), r < nrows.
hipError_t launch_sum_rows(const double* part, uint64_t ncols, uint32_t nrows, double* out, hipStream_t s);
hipError_t launch_f64_to_c64(float2* dst, const double2* src, uint64_t n, hipStream_t s);
hipError_t launch_c64_to_f64(double2* dst, const float2* src, uint64_t n, hipStream_t s);

}  // namespace qr

// MI355X (gfx950) FCIQMC walker-propagation engine: implementation of the
// C-ABI in include/fqmc.h.
//
// One call to fq_cycle runs the body of the reference's Monte Carlo cycle
// (src/fciqmc.f90:307-399) on the device:
//   spawning + death      production: k_det_pass (one thread per determinant:
//                         projected energy, initiator flag, decide_nattempts,
//                         stochastic death) then k_spawn (one thread per
//                         spawning attempt; parents found in a per-tile window
//                         of the attempt prefix sum; results written to the
//                         attempt's staging slot, then packed in attempt order
//                         by a prefix-sum compaction: no atomics).
//                         replay: k_replay_walk, one thread walking the list
//                         in the reference's order and consuming the uploaded
//                         dSFMT stream exactly as get_rand_close_open does.
//   sort                  production: LSD radix sort (8- or 9-bit digits, stable;
//                         short lists by one block in LDS) of the spawned list's
//                         sort values: combinatorial ranks, which order
//                         determinants as their bit strings do in fewer bits, or
//                         the bit strings where that saves no pass.
//                         replay: the reference's quicksort (src/sort.f90:213-396)
//                         on one thread, so equal keys keep its order.
//   self-annihilation,    k_run_count / k_runs: one thread per run of equal keys,
//   merge, rounding of    plain and initiator rules (src/spawn_data.F90:859-1101);
//   new determinants      the run's sort value looked up in the tile's window of
//                         the main list's values (src/annihilation.f90:294-486);
//                         new determinants rounded and listed.
//   rounding, compaction  k_round: stochastic rounding of small real populations
//                         (src/annihilation.f90:537-675), draws from Philox or from
//                         the replay stream at scan offsets.
//   insertion             k_scatter_main / k_scatter_new: merge-path placement
//                         of surviving main entries and new determinants into the
//                         other buffer, new K_ii from the Slater--Condon diagonal
//                         (src/annihilation.f90:677-901).
// fq_cycle_batch runs the same kernels over many independent instances held in
// one list; the heat-bath tables and the learned proposal are built here and
// in mlp.hip.
// Memory layout (HBM, structure of arrays): determinant word w of entry i at
// det[w*cap + i]; population of space s at pop[s*cap + i]; K_ii at kii[i].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <climits>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <functional>
#include <mutex>
#include <queue>
#include <thread>
#include <type_traits>
#include <vector>

#include "device_common.hpp"
#include "fqmc.h"
#include "mlp.hpp"

using fqd::Sys;

// ---------------------------------------------------------------------------
// Fixed scratch of fq_cycle_noalloc, for callers that cannot allocate device
// memory.  One region per scratch slot (int64 elements): the prefix sums'
// tile sums (slot 0) and tile offsets (slot 1), sized for every scan an
// engine can issue (at most 2^31 entries, tiles of 4096).  Every device holds
// its own copy until the process ends; host code reaches it only through the
// address hipGetSymbolAddress returns with that device current (the array's
// name is a host-side stand-in).  Calls that overlap on one device share it
// and race.
// ---------------------------------------------------------------------------
constexpr int kScratchSlots = 2;
constexpr int64_t kScratchSlotElems[kScratchSlots] = {(int64_t{1} << 19) + 64, (int64_t{1} << 19) + 64};
__host__ __device__ constexpr int64_t scratch_slot_offset(int slot) {
  int64_t off = 0;
  for (int k = 0; k < slot; ++k) off += (kScratchSlotElems[k] + 31) / 32 * 32;  // 256-byte aligned regions
  return off;
}
constexpr int64_t kScratchElems = scratch_slot_offset(kScratchSlots);
static __device__ __align__(256) int64_t scratch[kScratchElems];

namespace {

constexpr int kBlock = 256;
// Batched instances share one list: the instance index sits in bits 48..63 of
// word 0 above the orbital bits (systems of at most 48 spin orbitals).
constexpr int kInstShift = 48;
constexpr uint64_t kOrbMask = (uint64_t{1} << kInstShift) - 1;
constexpr int kMaxInst = 1 << 16;
constexpr int kRunTile = 4 * kBlock;   // sorted entries per run tile
constexpr int kMainTile = 4 * kBlock;  // main-list entries per rounding and insertion tile
// Counts of up to this many blocks or tiles are prefixed by every block that
// needs them (its threads add the counts before its own, work that grows with the
// square of the list); more of them are scanned first.  Both ways on an 18-site
// ring, scan against sums, us:
// * attempts of k_det_pass's blocks, with the scans of more than 8192 counts in
//   two launches or three: 87 and 80 for the determinant pass and k_att_scan at
//   16300 blocks (4.2e6 determinants), 104 and 104 at 21700, 167 and 194 at 42200;
// * run heads and new determinants of the run tiles (k_runs, k_round), and the
//   network's rows (k_mlp_rows): reduction 117 and 111, rounding and insertion 201
//   and 204 at 3900 tiles; 160 and 155, 347 and 360 at 5650; 411 and 438, 868 and
//   935 at 13800; rows 54 and 52 at 3900 tiles, 88 and 94 at 7800;
// * survivors of the main tiles (k_scatter_main, whose blocks add the whole list's
//   as well): rounding and insertion 42.7 and 41.4 at 2100 tiles, 55 and 57 at
//   3000, 101 and 109 at 5400, 272 and 375 at 15500.
constexpr int64_t kPrefixAttempts = 16384;
constexpr int64_t kPrefixRuns = 4096;
constexpr int64_t kPrefixMain = 2048;
constexpr int64_t kListSlotBytes = int64_t{1} << 20;  // a pinned slot of fq_download
// Words per spawned-list record (populations, flag), padded to 16-byte
// alignment so one record is one aligned read after the sort's permutation.
__host__ __device__ constexpr int rec_stride(int S) { return S == 1 ? 2 : 4; }

#define FQ_HIP(call)                                  \
  do {                                                \
    hipError_t err_ = (call);                         \
    if (err_ != hipSuccess) {                         \
      fprintf(stderr, "fqmc: %s failed: %s (%s:%d)\n", #call, hipGetErrorString(err_), __FILE__, __LINE__); \
      return FQ_ERR_DEVICE;                           \
    }                                                 \
  } while (0)

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline unsigned grid_for(int64_t n, int64_t per_block = kBlock) {
  int64_t g = ceil_div(n, per_block);
  if (g < 1) g = 1;
  return static_cast<unsigned>(g);
}

// Times of a cycle's phases: block 0 of a phase's first kernel notes the device's
// constant-rate clock as it starts, so the phases are timed without event packets
// between the kernels (a record costs the queue 2-4 us; a cycle took 16).
enum Stamp { kStBegin, kStProposal, kStScan, kStSpawn, kStSort, kStRuns, kStRound, kStFinish, kStEnd, kStamps };

// Per-cycle device counters.
struct Stats {
  double proj[FQ_MAX_SPACES];
  double d0[FQ_MAX_SPACES];
  int64_t ndeath;
  int64_t nspawn;          // spawned entries requested (may exceed capacity)
  int64_t spawn_overflow;
  int64_t total_attempts;
  int64_t nruns;
  int64_t nnew;            // surviving new determinants
  int64_t nmain;           // surviving main-list entries
  int64_t new_n;
  int64_t main_overflow;
  int64_t rng_pos;
  int64_t rng_failed;
  unsigned long long abs_pop[FQ_MAX_SPACES];  // sum |pop| after annihilation (encoded)
  int64_t mlp_rows;                           // determinants the network runs on
  int64_t sorted;                             // entries k_sort_small sorted
  int64_t resort;                             // 1: the list was too long for it (nothing downstream ran)
  int64_t spawn_begin, spawn_ticks;           // start of the last spawning launch; time of them all
  int64_t stamp[kStamps];                     // device clock at the start of the phases
};

// The semi-stochastic core as the projection kernels see it: CSR rows of the
// stored Hamiltonian (row i: H_ij over j in combined mode, the transpose
// H_ji in separate mode), the cycle's core populations vec[i * S + s] and
// the main-list position of each core determinant.
struct DetermDev {
  const int64_t* row;
  const int32_t* col;
  const double* mat;
  double* vec;
  int64_t* pos;
  int64_t nd;
  int separate;
};
// A determinant-pass flag bit above the initiator flags: the parent is a core
// determinant (its spawns onto the core are the deterministic projection's).
constexpr uint8_t kCoreFlag = 0x80;
constexpr uint8_t kInitFlagMask = 0x7f;

// ---------------------------------------------------------------------------
// Prefix sums.  Up to kSmallScanMax entries: one 1024-thread block (one
// launch).  Up to kPrefixTiles
// tiles: per-tile sums, then each tile adds the sums of the tiles before it
// itself and scans its entries (two launches).  More: the tile sums are
// scanned by the one-block scan in between (three launches).  out[n] = total.
// ---------------------------------------------------------------------------
constexpr int kScanItems = 16;
constexpr int64_t kScanTile = static_cast<int64_t>(kBlock) * kScanItems;
constexpr int kSmallBlock = 1024, kSmallItems = 8;
constexpr int64_t kSmallScanMax = kSmallBlock * kSmallItems;  // one chunk: a single block is latency-bound
constexpr int64_t kPrefixTiles = 2048;

__device__ __forceinline__ void stamp(Stats* st, int which) {
  if (blockIdx.x == 0 && threadIdx.x == 0) st->stamp[which] = wall_clock64();
}

// Inclusive scan of x over the 64 lanes of a wavefront.
__device__ __forceinline__ int64_t wave_inclusive_scan(int64_t x, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int64_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  return x;
}
__device__ __forceinline__ int64_t wave_sum(int64_t x) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) x += __shfl_xor(x, d, 64);
  return x;
}
// Sum of x over a kBlock-thread block (every thread receives it).
__device__ __forceinline__ int64_t block_sum(int64_t x, int64_t* wsh) {
  x = wave_sum(x);
  if ((threadIdx.x & 63) == 0) wsh[threadIdx.x >> 6] = x;
  __syncthreads();
  int64_t t = 0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) t += wsh[w];
  __syncthreads();
  return t;
}

// A list length read on the device when pn is given (launches sized by a
// bound n: production sorts, graph-captured cycles), clamped to the bound.
__device__ __forceinline__ int64_t list_len(const int64_t* __restrict__ pn, int64_t n) {
  if (!pn) return n;
  const int64_t v = *pn;
  return v < n ? v : n;
}
// The cycle index: read on the device in graph-captured cycles.
__device__ __forceinline__ uint32_t cycle_of(const uint32_t* __restrict__ pc, uint32_t cyc) { return pc ? *pc : cyc; }

template <class T>
__global__ __launch_bounds__(kBlock) void k_tile_sums(const T* __restrict__ in, int64_t n,
                                                      int64_t* __restrict__ sums) {
  __shared__ int64_t wsh[kBlock / 64];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile;
  int64_t acc = 0;
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k * kBlock + threadIdx.x;
    if (i < n) acc += in[i];
  }
  acc = block_sum(acc, wsh);
  if (threadIdx.x == 0) sums[blockIdx.x] = acc;
}

// Inclusive Hillis-Steele scan of sh[0..kBlock) in place.
__device__ __forceinline__ void block_inclusive_scan(int64_t* sh) {
  for (int h = 1; h < kBlock; h <<= 1) {
    const int64_t add = threadIdx.x >= h ? sh[threadIdx.x - h] : 0;
    __syncthreads();
    sh[threadIdx.x] += add;
    __syncthreads();
  }
}

// Exclusive scan of one tile (kScanItems consecutive entries per thread) plus
// the tile's offset: with prefix, the sum of part[0..tile) (part: tile sums);
// otherwise part[tile] (part: exclusive tile offsets).  The tile holding
// element n-1 also writes out[n] = total.
template <class T>
__global__ __launch_bounds__(kBlock) void k_tile_scan(const T* __restrict__ in, int64_t n,
                                                      const int64_t* __restrict__ part, int prefix,
                                                      int64_t* __restrict__ out) {
  __shared__ int64_t wsh[kBlock / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t off;
  if (prefix) {
    int64_t pre = 0;
    for (int64_t k = threadIdx.x; k < blockIdx.x; k += kBlock) pre += part[k];
    off = block_sum(pre, wsh);
  } else {
    off = part[blockIdx.x];
  }
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int64_t v[kScanItems];
  int64_t local = 0;
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    v[k] = i < n ? in[i] : 0;
    local += v[k];
  }
  const int64_t x = wave_inclusive_scan(local, lane);
  if (lane == 63) wsh[wave] = x;
  __syncthreads();
  int64_t wpre = 0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) wpre += w < wave ? wsh[w] : 0;
  int64_t run = off + wpre + x - local;
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    if (i < n) out[i] = run;
    run += v[k];
    if (i == n - 1) out[n] = run;
  }
}

// Exclusive scan of n entries on one block of kSmallBlock threads: chunks of
// kSmallBlock * kSmallItems with a running carry (one chunk for the small
// scans; many for the tile sums of a very long array).
template <class T>
__global__ __launch_bounds__(kSmallBlock) void k_scan_small(const T* __restrict__ in, int64_t n,
                                                            int64_t* __restrict__ out) {
  __shared__ int64_t wsh[kSmallBlock / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int64_t carry = 0;
  for (int64_t c0 = 0; c0 < n; c0 += static_cast<int64_t>(kSmallBlock) * kSmallItems) {
    const int64_t base = c0 + static_cast<int64_t>(tid) * kSmallItems;
    int64_t v[kSmallItems];
    int64_t local = 0;
#pragma unroll
    for (int k = 0; k < kSmallItems; ++k) {
      const int64_t i = base + k;
      v[k] = i < n ? in[i] : 0;
      local += v[k];
    }
    const int64_t x = wave_inclusive_scan(local, lane);
    if (lane == 63) wsh[wave] = x;
    __syncthreads();
    int64_t wpre = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kSmallBlock / 64; ++w) {
      const int64_t t = wsh[w];
      wpre += w < wave ? t : 0;
      total += t;
    }
    int64_t run = carry + wpre + x - local;
#pragma unroll
    for (int k = 0; k < kSmallItems; ++k) {
      const int64_t i = base + k;
      if (i < n) out[i] = run;
      run += v[k];
    }
    carry += total;
    __syncthreads();  // wsh is rewritten by the next chunk
  }
  if (tid == 0) out[n] = carry;
}

__global__ void k_set_zero_total(int64_t* __restrict__ out) { out[0] = 0; }

}  // namespace

struct fq_engine {
  int device = 0;
  hipStream_t stream = nullptr;
  Sys sys{};
  Sys* d_sysp = nullptr;    // device copy of sys (read by the spawning kernel)
  bool sys_dirty = true;    // sys changed since the last upload
  fq_params par{};
  int W = 1, S = 1;
  // device tables
  uint8_t* d_sym_diff = nullptr;
  int *d_sym_table = nullptr, *d_inv_sym = nullptr, *d_orb_sym = nullptr, *d_nbss = nullptr, *d_ssbf = nullptr;
  double *d_sp_eigv = nullptr, *d_h1 = nullptr, *d_eri = nullptr, *d_jmat = nullptr, *d_kmat = nullptr;
  double *d_s1j = nullptr, *d_s1k = nullptr;
  // Graph-captured batched cycles: while one is captured (capturing), the
  // main list's length is read on the device from dn and the cycle index from
  // dcyc (the graph's first copy fills both from pinned host memory, h_in),
  // and launches are sized by bounds.
  // online training of the learned proposal (fq_mlp_online): steps of batch
  // samples at the start of every online_every-th cycle
  int32_t online_every = 0, online_steps = 0;
  int64_t online_batch = 0;
  double online_lr = 0.0;
  int64_t online_runs = 0;
  bool capturing = false;
  const int64_t* dn = nullptr;
  const uint32_t* dcyc = nullptr;
  bool graph_on = false;
  char* h_in = nullptr;       // pinned: [n][cycle index][tau, shift, E_proj per instance]
  char* d_in = nullptr;
  double* h_god = nullptr;    // pinned copies the graph writes at its end
  int64_t* h_goi = nullptr;
  struct GraphEntry {
    int c;
    int64_t nb, tb;
    int sched;
    hipGraphExec_t exec;
  };
  std::vector<GraphEntry> graphs;
  // the tuner, per octave of the attempt bound: the chosen schedule (-1:
  // still trying candidates), cycles tried and each candidate's timings
  int sched[64];
  int tune_iter[64];
  std::vector<float> tune_ms[64][8];
  int last_oct = -1;          // octave of the last graph cycle
  int64_t graph_cycles = 0, eager_cycles = 0;
  hipEvent_t gev[2] = {nullptr, nullptr};
  // schedule knobs (the tuner's candidates): 8-bit radix digits only, and a
  // cap on the spawning grid (0: one block per tile)
  int digit8 = 0;
  int spawn_blocks = 0;
  double* d_recip = nullptr;  // 1.0 / k, k < kRecipN
  int* d_jpair = nullptr;     // choose_ij_mol's j index per pair index
  // heat-bath tables (excit_gen FQ_EXCIT_HEAT_BATH)
  double *d_hb_i = nullptr, *d_hb_ij = nullptr, *d_hb_ija = nullptr, *d_hb_ija_tot = nullptr, *d_hb_ija_u = nullptr;
  double *d_hb_ijab = nullptr, *d_hb_ijab_tot = nullptr, *d_hb_ijab_u = nullptr;
  int *d_hb_ija_k = nullptr, *d_hb_ijab_k = nullptr, *d_hb_bias = nullptr;
  // batched independent instances (fq_create_batch): instance index in bits
  // 48..63 of word 0; per-instance tables held by sub-engines
  bool batched = false;
  int ninst = 1;
  int key_bits = 0;                  // key bits the radix sort orders (nbasis, or 48 + instance bits)
  int rank_words = 0, rank_bits = 0;  // production sort on combinatorial ranks (0: on the bit strings)
  uint64_t* d_binom = nullptr;        // C(p, i), p < nbasis, 1 <= i <= nel, as (low, high) halves
  std::vector<fq_engine*> subs;
  Sys* d_sys_arr = nullptr;          // [ninst]
  double* d_ipar = nullptr;          // tau[ninst], shift[S][ninst], eproj_old[S][ninst]
  int64_t* d_ibound = nullptr;       // [2][ninst + 1]: instance bounds of the old and the new list
  int64_t* d_isb = nullptr;          // [ninst + 1]: instance bounds of the spawned list
  int64_t* d_iatt = nullptr;         // [ninst]: first attempt of each instance
  double* d_cterm = nullptr;         // [2S][cap]: per-determinant projected-energy and N_0 terms
  int64_t* d_cdeath = nullptr;       // [cap]
  // per-instance 256-entry block counts and offsets (old list, new list) and
  // the block partials of the estimator terms (2S), deaths and |N| (1 + S)
  int64_t *d_iblk_cnt = nullptr, *d_iblk_off = nullptr, *d_nblk_off = nullptr;
  double* d_ipart_d = nullptr;
  int64_t* d_ipart_i = nullptr;
  int64_t ipb = 0;  // partial stride: a bound of the blocks of either list
  double* d_iout_d = nullptr;        // [ninst][2S]
  int64_t* d_iout_i = nullptr;       // [ninst][4 + S]
  // learned proposal (excit_gen FQ_EXCIT_LEARNED): network, per-determinant weights
  fqm::Mlp mlp;
  float* mlp_tab = nullptr;  // rows x 2*nbasis, one row per determinant the network runs on
  float* mlp_flat = nullptr;  // 2*nbasis ones: weights of determinants without a row
  int64_t att_bound = -1;            // bound of the next cycle's attempts (-1: unknown)
  bool keys_ready = false;           // the spawning pass made this cycle's sort keys
  int64_t last_ns = -1;              // spawned entries last annihilated (-1: none on this list)
  int64_t resorts = 0;               // lists that outgrew the one-block sort they were given to
  int new_src = 0;                   // the sort's idle buffers after this cycle's passes
  // counts that the kernels that need their prefix add up themselves
  int64_t prefix_attempts = kPrefixAttempts, prefix_runs = kPrefixRuns, prefix_main = kPrefixMain;
  int64_t run_tiles = 0;             // run tiles of this cycle's spawned list (a bound of it while captured)
  int64_t mlp_tab_rows = 0;
  int cls_sorted = 0;          // the spin/irrep classes list their orbitals in ascending order
  int32_t* mlp_row = nullptr;  // [cap] this cycle's row of the weight table (-1: none)
  int64_t* mlp_idx = nullptr;  // [cap] determinants the network runs on
  // main list: determinants, K_ii and sort values in buffer cur, the insertion
  // writing the other; populations in pop, which the cycle has done with when
  // the insertion writes them from pop_new
  int64_t cap = 0, n = 0;
  int cur = 0;
  uint64_t* det[2] = {nullptr, nullptr};
  int64_t* pop = nullptr;       // S*cap
  double* kii[2] = {nullptr, nullptr};
  int64_t* pop_new = nullptr;   // S*cap, populations after death
  int64_t* att_off = nullptr;   // S*cap+1 attempt offsets (null: see att_offsets)
  uint64_t* mrank[2] = {nullptr, nullptr};  // sort_kw*cap + 1: the entries' sort values (ranks), as the list's buffers
  uint64_t* mmask = nullptr;    // surviving main entries, one bit each, by tiles of kMainTile
  uint16_t* mpre = nullptr;     // per word of mmask: survivors of its tile before it
  int32_t* mcnt = nullptr;      // survivors per tile
  int64_t* moff = nullptr;      // survivors before each tile; [tiles] = their number
  int64_t* mdraw = nullptr;     // cap+1 (replay rounding draws)
  int64_t* mdraw_off = nullptr;
  double* part_d = nullptr;     // 4 * (cap/256+1) block partials
  int64_t* part_i = nullptr;    // 2 * (cap/256+1)
  int64_t* blk_att = nullptr;   // cap/256+2: attempts of k_det_pass's blocks
  int64_t* blk_off = nullptr;   // their exclusive prefix (more than kPrefixAttempts of them)
  // spawning-attempt staging (one slot per attempt of a batch)
  int64_t bcap = 0;
  uint64_t* st_det = nullptr;   // W*bcap
  int64_t* st_pop = nullptr;    // bcap
  uint16_t* st_ent = nullptr;   // bcap: spawning space, parent's initiator flags from bit 8
  int32_t* tile_cnt = nullptr;  // successes per spawning tile (bcap / kSmallTile + 2)
  int64_t* tile_win = nullptr;  // parents of each tile's first and last attempt
  // spawned list
  int64_t scap = 0;
  uint64_t* sdet = nullptr;  // W*scap (in kbuf[1])
  int64_t* srec = nullptr;   // scap records: S populations then the flag, rec_stride(S) words each (in pbuf[1])
  // sort: keys (value << flag_bits | flags) and payload (populations), ping-pong
  int sort_kw = 1, flag_bits = 1, value_bits = 1;
  uint64_t* kbuf[2] = {nullptr, nullptr};  // sort_kw * scap
  int64_t* pbuf[2] = {nullptr, nullptr};   // S * scap
  uint32_t* perm = nullptr;                // scap: replay quicksort order
  int64_t* pass_cnt = nullptr;             // 512 * kSortBlocks digit counts of a pass's blocks
  int64_t* pass_off = nullptr;             // their exclusive prefix (+ total)
  int32_t* run_tcnt = nullptr;             // run heads per run tile
  int64_t* run_toff = nullptr;             // their exclusive prefix (more than kPrefixRuns tiles)
  int32_t* run_tfirst = nullptr;           // first head of each run tile (-1: none)
  int64_t* run_tpre = nullptr;             // sums of each run tile's entries before its first head
  int64_t* run_win = nullptr;              // main-list position of each run tile's first value; then the end
  // new determinants: per run tile (values and populations in the sort's idle
  // buffers, positions in new_pos[0]), then in one list
  int32_t* new_cnt = nullptr;    // per run tile
  int64_t* new_off = nullptr;    // their exclusive prefix (more than kPrefixRuns tiles)
  int32_t* new_pos[2] = {nullptr, nullptr};  // scap: insertion positions (non-decreasing): staged, listed
  uint64_t* new_val = nullptr;   // sort_kw*scap: sort values of the new determinants
  int64_t* new_pop = nullptr;    // S*scap: their populations
  int64_t* abs_part = nullptr;   // |N| sums of the insertion's blocks
  int64_t* ndraw = nullptr;      // replay: rounding draws of each run tile's candidates
  int64_t* ndraw_off = nullptr;
  // scan scratch
  std::vector<int64_t*> scan_tmp;
  std::vector<int64_t> scan_tmp_cap;
  // fq_cycle_spawn .. fq_cycle_finish: a cycle split at the spawned list (replay mode)
  bool pending = false;
  uint32_t pend_cyc = 0;
  int64_t pend_rng_pos = 0;   // stream position after the spawning pass
  int64_t pend_ns = 0;        // entries this engine spawned
  Stats pend_stats{};         // the spawning pass's counters
  // fq_cycle_noalloc: scratch slots come from the device's fixed array
  int64_t* fixed_scratch = nullptr;  // device address of `scratch` on this engine's device (null: unavailable)
  bool noalloc = false;              // inside fq_cycle_noalloc
  bool scratch_short = false;        // a request exceeded its fixed slot
  // replay stream
  double* rng_buf = nullptr;
  int64_t rng_cap = 0, rng_pos = 0, rng_end = 0;
  // per-cycle
  Stats* d_stats = nullptr;
  Stats* h_pin = nullptr;  // pinned: the cycle's finished stats (k_finish)
  Stats h_stats{};
  uint64_t cycle_index = 0;
  // fq_download's pinned slots (one block of them, made on first use), their
  // events, and the streams they share with the engine's (a stream takes ~1 ms to make)
  static constexpr int kListSlots = 6, kListStreams = 3;
  hipStream_t list_stream[kListStreams] = {};
  std::mutex list_mutex;  // a download at a time: they share the slots
  uint64_t* list_buf = nullptr;
  int list_slots = 0;
  hipEvent_t list_ev[kListSlots] = {};
  // the spawned-list length, spawn overflow and attempt total, copied behind
  // the spawning kernels into pinned memory (h_len) and marked by ev_len
  int64_t* h_len = nullptr;
  hipEvent_t ev_len = nullptr;
  int64_t spawn_bound = 0;  // attempts the cycle's spawning launches covered
  // semi-stochastic core (fq_semi_stoch_init): its determinants (word-major,
  // sorted as the main list; also in sys.determ), the Hamiltonian among them
  // as CSR rows (the transpose for separate annihilation), and per cycle the
  // core populations and their main-list positions
  int64_t ndeterm = 0, determ_nnz = 0;
  int determ_separate = 0;
  uint64_t* d_determ = nullptr;
  int64_t* d_drow = nullptr;
  int32_t* d_dcol = nullptr;
  double* d_dmat = nullptr;
  double* d_dvec = nullptr;
  int64_t* d_dpos = nullptr;
  float t_spawn = 0, t_annih = 0, t_total = 0;
  double ms_per_tick = 1e-5;  // of the device clock
  int spawn_launches = 0;
  fq_profile_out prof{};
  int radix_passes = 0;
};

namespace {

// ---- device allocation helpers ---------------------------------------------
template <class T>
int dalloc(T** p, int64_t count) {
  if (count <= 0) count = 1;
  if (hipMalloc(reinterpret_cast<void**>(p), sizeof(T) * static_cast<size_t>(count)) != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();  // the caller may do without it
    return FQ_ERR_NOMEM;
  }
  return FQ_OK;
}
template <class T>
void dfree(T*& p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

// What a cycle needs of its determinants until their spawns are packed lies in
// the list's idle buffer, which the insertion writes after that: the attempts
// per (det, space) entry (4 S <= 8 bytes) with the K_ii, the parents' initiator
// flags (one byte) with the determinants, and, where the sort values are two
// words, the attempt offsets (8 S <= 16 bytes) with those.  So a slot of the
// main list takes no more memory with its sort values kept than without.
int32_t* att_counts(const fq_engine* e) { return reinterpret_cast<int32_t*>(e->kii[1 - e->cur]); }
uint8_t* parent_flags(const fq_engine* e) { return reinterpret_cast<uint8_t*>(e->det[1 - e->cur]); }
int64_t* att_offsets(const fq_engine* e) {
  return e->att_off ? e->att_off : reinterpret_cast<int64_t*>(e->mrank[1 - e->cur]);
}

// Device address of the fixed scratch array on `device` (current), looked up
// once per device; null if the lookup fails.
int64_t* fixed_scratch_address(int device) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static int64_t* addr[kMaxDevices] = {};
  static bool looked[kMaxDevices] = {};
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(mu);
  if (!looked[device]) {
    void* p = nullptr;
    const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess) {
      fprintf(stderr, "fqmc: hipGetSymbolAddress(scratch) on device %d failed: %s\n", device,
              hipGetErrorString(err));
      p = nullptr;
    }
    addr[device] = static_cast<int64_t*>(p);
    looked[device] = true;
  }
  return addr[device];
}

// Scratch buffer `slot` of at least `need` elements (grown on demand; inside
// fq_cycle_noalloc, the slot's region of the fixed array, or null when the
// request exceeds it).  Captured graphs hold the buffer's address, so from
// fq_batch_graph on, which sizes it for the engine's longest scan, it stays.
int64_t* scan_scratch(fq_engine* e, int slot, int64_t need) {
  if (e->noalloc) {
    if (slot >= kScratchSlots || need > kScratchSlotElems[slot]) {
      e->scratch_short = true;
      return nullptr;
    }
    return e->fixed_scratch + scratch_slot_offset(slot);
  }
  while (static_cast<int>(e->scan_tmp.size()) <= slot) {
    e->scan_tmp.push_back(nullptr);
    e->scan_tmp_cap.push_back(0);
  }
  if (e->scan_tmp_cap[slot] < need) {
    if (e->h_in) return nullptr;
    dfree(e->scan_tmp[slot]);
    if (dalloc(&e->scan_tmp[slot], need) != FQ_OK) {
      e->scan_tmp_cap[slot] = 0;
      return nullptr;
    }
    e->scan_tmp_cap[slot] = need;
  }
  return e->scan_tmp[slot];
}

// Exclusive scan: out[0..n] with out[n] = total (in and out distinct).
template <class T>
int scan_exclusive(fq_engine* e, const T* in, int64_t* out, int64_t n) {
  if (n == 0) {
    hipLaunchKernelGGL(k_set_zero_total, dim3(1), dim3(1), 0, e->stream, out);
    return FQ_OK;
  }
  if (n <= kSmallScanMax) {
    hipLaunchKernelGGL(k_scan_small<T>, dim3(1), dim3(kSmallBlock), 0, e->stream, in, n, out);
    return FQ_OK;
  }
  const int64_t nb = ceil_div(n, kScanTile);
  int64_t* sums = scan_scratch(e, 0, nb);
  if (!sums) return FQ_ERR_NOMEM;
  hipLaunchKernelGGL(k_tile_sums<T>, dim3(static_cast<unsigned>(nb)), dim3(kBlock), 0, e->stream, in, n, sums);
  if (nb <= kPrefixTiles) {
    hipLaunchKernelGGL(k_tile_scan<T>, dim3(static_cast<unsigned>(nb)), dim3(kBlock), 0, e->stream, in, n, sums, 1,
                       out);
    return FQ_OK;
  }
  int64_t* offs = scan_scratch(e, 1, nb + 1);
  if (!offs) return FQ_ERR_NOMEM;
  hipLaunchKernelGGL(k_scan_small<int64_t>, dim3(1), dim3(kSmallBlock), 0, e->stream, sums, nb, offs);
  hipLaunchKernelGGL(k_tile_scan<T>, dim3(static_cast<unsigned>(nb)), dim3(kBlock), 0, e->stream, in, n, offs, 0, out);
  return FQ_OK;
}

// ---------------------------------------------------------------------------
// Kernels: spawning and death
// ---------------------------------------------------------------------------
__device__ __forceinline__ void load_det(const uint64_t* det, int64_t cap, int W, int64_t i, uint64_t* f) {
#pragma unroll
  for (int w = 0; w < FQ_MAX_WORDS; ++w) f[w] = w < W ? det[w * cap + i] : 0;
}

static_assert(sizeof(Stats) % sizeof(int64_t) == 0, "Stats is cleared and copied as int64 words");
// A cycle's first kernel clears its counters (no later kernel runs beside it) and notes its start.
__device__ __forceinline__ void clear_stats(Stats* st) {
  if (blockIdx.x == 0 && threadIdx.x < sizeof(Stats) / sizeof(int64_t)) {
    constexpr unsigned begin = offsetof(Stats, stamp) / sizeof(int64_t) + kStBegin;
    reinterpret_cast<int64_t*>(st)[threadIdx.x] = threadIdx.x == begin ? static_cast<int64_t>(wall_clock64()) : 0;
  }
}
// Tree sums of NQ arrays of kBlock values in LDS (value t plus value t + h for
// h = 128, 64, ..., 1) into their first elements; the last six levels within
// the first wavefront.  Every thread of the block calls it, after a barrier.
template <int NQ>
__device__ __forceinline__ void block_tree_sum(double (&sh)[NQ][kBlock], int tid) {
#pragma unroll
  for (int h = kBlock / 2; h >= 64; h >>= 1) {
    if (tid < h)
      for (int q = 0; q < NQ; ++q) sh[q][tid] += sh[q][tid + h];
    __syncthreads();
  }
  if (tid < 64) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      double x = sh[q][tid];
#pragma unroll
      for (int h = 32; h > 0; h >>= 1) x += __shfl_down(x, h, 64);  // lanes past 64 - h add their own value: unused
      if (tid == 0) sh[q][0] = x;
    }
  }
}

// Production: per determinant (loop body of src/fciqmc.f90:315-374 minus the
// spawning attempts).  Block partial sums (projected energy, reference
// population, deaths) are reduced in a fixed order by k_finish, so the
// estimators are deterministic and no global atomics are issued.  A
// semi-stochastic core determinant (set_determ_info) records its population
// and position for the projection, is flagged an initiator with kCoreFlag,
// and skips death.  Each block also sums its attempts (blk_att, for k_att_scan).
template <int S>
__global__ __launch_bounds__(kBlock) void k_det_pass(Sys s, int64_t n, int64_t cap, const uint64_t* __restrict__ det,
                                                     const int64_t* __restrict__ pop, const double* __restrict__ kii,
                                                     int64_t* __restrict__ pop_new, int32_t* __restrict__ nat,
                                                     uint8_t* __restrict__ flags, double tau, double sh0, double sh1,
                                                     double e0, double e1, uint64_t seed, uint32_t cyc,
                                                     double* __restrict__ part_d, int64_t* __restrict__ part_i,
                                                     double* __restrict__ dvec, int64_t* __restrict__ dpos,
                                                     int64_t* __restrict__ blk_att, Stats* __restrict__ st) {
  __shared__ double sh_d[2 * S][kBlock];
  __shared__ int64_t wsh[kBlock / 64];
  clear_stats(st);
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  double proj[FQ_MAX_SPACES] = {0.0, 0.0}, d0[FQ_MAX_SPACES] = {0.0, 0.0};
  int64_t ndeath = 0, att = 0;
  if (i < n) {
    uint64_t f[FQ_MAX_WORDS];
    load_det(det, cap, s.W, i, f);
    double rp[FQ_MAX_SPACES] = {0.0, 0.0};
    int64_t p[FQ_MAX_SPACES] = {0, 0};
    for (int sp = 0; sp < S; ++sp) {
      p[sp] = pop[sp * cap + i];
      rp[sp] = static_cast<double>(p[sp]) / static_cast<double>(s.rf);
    }
    const int64_t ci = s.ndeterm > 0 ? fqd::core_index(s, f) : -1;
    if (ci >= 0) {
      for (int sp = 0; sp < S; ++sp) dvec[ci * S + sp] = rp[sp];
      dpos[ci] = i;
    }
    flags[i] = ci >= 0 ? kCoreFlag : static_cast<uint8_t>(fqd::parent_flag(s, rp));
    const double K = kii[i];
    for (int sp = 0; sp < S; ++sp) {
      fqd::proj_energy_term(s, f, rp[sp], proj[sp], d0[sp]);
      const uint32_t hi = static_cast<uint32_t>(i >> 32) ^ (static_cast<uint32_t>(sp) << 28);
      fqd::Philox rng(seed, static_cast<uint32_t>(i), hi, cyc ^ (fqd::kDrawNattempts << 24));
      const int32_t na = fqd::decide_nattempts(rng, rp[sp]);
      nat[i * S + sp] = na;
      att += na;
      int64_t q = p[sp];
      if (ci < 0) {
        fqd::Philox rd(seed, static_cast<uint32_t>(i), hi, cyc ^ (fqd::kDrawDeath << 24));
        ndeath += fqd::death(rd, tau, K, sp == 0 ? sh0 : sh1, sp == 0 ? e0 : e1, q);
      }
      pop_new[sp * cap + i] = q;
    }
  }
  for (int sp = 0; sp < S; ++sp) {
    sh_d[2 * sp][threadIdx.x] = proj[sp];
    sh_d[2 * sp + 1][threadIdx.x] = d0[sp];
  }
  ndeath = block_sum(ndeath, wsh);  // its barriers publish sh_d
  att = block_sum(att, wsh);
  block_tree_sum<2 * S>(sh_d, threadIdx.x);
  if (threadIdx.x == 0) {
    for (int q = 0; q < 2 * S; ++q) part_d[q * gridDim.x + blockIdx.x] = sh_d[q][0];
    part_i[blockIdx.x] = ndeath;
    blk_att[blockIdx.x] = att;
  }
}

// End of a cycle, one block: the k_det_pass block partials (nb of them; 0: the
// estimators are already in the stats) in a fixed order -- thread t of the first
// 256 adds blocks t, t + 256, ..., then a tree -- while the other threads add
// the insertion's |N| block sums (exact integers: any order gives the same
// totals); the finished stats go to pinned host memory from here, so no copy
// follows.
constexpr int kFinishBlock = 1024;
template <int S>
__global__ __launch_bounds__(kFinishBlock) void k_finish(const double* __restrict__ part_d,
                                                         const int64_t* __restrict__ part_i, int nb,
                                                         const int64_t* __restrict__ abs_part, int64_t ld,
                                                         int64_t nabs, Stats* __restrict__ st,
                                                         Stats* __restrict__ host) {
  constexpr int NQ = 2 * S;
  __shared__ double sh[NQ][kBlock];
  __shared__ int64_t wi[1 + S][kFinishBlock / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  stamp(st, kStFinish);
  double acc[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) acc[q] = 0.0;
  int64_t ai = 0, ap[FQ_MAX_SPACES] = {0, 0};
  if (tid < kBlock) {
    // blocks t, t + 256, ... added in that order; 16 (pairs: 8, within the registers) are loaded ahead at a time
    constexpr int kAhead = 16 / S;
    for (int b0 = tid; b0 < nb; b0 += kAhead * kBlock) {
      double v[kAhead][NQ];
      int64_t vi[kAhead];
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int b = b0 + k * kBlock;
#pragma unroll
        for (int q = 0; q < NQ; ++q) v[k][q] = b < nb ? part_d[q * nb + b] : 0.0;
        vi[k] = b < nb ? part_i[b] : 0;
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        if (b0 + k * kBlock < nb) {
#pragma unroll
          for (int q = 0; q < NQ; ++q) acc[q] = acc[q] + v[k][q];
          ai += vi[k];
        }
      }
    }
    for (int q = 0; q < NQ; ++q) sh[q][tid] = acc[q];
  } else {
    for (int sp = 0; sp < S; ++sp)
#pragma unroll 4
      for (int64_t b = tid - kBlock; b < nabs; b += kFinishBlock - kBlock) ap[sp] += abs_part[sp * ld + b];
  }
  ai = wave_sum(ai);
  for (int sp = 0; sp < S; ++sp) ap[sp] = wave_sum(ap[sp]);
  if (lane == 0) {
    wi[0][wave] = ai;
    for (int sp = 0; sp < S; ++sp) wi[1 + sp][wave] = ap[sp];
  }
  __syncthreads();
  block_tree_sum<NQ>(sh, tid);
  if (tid == 0) {
    int64_t t[1 + FQ_MAX_SPACES] = {0, 0, 0};
    for (int w = 0; w < kFinishBlock / 64; ++w)
      for (int q = 0; q < 1 + S; ++q) t[q] += wi[q][w];
    if (nb > 0) {
      for (int sp = 0; sp < S; ++sp) {
        st->proj[sp] = sh[2 * sp][0];
        st->d0[sp] = sh[2 * sp + 1][0];
      }
      st->ndeath = t[0];
    }
    for (int sp = 0; sp < S; ++sp) st->abs_pop[sp] = static_cast<unsigned long long>(t[1 + sp]);
    st->stamp[kStEnd] = wall_clock64();
  }
  __syncthreads();
  if (tid < static_cast<int>(sizeof(Stats) / sizeof(int64_t)))
    reinterpret_cast<int64_t*>(host)[tid] = reinterpret_cast<const volatile int64_t*>(st)[tid];
}

// Last entry e in [lo, hi] with att_off[e] <= t.
__device__ __forceinline__ int64_t parent_of(const int64_t* __restrict__ att_off, int64_t t, int64_t lo, int64_t hi) {
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if (att_off[mid] <= t)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// Attempts per spawning tile: kSpawnTile, or kSmallTile for cycles whose
// attempts would not fill the chip with tiles of 1024 (a tile's four rounds run
// one after the other in its block: 39 us for 10^4 attempts on 26 orbitals, 16
// with four times the blocks; 195 and 105 us for 3.4e5 of the heat-bath generator).
constexpr int kSpawnTile = 4 * kBlock, kSmallTile = kBlock;
constexpr int64_t kSmallTileMax = 512 * kSpawnTile;  // attempts up to which the small tile is used

// Attempt offsets: exclusive scan of the attempts of the nent (det, space)
// entries, kScanTile entries a block, out[nent] = total.  part: the sums of
// k_det_pass's blocks (`per` entries each, nblk of them), added up by every
// block for its offset; poff, when given, is their exclusive prefix (lists of
// more than kPrefixAttempts blocks).  The block that holds the first or last attempt
// of a spawning tile (1 << tile_bits attempts, the first ntile tiles) looks its
// parent up among the starts it keeps in LDS and notes it as that end of the
// tile's parent window, so no search precedes the spawning kernel.  (2.8e6
// entries, 1.1e7 attempts, the densest of them in the first blocks: 34 us;
// tile sums, scan and a search of the offsets per tile took 46, in four
// launches.)
__global__ __launch_bounds__(kBlock) void k_att_scan(const int32_t* __restrict__ in, int64_t nent,
                                                     const int64_t* __restrict__ part, int64_t nblk, int per,
                                                     const int64_t* __restrict__ poff, int64_t* __restrict__ out,
                                                     int64_t* __restrict__ tile_win, int64_t ntile, int tile_bits,
                                                     Stats* __restrict__ st) {
  __shared__ int64_t wsh[kBlock / 64];
  stamp(st, kStScan);
  __shared__ int64_t start[kScanTile + 1];  // first attempt of each entry of the block; then the end
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t b0 = static_cast<int64_t>(blockIdx.x) * (kScanTile / per);
  int64_t off, total;
  if (poff) {
    off = poff[b0 < nblk ? b0 : nblk];
    total = poff[nblk];
  } else {
    int64_t pre = 0, all = 0;
#pragma unroll 4
    for (int64_t k = threadIdx.x; k < nblk; k += kBlock) {
      const int64_t v = part[k];
      all += v;
      pre += k < b0 ? v : 0;
    }
    off = block_sum(pre, wsh);
    total = block_sum(all, wsh);
  }
  // a wavefront's 64 x kScanItems entries, 64 consecutive ones a round (coalesced)
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + wave * (64 * kScanItems) + lane;
  int32_t v[kScanItems];
  int64_t local = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + 64 * k;
    v[k] = i < nent ? in[i] : 0;
    local += v[k];
  }
  local = wave_sum(local);
  if (lane == 0) wsh[wave] = local;
  __syncthreads();
  int64_t carry = off;  // attempts before the wavefront's round
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) carry += w < wave ? wsh[w] : 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + 64 * k;
    const int64_t end = carry + wave_inclusive_scan(static_cast<int64_t>(v[k]), lane), run = end - v[k];
    if (i < nent) out[i] = run;
    start[(wave * kScanItems + k) * 64 + lane] = run;
    carry = __shfl(end, 63, 64);
  }
  if (threadIdx.x == kBlock - 1) start[kScanTile] = carry;  // the block's last wavefront, lane 63
  __syncthreads();
  // entry of attempt x of this block: the last one starting at or before it (it has attempts)
  auto entry_of = [&](int64_t x) {
    int lo = 0, hi = static_cast<int>(kScanTile) - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (start[mid] <= x)
        lo = mid;
      else
        hi = mid - 1;
    }
    return static_cast<int64_t>(blockIdx.x) * kScanTile + lo;
  };
  const int64_t beg = off, fin = start[kScanTile];
  for (int64_t t = (beg >> tile_bits) + threadIdx.x; (t << tile_bits) < fin && t < ntile; t += kBlock) {
    const int64_t t0 = t << tile_bits, t1 = t0 + (int64_t{1} << tile_bits), last = (t1 < total ? t1 : total) - 1;
    if (t0 >= beg) tile_win[2 * t] = entry_of(t0);
    // (a block without attempts, past the total, must not take the last tile's end)
    if (last >= beg && last < fin) tile_win[2 * t + 1] = entry_of(last);
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[nent] = total;
}

// Philox blocks of an attempt's stream generated before its generator runs
// (two draws each: the single/double choice, the orbital choices with their
// first rejection redraws, the spawn rounding).  On mol26 (renormalised
// generator) k_spawn took 474, 465, 454 and 425 us with 0, 2, 3 and 4 blocks;
// 4 keeps its 80 VGPRs (6 waves per SIMD).  A Hubbard attempt draws the pair and
// the rounding, and more only if it spawns: one block (114 -> 112 us for 1.5e6
// attempts on an 18-site ring; with the one-byte partner table, 104).
constexpr int spawn_pre(int g) { return g == fqd::kGenHubK ? 1 : 4; }
// Wavefronts per SIMD the registers are held to.
constexpr int spawn_waves(int g, bool batched) { return g == fqd::kGenMolRenorm && !batched ? 6 : 4; }
constexpr int kRecipN = 4096;  // entries of the host-made reciprocal table

// Parent windows of the tiles of the batch [t_begin, t_end) (kSpawnTile
// attempts each; one thread per tile), for cycles whose attempts take more than
// one batch; t_end is clamped to the attempt total att_off[nent].
__global__ void k_tile_bounds(int64_t nent, const int64_t* __restrict__ att_off, int64_t t_begin, int64_t t_end,
                              int64_t* __restrict__ tile_win) {
  const int64_t tot = att_off[nent];
  t_end = t_end < tot ? t_end : tot;
  const int64_t tile = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t t0 = t_begin + tile * kSpawnTile;
  if (t0 >= t_end) return;
  const int64_t t1 = (t0 + kSpawnTile < t_end) ? t0 + kSpawnTile : t_end;
  const int64_t p0 = parent_of(att_off, t0, 0, nent - 1);
  tile_win[2 * tile] = p0;
  tile_win[2 * tile + 1] = parent_of(att_off, t1 - 1, p0, nent - 1);
}
constexpr int kSpawnWin = 1024;          // parent-window entries staged in LDS

// ---------------------------------------------------------------------------
// Sort keys.  A spawned entry's key is v << flag_bits | flags over kw 64-bit
// words (kw = 1 or 2): v is the determinant's combinatorial rank (or, for
// batched instances, its encoded word 0, instance index included), flags its
// initiator flag bits (one per space).  Ordering the v fields orders
// determinants as the main list does (last word most significant,
// src/bit_utils.F90:452-480); the LSD radix passes order only the digits of
// v and are stable, so equal determinants keep spawned (attempt) order.  The
// entry's populations travel with the key through the passes (the payload),
// so the run reduction reads everything contiguously, and the determinant is
// recovered from v.
//
// Combinatorial rank: for a bit string with set bits p_1 < ... < p_k
// (0-based), rank = sum_i C(p_i, i).  For a fixed number of set bits this is
// a bijection onto [0, C(nbasis, k)) that preserves the strings' numeric
// order, so the sort needs ceil(log2 C(nbasis, nel)) bits instead of nbasis
// (34 instead of 52 for 10 electrons in 52 spin orbitals).  binom holds
// C(p, i) for p < nbasis, 1 <= i <= nel as (low, high) 64-bit halves.
// ---------------------------------------------------------------------------
struct KeyPlan {
  int kw;          // key words
  int flag_bits;   // width of the flag field (the number of spaces)
  int rank;        // 1: v = combinatorial rank; 0: v = determinant word 0
  int nel, nbasis;
  const uint64_t* binom;
  int binom_lds;   // stage the table in dynamic LDS (k_pack_tiles, k_scatter_new)
};
constexpr int kMaxPasses = 16;
struct DigitPlan {
  int np;                  // passes
  int shift[kMaxPasses];   // first key bit of each pass's digit
  int bits[kMaxPasses];    // digit width (8 or 9)
};
// Keys per thread of a sort tile: the tile's keys and payload sit in LDS.  Lists
// that tiles of kSmallSortItems keys a thread spread over at most kSortBlocks
// blocks take those: with the large tiles 2e5 keys ran on 49 of the 256 CUs
// (count and scatter of a 9-bit pass 10 and 13.5 us; 7.4 and 9.2 now).
__host__ __device__ constexpr int sort_items(int kw, int S) { return kw + S <= 2 ? 16 : 8; }
constexpr int kSmallSortItems = 4;
constexpr int kSortBlocks = 512;  // blocks of a radix pass (each owns a contiguous range of tiles)

// STRIDE: words per entry of the table (2: low and high; 1: low words only).
// One-word keys need the sums modulo 2^64 only, so the high words are left out.
template <int KW, int STRIDE>
__device__ __forceinline__ void make_key(const KeyPlan& kp, const uint64_t* f, int W, uint64_t flags, uint64_t* key) {
  using V = typename std::conditional<KW == 1, uint64_t, unsigned __int128>::type;
  static_assert(KW == 1 || STRIDE == 2, "two-word keys read both words");
  V v = 0;
  if (kp.rank) {
    int k = 0;
    FQ_FOR_WORDS(w, W) {
      for (uint64_t x = f[w]; x && k < kp.nel; x &= x - 1) {
        const int p = (w << 6) + __builtin_ctzll(x);
        if (p >= kp.nbasis) break;  // not a determinant of this system (caller-supplied list)
        const uint64_t* c = kp.binom + STRIDE * (p * kp.nel + k);
        if constexpr (KW == 1)
          v += c[0];
        else
          v += (static_cast<unsigned __int128>(c[1]) << 64) | c[0];
        ++k;
      }
    }
  } else {
    v = f[0];
  }
  const V k = (v << kp.flag_bits) | (flags & ((uint64_t{1} << kp.flag_bits) - 1));
  key[0] = static_cast<uint64_t>(k);
  if constexpr (KW == 2) key[1] = static_cast<uint64_t>(k >> 64);
}
// The same, the table in global memory, key words chosen at run time.
__device__ __forceinline__ void make_key_any(const KeyPlan& kp, const uint64_t* f, int W, uint64_t flags,
                                             uint64_t* key) {
  if (kp.kw == 1)
    make_key<1, 2>(kp, f, W, flags, key);
  else
    make_key<2, 2>(kp, f, W, flags, key);
}

// Production: one thread per spawning attempt.  Each block takes tiles of
// T consecutive attempts of the batch [t_begin, t_end); the parents
// of a tile's first and last attempts bound a short window of the attempt
// prefix sum (n*S (det, space) entries, det-major) in which each thread
// searches its own parent.  The successful attempts of a tile are ranked in
// attempt order (wavefront ballots plus per-wave totals) and written
// contiguously from the tile's first staging slot, with the tile's count in
// tile_cnt; k_pack_tiles then copies the tiles, in order, into the spawned list.
template <int G, bool B, int T>
__global__ __launch_bounds__(kBlock, spawn_waves(G, B)) void k_spawn(const Sys* __restrict__ sdev, int64_t nent, int64_t cap, int64_t t_begin, int64_t t_end,
                                                  const int64_t* __restrict__ att_off,
                                                  const uint64_t* __restrict__ det, const int64_t* __restrict__ pop,
                                                  double tau, uint64_t seed, uint32_t cyc, int64_t bcap,
                                                  uint64_t* __restrict__ st_det, int64_t* __restrict__ st_pop,
                                                  uint16_t* __restrict__ st_ent, int32_t* __restrict__ tile_cnt,
                                                  const int64_t* __restrict__ tile_win,
                                                  const uint8_t* __restrict__ pflags,
                                                  const Sys* __restrict__ sys_arr, const int64_t* __restrict__ iatt,
                                                  const double* __restrict__ itau, const uint32_t* __restrict__ pcyc,
                                                  Stats* __restrict__ st) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->spawn_begin = wall_clock64();
    if (t_begin == 0) st->stamp[kStSpawn] = st->spawn_begin;
  }
  cyc = cycle_of(pcyc, cyc);
  // the system descriptor is read from device memory (scalar loads on use)
  // rather than passed by value: its many table pointers would otherwise sit
  // in scalar registers for the whole kernel and spill into vector lanes
  const Sys& s = *sdev;
  __shared__ int32_t wcount[kBlock / 64];
  // att_off[lo + k] - t0 (clamped below at -1: every such entry starts at or
  // before the tile's first attempt) when the window fits
  __shared__ int32_t watt[kSpawnWin];
  // heat-bath: each thread's nel on-the-fly weights in a column of dynamic LDS
  fqd::HbBuf hb;
  if constexpr (G == fqd::kGenHeatBath) {
    extern __shared__ double hb_lds[];
    hb = fqd::HbBuf{hb_lds + threadIdx.x, kBlock};
  }
  // Renormalised and learned generators decide single vs double on an
  // attempt's first draw: those tiles are processed doubles first and singles
  // last (their code paths differ), results parked in LDS by attempt, so a
  // wavefront seldom runs both paths; successes are still compacted in
  // attempt order.
  constexpr bool kPart = (G == fqd::kGenMolRenorm || G == fqd::kGenLearned) && !B;
  __shared__ int16_t order[kPart ? T : 1];   // processing slot -> attempt in tile
  __shared__ int64_t rpop[kPart ? T : 1];    // results by attempt in tile
  __shared__ int32_t rent[kPart ? T : 1];    // parent entry - lo
  __shared__ int32_t wcs[kBlock / 64];
  uint64_t* rdet = nullptr;                            // [w * T + r], dynamic LDS
  const float* aff_lds = nullptr;  // learned: affinity table then flat row, after rdet
  const float* flat_lds = nullptr;
  if constexpr (kPart) {
    extern __shared__ uint64_t part_lds[];
    rdet = part_lds;
    if constexpr (G == fqd::kGenLearned) {
      float* a = reinterpret_cast<float*>(part_lds + s.W * T);
      const int na = s.nbasis * s.nbasis;
      for (int k = threadIdx.x; k < na + 2 * s.nbasis; k += kBlock)
        a[k] = k < na ? s.mlp_aff[k] : s.mlp_flat[k - na];
      aff_lds = a;
      flat_lds = a + na;
      __syncthreads();
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long below = (1ull << lane) - 1;
  const int64_t ntiles = (t_end - t_begin + T - 1) / T;  // tiles the host sized for
  if (const int64_t tot = att_off[nent]; tot < t_end) t_end = tot;  // the host may pass a bound
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t t0 = t_begin + tile * T;
    if (t0 >= t_end) {  // past the total (block-uniform)
      if (threadIdx.x == 0) tile_cnt[tile] = 0;
      continue;
    }
    const int64_t t1 = (t0 + T < t_end) ? t0 + T : t_end;
    const int tn = static_cast<int>(t1 - t0);
    const int64_t lo = tile_win[2 * tile], hi = tile_win[2 * tile + 1];
    const bool staged = hi - lo < kSpawnWin;
    if (staged)
      for (int64_t k = threadIdx.x; k <= hi - lo; k += kBlock) {
        const int64_t v = att_off[lo + k] - t0;
        watt[k] = static_cast<int32_t>(v < -1 ? -1 : v);
      }
    __syncthreads();
    // one spawning attempt t (tile-relative r): its parent entry e, the
    // spawned population and the child determinant
    auto attempt = [&](int64_t t, int r, int64_t& e, int64_t& nspawn, uint64_t* child) {
      if (staged) {  // last k in [0, hi - lo] with att_off[lo + k] <= t
        int a = 0, b = static_cast<int>(hi - lo);
        while (a < b) {
          const int mid = (a + b + 1) >> 1;
          if (watt[mid] <= r)
            a = mid;
          else
            b = mid - 1;
        }
        e = lo + a;
      } else {
        e = parent_of(att_off, t, lo, hi);
      }
      const int sp = static_cast<int>(e % s.S);
      const int64_t i = e / s.S;
      uint64_t f[FQ_MAX_WORDS];
      load_det(det, cap, s.W, i, f);
      const int64_t parent = pop[sp * cap + i];
      if constexpr (B) {
        // batched instances: the instance's tables, time step, key and attempt
        // numbering.  Attempts are numbered instance by instance, so a wavefront
        // seldom holds two: its instances are taken one after the other, the
        // descriptor in scalar registers
        const int mine = static_cast<int>(f[0] >> kInstShift);
        f[0] &= kOrbMask;
        bool todo = true;
        while (todo) {
          const int inst = __builtin_amdgcn_readfirstlane(mine);
          if (inst == mine) {
            const int64_t trel = t - iatt[inst];
            fqd::PhiloxPre<spawn_pre(G)> rng(seed + static_cast<uint64_t>(inst), static_cast<uint32_t>(trel),
                                             static_cast<uint32_t>(trel >> 32), cyc ^ (fqd::kDrawAttempt << 24));
            nspawn = fqd::spawn_attempt<G>(sys_arr[inst], rng, f, nullptr, parent, itau[inst], child);
            if (nspawn != 0) child[0] |= static_cast<uint64_t>(inst) << kInstShift;
            todo = false;
          }
        }
      } else {
        const uint32_t t_lo = static_cast<uint32_t>(t), t_hi = static_cast<uint32_t>(t >> 32);
        const uint32_t purpose = cyc ^ (fqd::kDrawAttempt << 24);
        using Rng = fqd::PhiloxPre<spawn_pre(G)>;
        // partitioned tiles: the attempt's first block is parked in its result slots
        Rng rng = kPart ? Rng(seed, t_lo, t_hi, purpose, static_cast<uint64_t>(rpop[kPart ? r : 0]), rdet[kPart ? r : 0])
                        : Rng(seed, t_lo, t_hi, purpose);
        const float* wrow = nullptr;
        if constexpr (G == fqd::kGenLearned) {
          const int32_t row = s.mlp_row[i];
          if (row >= 0) wrow = s.mlp_tab + row * s.mlp_ld;
        }
        nspawn = fqd::spawn_attempt<G>(s, rng, f, wrow, parent, tau, child, hb, aff_lds, flat_lds);
        // a core parent's spawn onto the core is the deterministic projection's
        if (s.ndeterm > 0 && nspawn != 0 && (pflags[i] & kCoreFlag) && fqd::core_index(s, child) >= 0) nspawn = 0;
      }
    };
    if constexpr (kPart) {
      // processing order: doubles from the front, singles from the back
      int32_t nd = 0, ns = 0;
      for (int k = 0; k < T / kBlock; ++k) {
        const int r = k * kBlock + threadIdx.x;
        bool single = false;
        if (r < tn) {
          const int64_t t = t0 + r;
          fqd::Philox rng(seed, static_cast<uint32_t>(t), static_cast<uint32_t>(t >> 32),
                          cyc ^ (fqd::kDrawAttempt << 24));
          single = rng.next() < s.psingle;
          // the block stays in the attempt's result slots until the attempt is made
          rpop[r] = static_cast<int64_t>(static_cast<uint64_t>(rng.o1) << 32 | rng.o0);
          rdet[r] = static_cast<uint64_t>(rng.o3) << 32 | rng.o2;
        }
        const unsigned long long bd = __ballot(r < tn && !single), bs = __ballot(r < tn && single);
        if (lane == 0) {
          wcount[wave] = __popcll(bd);
          wcs[wave] = __popcll(bs);
        }
        __syncthreads();
        int32_t pd = nd + __popcll(bd & below), ps = ns + __popcll(bs & below);
        for (int w = 0; w < kBlock / 64; ++w) {
          if (w < wave) {
            pd += wcount[w];
            ps += wcs[w];
          }
          nd += wcount[w];
          ns += wcs[w];
        }
        if (r < tn) order[single ? tn - 1 - ps : pd] = static_cast<int16_t>(r);
        __syncthreads();
      }
      for (int k = 0; k < T / kBlock; ++k) {
        const int q = k * kBlock + threadIdx.x;
        if (q < tn) {
          const int r = order[q];
          int64_t e = 0, nspawn = 0;
          uint64_t child[FQ_MAX_WORDS] = {0, 0};
          attempt(t0 + r, r, e, nspawn, child);
          FQ_FOR_WORDS(w, s.W) rdet[w * T + r] = child[w];
          rpop[r] = nspawn;
          rent[r] = static_cast<int32_t>(e - lo);
        }
      }
      __syncthreads();
    }
    int32_t run = 0;  // successes of this tile so far (all threads hold the same value)
    for (int k = 0; k < T / kBlock; ++k) {
      const int r = k * kBlock + threadIdx.x;
      const bool valid = r < tn;
      int64_t e = 0, nspawn = 0;
      uint64_t child[FQ_MAX_WORDS] = {0, 0};
      if (valid) {
        if constexpr (kPart) {
          nspawn = rpop[r];
          e = lo + rent[r];
          FQ_FOR_WORDS(w, s.W) child[w] = rdet[w * T + r];
        } else {
          attempt(t0 + r, r, e, nspawn, child);
        }
      }
      // rank this round's successes in attempt order (wave ballot + per-wave totals)
      const bool ok = valid && nspawn != 0;
      const unsigned long long bal = __ballot(ok);
      if (lane == 0) wcount[wave] = __popcll(bal);
      __syncthreads();
      int32_t pos = run + __popcll(bal & below);
      int32_t round_total = 0;
      for (int w = 0; w < kBlock / 64; ++w) {
        if (w < wave) pos += wcount[w];
        round_total += wcount[w];
      }
      if (ok) {  // compacted into the tile's region of the staging arrays
        const int64_t u = (t0 - t_begin) + pos;
        FQ_FOR_WORDS(w, s.W) st_det[w * bcap + u] = child[w];
        st_pop[u] = nspawn;
        // the spawning space and the parent's initiator flags (the sort key's flag bits)
        st_ent[u] = static_cast<uint16_t>((e % s.S) | (s.initiator ? (pflags[e / s.S] & kInitFlagMask) << 8 : 0));
      }
      run += round_total;
      __syncthreads();
    }
    if (threadIdx.x == 0) tile_cnt[tile] = run;
    __syncthreads();
  }
}

// Pack each tile's compacted successes into the spawned list in attempt order,
// as sort keys (made here, the binomial table staged in LDS) and payload (the
// population in its space's word, 0 in the other).  A block takes a contiguous
// range of tiles and adds the counts of the tiles before it for its place (at
// most 2048 blocks, so the work grows with the tiles only: 70 us with the packing
// of 2.8e6 entries from the 6e4 tiles of 3e7 determinants).
// first: the cycle's only batch -- the list starts empty and block 0 records
// its length and the attempt total (*ptot; more than tlim >= 0 of them: some
// were not made); else the entries follow those of earlier batches (st->nspawn).
// st_ent holds the spawning space and, from bit 8, the parent's initiator flags.
template <int KW>
__global__ __launch_bounds__(kBlock) void k_pack_tiles(int W, int S, int64_t ntiles, int tile_size,
                                                       const int32_t* __restrict__ tile_cnt,
                                                       const uint64_t* __restrict__ st_det,
                                                       const int64_t* __restrict__ st_pop,
                                                       const uint16_t* __restrict__ st_ent, int64_t bcap,
                                                       int64_t scap, KeyPlan kp, uint64_t* __restrict__ keys,
                                                       int64_t* __restrict__ pay, Stats* __restrict__ st, int first,
                                                       const int64_t* __restrict__ ptot, int64_t tlim) {
  extern __shared__ uint64_t binom_lds[];
  __shared__ int64_t wsh[kBlock / 64];
  if (blockIdx.x == 0 && threadIdx.x == 0) st->spawn_ticks += wall_clock64() - st->spawn_begin;
  if (kp.rank && kp.binom_lds) {  // blocks loop over tiles, so each stages the table once
    const int nw = KW * kp.nbasis * kp.nel;
    for (int k = threadIdx.x; k < nw; k += kBlock) binom_lds[k] = kp.binom[KW == 1 ? 2 * k : k];
  }
  const int64_t per = (ntiles + gridDim.x - 1) / gridDim.x;
  const int64_t tile0 = blockIdx.x * per, tile1 = tile0 + per < ntiles ? tile0 + per : ntiles;
  int64_t base = first ? 0 : st->nspawn;
  {
    const int64_t upto = blockIdx.x == 0 ? ntiles : (tile0 < ntiles ? tile0 : ntiles);
    int64_t x = 0;
#pragma unroll 4
    for (int64_t k = threadIdx.x; k < upto; k += kBlock) x += tile_cnt[k];
    x = block_sum(x, wsh);  // its barriers also publish the table
    if (blockIdx.x == 0) {  // the batch's length
      if (first && threadIdx.x == 0) {
        st->nspawn = x;
        st->total_attempts = *ptot;
        if (tlim >= 0 && *ptot > tlim) st->spawn_overflow = 1;  // attempts past the launch's bound were not made
      }
    } else {
      base += x;
    }
  }
  for (int64_t tile = tile0; tile < tile1; ++tile) {
    const int64_t cnt = tile_cnt[tile];
    for (int64_t j = threadIdx.x; j < cnt; j += kBlock) {
      const int64_t u = tile * tile_size + j;
      const int64_t slot = base + j;
      if (slot >= scap) {
        st->spawn_overflow = 1;
        continue;
      }
      const int e = st_ent[u], sp = e & 0xff;
      uint64_t f[FQ_MAX_WORDS] = {0, 0};
      FQ_FOR_WORDS(w, W) f[w] = st_det[w * bcap + u];
      const int64_t v = st_pop[u];
      for (int q = 0; q < S; ++q) pay[q * scap + slot] = (q == sp) ? v : 0;
      uint64_t k[KW];
      if (kp.binom_lds) {
        KeyPlan lp = kp;
        lp.binom = binom_lds;
        make_key<KW, KW>(lp, f, W, static_cast<uint64_t>(e >> 8), k);
      } else {
        make_key<KW, 2>(kp, f, W, static_cast<uint64_t>(e >> 8), k);
      }
#pragma unroll
      for (int w = 0; w < KW; ++w) keys[w * scap + slot] = k[w];
    }
    base += cnt;
  }
}

// After a batch that is not the cycle's only one: its entries join the length.
__global__ __launch_bounds__(kBlock) void k_add_spawned(const int32_t* __restrict__ tile_cnt, int64_t ntiles,
                                                        const int64_t* __restrict__ ptot, Stats* __restrict__ st) {
  __shared__ int64_t wsh[kBlock / 64];
  int64_t x = 0;
  for (int64_t k = threadIdx.x; k < ntiles; k += kBlock) x += tile_cnt[k];
  x = block_sum(x, wsh);
  if (threadIdx.x == 0) {
    st->nspawn += x;
    st->total_attempts = *ptot;
  }
}

// ---------------------------------------------------------------------------
// Batched instances
// ---------------------------------------------------------------------------
// bound[k] = first position in the sorted list whose instance index is >= k.
__global__ void k_inst_bounds(const uint64_t* __restrict__ w0, int64_t n, int ninst, int shift,
                              int64_t* __restrict__ bound, const int64_t* __restrict__ pn) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k > ninst) return;
  n = list_len(pn, n);
  if (k == ninst) {
    bound[k] = n;
    return;
  }
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (static_cast<int>(w0[mid] >> shift) < k)
      lo = mid + 1;
    else
      hi = mid;
  }
  bound[k] = lo;
}

// k_det_pass for a batched list: each determinant uses its instance's tables,
// time step, shift and key; Philox counters count determinants from the
// instance's first, so an instance follows the same chain as alone.  The
// estimator terms go to per-determinant arrays for per-instance sums.
__global__ __launch_bounds__(kBlock) void k_det_pass_batch(Sys s, const Sys* __restrict__ sys_arr,
                                                           const int64_t* __restrict__ bound,
                                                           const double* __restrict__ ipar, int ninst, int64_t n,
                                                           int64_t cap, const uint64_t* __restrict__ det,
                                                           const int64_t* __restrict__ pop,
                                                           const double* __restrict__ kii,
                                                           int64_t* __restrict__ pop_new, int32_t* __restrict__ nat,
                                                           uint8_t* __restrict__ flags, uint64_t seed, uint32_t cyc,
                                                           double* __restrict__ cterm,
                                                           int64_t* __restrict__ cdeath,
                                                           const int64_t* __restrict__ pn,
                                                           const uint32_t* __restrict__ pcyc,
                                                           int64_t* __restrict__ blk_att, Stats* __restrict__ st) {
  __shared__ int64_t wsh[kBlock / 64];
  clear_stats(st);
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  int64_t att = 0;
  if (i < list_len(pn, n)) {
    cyc = cycle_of(pcyc, cyc);
    uint64_t f[FQ_MAX_WORDS];
    load_det(det, cap, s.W, i, f);
    const int inst = static_cast<int>(f[0] >> kInstShift);
    f[0] &= kOrbMask;
    const Sys& si = sys_arr[inst];
    const int64_t irel = i - bound[inst];
    const double tau = ipar[inst];
    double rp[FQ_MAX_SPACES] = {0.0, 0.0};
    int64_t p[FQ_MAX_SPACES] = {0, 0};
    for (int sp = 0; sp < s.S; ++sp) {
      p[sp] = pop[sp * cap + i];
      rp[sp] = static_cast<double>(p[sp]) / static_cast<double>(s.rf);
    }
    flags[i] = static_cast<uint8_t>(fqd::parent_flag(s, rp));
    const double K = kii[i];
    int64_t ndeath = 0;
    for (int sp = 0; sp < s.S; ++sp) {
      double proj = 0.0, d0 = 0.0;
      fqd::proj_energy_term(si, f, rp[sp], proj, d0);
      cterm[(2 * sp) * cap + i] = proj;
      cterm[(2 * sp + 1) * cap + i] = d0;
      const uint32_t hi = static_cast<uint32_t>(irel >> 32) ^ (static_cast<uint32_t>(sp) << 28);
      const uint64_t key = seed + static_cast<uint64_t>(inst);
      fqd::Philox rng(key, static_cast<uint32_t>(irel), hi, cyc ^ (fqd::kDrawNattempts << 24));
      const int32_t na = fqd::decide_nattempts(rng, rp[sp]);
      nat[i * s.S + sp] = na;
      att += na;
      fqd::Philox rd(key, static_cast<uint32_t>(irel), hi, cyc ^ (fqd::kDrawDeath << 24));
      int64_t q = p[sp];
      const double sh = ipar[ninst + sp * ninst + inst], eo = ipar[(1 + s.S) * ninst + sp * ninst + inst];
      ndeath += fqd::death(rd, tau, K, sh, eo, q);
      pop_new[sp * cap + i] = q;
    }
    cdeath[i] = ndeath;
  } else if (i < n) {  // past the list in a launch sized by a bound: no attempts
    for (int sp = 0; sp < s.S; ++sp) nat[i * s.S + sp] = 0;
  }
  att = block_sum(att, wsh);
  if (threadIdx.x == 0) blk_att[blockIdx.x] = att;
}

// First attempt index of each instance: attempts are numbered over the
// (determinant, space) entries in list order.
__global__ void k_inst_att(int ninst, int S, const int64_t* __restrict__ bound, const int64_t* __restrict__ att_off,
                           int64_t* __restrict__ iatt) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < ninst) iatt[k] = att_off[S * bound[k]];
}

// Per-instance cycle results: projected-energy terms, N_0 and deaths over the
// old list, attempts, spawned entries, occupied determinants and sum |N| over
// the new list.  The floating-point sums repeat the single-instance reduction
// exactly: blocks of 256 determinants counted from the instance's first, each
// reduced by the k_det_pass tree (k_inst_part, one block per such block of
// every instance), then block b added to partial b mod 256 in order and the
// k_finish tree (k_inst_stats, one block per instance), so a batched
// instance reports the same estimators, bit for bit, as it alone.
// Blocks of 256 entries per instance of a list with instance bounds b.
__global__ void k_inst_nblk(int ninst, const int64_t* __restrict__ b, int64_t* __restrict__ cnt) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < ninst) cnt[k] = (b[k + 1] - b[k] + kBlock - 1) / kBlock;
}
// The instance owning global block blk: the last k with off[k] <= blk.
__device__ __forceinline__ int inst_of_block(const int64_t* __restrict__ off, int ninst, int64_t blk) {
  int lo = 0, hi = ninst - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= blk)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}
// One block per 256-entry block of every instance (grid: a bound of their
// number).  Old list (ob, off): the tree sums of the 2S estimator terms and the
// deaths; new list (nbd, noff): sum |N| per space.
__global__ __launch_bounds__(kBlock) void k_inst_part(int ninst, int S, int64_t cap, const int64_t* __restrict__ ob,
                                                      const int64_t* __restrict__ off, const double* __restrict__ cterm,
                                                      const int64_t* __restrict__ cdeath,
                                                      const int64_t* __restrict__ nbd, const int64_t* __restrict__ noff,
                                                      const int64_t* __restrict__ pop, int64_t pb,
                                                      double* __restrict__ part_d, int64_t* __restrict__ part_i) {
  __shared__ double shd[2 * FQ_MAX_SPACES][kBlock];
  __shared__ int64_t wsh[kBlock / 64];
  const int tid = threadIdx.x;
  const int64_t blk = blockIdx.x;
  const int64_t nold = off[ninst], nnew = noff[ninst];
  if (blk < nold) {
    const int k = inst_of_block(off, ninst, blk);
    const int64_t i = ob[k] + (blk - off[k]) * kBlock + tid;
    const bool in = i < ob[k + 1];
    for (int q = 0; q < 2 * FQ_MAX_SPACES; ++q) shd[q][tid] = (q < 2 * S && in) ? cterm[q * cap + i] : 0.0;
    __syncthreads();
    for (int h = kBlock / 2; h > 0; h >>= 1) {
      if (tid < h)
        for (int q = 0; q < 2 * FQ_MAX_SPACES; ++q) shd[q][tid] += shd[q][tid + h];
      __syncthreads();
    }
    const int64_t d = block_sum(in ? cdeath[i] : 0, wsh);
    if (tid == 0) {
      for (int q = 0; q < 2 * S; ++q) part_d[q * pb + blk] = shd[q][0];
      part_i[blk] = d;
    }
  }
  if (blk < nnew) {
    const int k = inst_of_block(noff, ninst, blk);
    const int64_t i = nbd[k] + (blk - noff[k]) * kBlock + tid;
    const bool in = i < nbd[k + 1];
    for (int sp = 0; sp < S; ++sp) {
      int64_t p = in ? pop[sp * cap + i] : 0;
      p = p < 0 ? -p : p;
      const int64_t t = block_sum(p, wsh);
      if (tid == 0) part_i[(1 + sp) * pb + blk] = t;
    }
  }
}
// One block per instance: its block partials added in k_finish's
// order, then the outputs.
__global__ __launch_bounds__(kBlock) void k_inst_stats(int ninst, int S, const int64_t* __restrict__ ob,
                                                       const int64_t* __restrict__ nbd, const int64_t* __restrict__ sb,
                                                       const int64_t* __restrict__ off,
                                                       const int64_t* __restrict__ noff, int64_t pb,
                                                       const double* __restrict__ part_d,
                                                       const int64_t* __restrict__ part_i,
                                                       const int64_t* __restrict__ att_off,
                                                       double* __restrict__ out_d, int64_t* __restrict__ out_i) {
  __shared__ double shd[2 * FQ_MAX_SPACES][kBlock];
  __shared__ int64_t shi[1 + FQ_MAX_SPACES][kBlock];
  const int k = blockIdx.x, tid = threadIdx.x;
  const int nq = 2 * S;
  double acc[2 * FQ_MAX_SPACES] = {0.0, 0.0, 0.0, 0.0};
  int64_t acci[1 + FQ_MAX_SPACES] = {0, 0, 0};
  for (int64_t vb = tid; vb < off[k + 1] - off[k]; vb += kBlock) {
    for (int q = 0; q < nq; ++q) acc[q] = acc[q] + part_d[q * pb + off[k] + vb];
    acci[0] += part_i[off[k] + vb];
  }
  for (int64_t vb = tid; vb < noff[k + 1] - noff[k]; vb += kBlock)
    for (int sp = 0; sp < S; ++sp) acci[1 + sp] += part_i[(1 + sp) * pb + noff[k] + vb];
  for (int q = 0; q < 2 * FQ_MAX_SPACES; ++q) shd[q][tid] = acc[q];
  for (int q = 0; q < 1 + FQ_MAX_SPACES; ++q) shi[q][tid] = acci[q];
  __syncthreads();
  for (int h = kBlock / 2; h > 0; h >>= 1) {
    if (tid < h) {
      for (int q = 0; q < 2 * FQ_MAX_SPACES; ++q) shd[q][tid] += shd[q][tid + h];
      for (int q = 0; q < 1 + FQ_MAX_SPACES; ++q) shi[q][tid] += shi[q][tid + h];
    }
    __syncthreads();
  }
  if (tid == 0) {
    const int64_t a = ob[k], b = ob[k + 1];
    for (int q = 0; q < nq; ++q) out_d[k * nq + q] = shd[q][0];
    int64_t* o = out_i + k * (4 + S);
    o[0] = shi[0][0];                          // deaths
    o[1] = att_off[S * b] - att_off[S * a];    // attempts
    o[2] = sb[k + 1] - sb[k];                  // spawned entries
    o[3] = nbd[k + 1] - nbd[k];                // occupied determinants
    for (int sp = 0; sp < S; ++sp) o[4 + sp] = shi[1 + sp][0];
  }
}

// Replay: the whole spawning/death loop on one thread, in reference order.
// determ_proj_combined_annihil (src/semi_stoch.F90:897-975) for one core
// determinant and space: -tau (sum_j H_ij v_j + (E_old * 0 - S) v_i), the
// row summed in column order (csrpgemv_single_row, lib/local/csr.f90:206-235);
// 0 is rho - w, the quasi-Newton weight difference without quasi-Newton.
__device__ __forceinline__ double determ_combined(const DetermDev& dd, int S, int64_t row, int sp, double tau,
                                                  double shift, double eold) {
  double out = 0.0;
  for (int64_t k = dd.row[row]; k < dd.row[row + 1]; ++k) out = out + dd.mat[k] * dd.vec[dd.col[k] * S + sp];
  return -tau * (out + (eold * (1.0 - 1.0) - 1.0 * shift) * dd.vec[row * S + sp]);
}
// determ_proj_separate_annihil (src/semi_stoch.F90:1009-1094): the shift term
// -(tau (E_old * 0 - S)) v_i, then (-tau T_ik) v_k added over the stored
// transpose's row i in order, as the reference's transposed product
// (csrpgemv, lib/local/csr.f90:148-204) accumulates element i.
__device__ __forceinline__ double determ_separate(const DetermDev& dd, int S, int64_t row, int sp, double tau,
                                                  double shift, double eold) {
  const double a = -1.0 * tau;
  double y = -(tau * (eold * (1.0 - 1.0) - shift * 1.0)) * dd.vec[row * S + sp];
  for (int64_t k = dd.row[row]; k < dd.row[row + 1]; ++k) y = y + a * dd.mat[k] * dd.vec[dd.col[k] * S + sp];
  return y;
}

// Semi-stochastic core (dd.nd > 0, set_determ_info and the determ_parent
// branches of src/fciqmc.f90:330-372): a core parent is an initiator, its
// spawns onto the core are cancelled and its death is left to the
// deterministic projection, which follows the loop (determ_projection,
// src/semi_stoch.F90:859-1094) with one rounding draw per core determinant
// and space.
__global__ void k_replay_walk(Sys s, int64_t n, int64_t cap, const uint64_t* __restrict__ det,
                              const int64_t* __restrict__ pop, const double* __restrict__ kii,
                              int64_t* __restrict__ pop_new, double tau, double sh0, double sh1, double e0,
                              double e1, const double* __restrict__ rbuf, int64_t rpos, int64_t rend, int64_t scap,
                              uint64_t* __restrict__ sdet, int64_t* __restrict__ srec, Stats* __restrict__ st,
                              DetermDev dd) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  stamp(st, kStBegin);
  fqd::ReplayRng rng{rbuf, rpos, rend, false};
  double proj[FQ_MAX_SPACES] = {0.0, 0.0}, d0[FQ_MAX_SPACES] = {0.0, 0.0};
  int64_t ndeath = 0, nspawn_total = 0, attempts = 0;
  bool overflow = false;
  for (int64_t i = 0; i < n && !rng.failed; ++i) {
    uint64_t f[FQ_MAX_WORDS];
    load_det(det, cap, s.W, i, f);
    double rp[FQ_MAX_SPACES] = {0.0, 0.0};
    int64_t p[FQ_MAX_SPACES] = {0, 0};
    for (int sp = 0; sp < s.S; ++sp) {
      p[sp] = pop[sp * cap + i];
      rp[sp] = static_cast<double>(p[sp]) / static_cast<double>(s.rf);
    }
    const int64_t ci = dd.nd > 0 ? fqd::core_index(s, f) : -1;
    if (ci >= 0) {
      for (int sp = 0; sp < s.S; ++sp) dd.vec[ci * s.S + sp] = rp[sp];
      dd.pos[ci] = i;
    }
    const int64_t flag = ci >= 0 ? 0 : fqd::parent_flag(s, rp);
    for (int sp = 0; sp < s.S; ++sp) {
      fqd::proj_energy_term(s, f, rp[sp], proj[sp], d0[sp]);
      const int nat = fqd::decide_nattempts(rng, rp[sp]);
      attempts += nat;
      for (int a = 0; a < nat && !rng.failed; ++a) {
        uint64_t child[FQ_MAX_WORDS] = {0, 0};
        int64_t ns = fqd::spawn_attempt(s, rng, f, nullptr, p[sp], tau, child);
        if (ns != 0 && ci >= 0 && fqd::core_index(s, child) >= 0) ns = 0;
        if (ns != 0) {
          if (nspawn_total + 1 > scap) {
            overflow = true;
          } else {
            const int64_t slot = nspawn_total++;
            FQ_FOR_WORDS(w, s.W) sdet[w * scap + slot] = child[w];
            int64_t* rec = srec + slot * rec_stride(s.S);
            for (int q = 0; q < s.S; ++q) rec[q] = (q == sp) ? ns : 0;
            rec[s.S] = s.initiator ? flag : 0;
          }
        }
      }
      int64_t q = p[sp];
      if (ci < 0) ndeath += fqd::death(rng, tau, kii[i], sp == 0 ? sh0 : sh1, sp == 0 ? e0 : e1, q);
      p[sp] = q;
      pop_new[sp * cap + i] = q;
    }
  }
  if (dd.nd > 0 && !rng.failed) {
    const double sh[FQ_MAX_SPACES] = {sh0, sh1}, eo[FQ_MAX_SPACES] = {e0, e1};
    if (!dd.separate) {
      for (int64_t row = 0; row < dd.nd && !rng.failed; ++row)
        for (int sp = 0; sp < s.S; ++sp) {
          const int64_t ns = fqd::stoch_encode(rng, determ_combined(dd, s.S, row, sp, tau, sh[sp], eo[sp]), s.rf);
          if (nspawn_total + 1 > scap) {
            overflow = true;
            continue;
          }
          const int64_t slot = nspawn_total++;
          FQ_FOR_WORDS(w, s.W) sdet[w * scap + slot] = s.determ[w * dd.nd + row];
          int64_t* rec = srec + slot * rec_stride(s.S);
          for (int q = 0; q < s.S; ++q) rec[q] = (q == sp) ? ns : 0;
          rec[s.S] = 0;
        }
    } else {
      // every row's projection first, then the rounding draws row by row
      for (int64_t row = 0; row < dd.nd; ++row)
        for (int sp = 0; sp < s.S; ++sp)
          dd.vec[(dd.nd + row) * s.S + sp] = determ_separate(dd, s.S, row, sp, tau, sh[sp], eo[sp]);
      for (int64_t row = 0; row < dd.nd && !rng.failed; ++row)
        for (int sp = 0; sp < s.S; ++sp) {
          const int64_t ns = fqd::stoch_encode(rng, dd.vec[(dd.nd + row) * s.S + sp], s.rf);
          pop_new[sp * cap + dd.pos[row]] += ns;
        }
    }
  }
  for (int sp = 0; sp < FQ_MAX_SPACES; ++sp) {
    st->proj[sp] = proj[sp];
    st->d0[sp] = d0[sp];
  }
  st->ndeath = ndeath;
  st->nspawn = nspawn_total;
  st->spawn_overflow = overflow ? 1 : 0;
  st->total_attempts = attempts;
  st->rng_pos = rng.pos;
  st->rng_failed = rng.failed ? 1 : 0;
  stamp(st, kStScan);
}

// ---------------------------------------------------------------------------
// Kernels: sorting
// ---------------------------------------------------------------------------
// Unsigned multi-word comparison, last word most significant (bit_str_cmp).
__device__ __forceinline__ int key_cmp(const uint64_t* keys, int64_t stride, int W, int64_t a, int64_t b) {
  for (int w = W - 1; w >= 0; --w) {
    const uint64_t x = keys[w * stride + a], y = keys[w * stride + b];
    if (x < y) return -1;
    if (x > y) return 1;
  }
  return 0;
}

// Sort passes use DB-bit digits (8 or 9; 1 << DB buckets) of the key's value
// field: the host mixes the two widths to cover it in the fewest passes
// (34 bits: 9+9+8+8).  Digit of a KW-word key starting at bit `shift`.
template <int KW>
__device__ __forceinline__ uint32_t key_digit(const uint64_t* k, int shift, uint32_t mask) {
  if constexpr (KW == 1) {
    return static_cast<uint32_t>(k[0] >> shift) & mask;
  } else {
    const uint64_t x = shift >= 64 ? (k[1] >> (shift - 64))
                       : shift == 0 ? k[0]
                                    : ((k[0] >> shift) | (k[1] << (64 - shift)));
    return static_cast<uint32_t>(x) & mask;
  }
}

// Lanes of the wavefront holding the same DB-bit digit as this lane (among
// the `valid` ones): DB ballots.
template <int DB>
__device__ __forceinline__ unsigned long long match_digit(uint32_t d, bool valid) {
  unsigned long long peers = __ballot(valid);
#pragma unroll
  for (int b = 0; b < DB; ++b) {
    const bool bit = (d >> b) & 1;
    const unsigned long long m = __ballot(bit);
    peers &= bit ? m : ~m;
  }
  return peers;
}

// Exclusive scan of x over the block (every thread receives its prefix);
// tot receives the block total.
__device__ __forceinline__ uint32_t block_exclusive_u32(uint32_t x, uint32_t* wsh, uint32_t& tot) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t inc = x;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(inc, d, 64);
    if (lane >= d) inc += y;
  }
  if (lane == 63) wsh[wave] = inc;
  __syncthreads();
  uint32_t pre = 0;
  tot = 0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) {
    pre += w < wave ? wsh[w] : 0;
    tot += wsh[w];
  }
  __syncthreads();
  return pre + inc - x;
}

// Radix pass, reduce-then-scan over a fixed grid: block b owns the sort tiles
// [b * tpb, (b + 1) * tpb) (tiles of kBlock * sort_items keys; tpb from the
// list length on the device and the grid, so the host need not know the
// length, only a bound of it).  k_pass_count writes the
// block's digit counts (adds in LDS: the counts need no order, and ranking the
// digits by ballots took 26 and 23 us for 4.3e6 keys against 13 and 12 for the low
// 9-bit and the high 8-bit digits) digit-major, cnt[d * nblk + b]; their exclusive scan
// gives every block the global start of each digit's keys from its range, and
// k_pass_scatter walks its tiles in order, ranks each tile's keys by digit in
// input order (stable), and writes keys and payload (S population words) to
// their sorted positions.  No block waits on another.
template <int KW, int S, int DB, int R>
__global__ __launch_bounds__(kBlock) void k_pass_count(const uint64_t* __restrict__ keys,
                                                       const int64_t* __restrict__ pn, int64_t nb, int64_t stride,
                                                       int shift, int64_t* __restrict__ cnt,
                                                       Stats* __restrict__ st) {
  constexpr int NB = 1 << DB, T = kBlock * R, NW = kBlock / 64;
  __shared__ uint32_t h[NW][NB];  // a histogram per wavefront: equal digits within one only serialise its own adds
  if (st) stamp(st, kStSort);  // the first pass
  for (int d = threadIdx.x; d < NW * NB; d += kBlock) (&h[0][0])[d] = 0;
  __syncthreads();
  const int64_t n = list_len(pn, nb);
  const int64_t tpb = ((n + T - 1) / T + gridDim.x - 1) / gridDim.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t lo = static_cast<int64_t>(blockIdx.x) * tpb * T;
  const int64_t hi = lo + tpb * T < n ? lo + tpb * T : n;
  for (int64_t base = lo; base < hi; base += T) {
    uint32_t d[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {  // every load of the tile in flight before the adds
      const int64_t i = base + r * kBlock + threadIdx.x;
      uint64_t k[KW];
#pragma unroll
      for (int w = 0; w < KW; ++w) k[w] = i < hi ? keys[w * stride + i] : 0;
      d[r] = key_digit<KW>(k, shift, NB - 1);
    }
    // the first lane's digit is added once for all lanes that hold it (later
    // passes see long stretches of one digit), the others one by one
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bool valid = base + r * kBlock + threadIdx.x < hi;
      const uint32_t d0 = __builtin_amdgcn_readfirstlane(d[r]);
      const unsigned long long same = __ballot(valid && d[r] == d0);
      if (lane == 0 && same) atomicAdd(&h[wave][d0], static_cast<uint32_t>(__popcll(same)));
      if (valid && d[r] != d0) atomicAdd(&h[wave][d[r]], 1u);
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < NB; d += kBlock) {
    uint32_t c = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) c += h[w][d];
    cnt[static_cast<int64_t>(d) * gridDim.x + blockIdx.x] = c;
  }
}

// Per digit d (one block each, nb <= kSortBlocks block counts in its row):
// the row's exclusive prefix, in place, and the digit total in tot[d].
__global__ __launch_bounds__(kSortBlocks) void k_pass_rowscan(int nb, int64_t* __restrict__ cnt,
                                                              int64_t* __restrict__ tot) {
  __shared__ int64_t wsh[kSortBlocks / 64];
  const int d = blockIdx.x, b = threadIdx.x, lane = b & 63, wave = b >> 6;
  const int64_t v = b < nb ? cnt[static_cast<int64_t>(d) * nb + b] : 0;
  const int64_t x = wave_inclusive_scan(v, lane);
  if (lane == 63) wsh[wave] = x;
  __syncthreads();
  int64_t pre = 0, t = 0;
#pragma unroll
  for (int w = 0; w < kSortBlocks / 64; ++w) {
    pre += w < wave ? wsh[w] : 0;
    t += wsh[w];
  }
  if (b < nb) cnt[static_cast<int64_t>(d) * nb + b] = pre + x - v;
  if (b == 0) tot[d] = t;
}

template <int KW, int S, int DB, int R>
__global__ __launch_bounds__(kBlock) void k_pass_scatter(const uint64_t* __restrict__ kin,
                                                         const int64_t* __restrict__ pin, uint64_t* __restrict__ kout,
                                                         int64_t* __restrict__ pout, const int64_t* __restrict__ pn,
                                                         int64_t nb, int64_t stride, int shift,
                                                         const int64_t* __restrict__ off,
                                                         const int64_t* __restrict__ dtot) {
  constexpr int NB = 1 << DB, T = kBlock * R, NW = kBlock / 64;
  const int64_t n = list_len(pn, nb);
  const int64_t tpb = ((n + T - 1) / T + gridDim.x - 1) / gridDim.x;
  constexpr uint32_t MASK = NB - 1;
  __shared__ uint64_t sk[KW][T];
  __shared__ int64_t sp[S][T];
  __shared__ uint32_t wc[NW][NB];  // per-wave running digit counts, then per-wave exclusive prefixes
  __shared__ uint32_t toff[NB];    // tile-local start of each digit
  __shared__ int64_t run[NB];      // global position of the next key of each digit from this block
  __shared__ uint32_t wsh[NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  {
    // digit starts: exclusive scan of the digit totals (every block), plus
    // the keys of this digit in the blocks before this one
    constexpr int DPT = NB / kBlock;
    uint32_t t[DPT], sum = 0;
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
      t[j] = static_cast<uint32_t>(dtot[tid * DPT + j]);
      sum += t[j];
    }
    uint32_t all;
    uint32_t st = block_exclusive_u32(sum, wsh, all);
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
      const int d = tid * DPT + j;
      run[d] = static_cast<int64_t>(st) + off[static_cast<int64_t>(d) * gridDim.x + blockIdx.x];
      st += t[j];
    }
  }
  const int64_t lo = static_cast<int64_t>(blockIdx.x) * tpb * T;
  const int64_t hi = lo + tpb * T < n ? lo + tpb * T : n;
  for (int64_t base = lo; base < hi; base += T) {
    for (int k = tid; k < NW * NB; k += kBlock) (&wc[0][0])[k] = 0;
    __syncthreads();
    // wavefront w ranks keys [base + w*64*R, base + (w+1)*64*R) round by round
    const int64_t wbase = base + static_cast<int64_t>(wave) * 64 * R;
    uint64_t key[R][KW];
    int64_t pay[R][S];
    uint32_t dig[R], rnk[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t i = wbase + r * 64 + lane;
      const bool v = i < hi;
#pragma unroll
      for (int w = 0; w < KW; ++w) key[r][w] = v ? kin[w * stride + i] : 0;
#pragma unroll
      for (int q = 0; q < S; ++q) pay[r][q] = v ? pin[q * stride + i] : 0;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bool valid = wbase + r * 64 + lane < hi;
      const uint32_t d = key_digit<KW>(key[r], shift, MASK);
      dig[r] = d;
      const unsigned long long peers = match_digit<DB>(d, valid);
      const uint32_t below = static_cast<uint32_t>(__popcll(peers & ((1ull << lane) - 1)));
      const uint32_t old = valid ? wc[wave][d] : 0;
      __builtin_amdgcn_wave_barrier();
      if (valid && below == 0) wc[wave][d] = old + static_cast<uint32_t>(__popcll(peers));
      __builtin_amdgcn_wave_barrier();
      rnk[r] = old + below;
    }
    __syncthreads();
    // tile digit counts (wc becomes the waves' exclusive prefixes per digit)
    constexpr int DPT = NB / kBlock;
    uint32_t cnt[DPT], tsum = 0;
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
      const int d = tid * DPT + j;
      uint32_t c = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const uint32_t x = wc[w][d];
        wc[w][d] = c;
        c += x;
      }
      cnt[j] = c;
      tsum += c;
    }
    uint32_t ttot;
    uint32_t to = block_exclusive_u32(tsum, wsh, ttot);
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
      toff[tid * DPT + j] = to;
      to += cnt[j];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (wbase + r * 64 + lane < hi) {
        const uint32_t d = dig[r];
        const uint32_t pos = toff[d] + wc[wave][d] + rnk[r];
#pragma unroll
        for (int w = 0; w < KW; ++w) sk[w][pos] = key[r][w];
#pragma unroll
        for (int q = 0; q < S; ++q) sp[q][pos] = pay[r][q];
      }
    }
    __syncthreads();
    const int tn = static_cast<int>(hi - base < T ? hi - base : T);
    for (int p = tid; p < tn; p += kBlock) {
      uint64_t k[KW];
#pragma unroll
      for (int w = 0; w < KW; ++w) k[w] = sk[w][p];
      const uint32_t d = key_digit<KW>(k, shift, MASK);
      const int64_t g = run[d] + (p - static_cast<int>(toff[d]));
#pragma unroll
      for (int w = 0; w < KW; ++w) kout[w * stride + g] = k[w];
#pragma unroll
      for (int q = 0; q < S; ++q) pout[q * stride + g] = sp[q][p];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < DPT; ++j) run[tid * DPT + j] += cnt[j];
    // (the next tile's first barrier orders these updates before their use)
  }
}

// A short spawned list sorted by one block in LDS: (value, index) packed in one
// word per entry, idx_bits of index, stable LSD passes of 9-bit digits over the
// value; keys and payload are then gathered by index.  Wavefront w keeps a
// contiguous 1/16 of the entries, 64 at a time, in registers between the passes.
// One launch for the three per digit of the passes over memory, which for short
// lists are launch after launch of 3-11 us: 3800 entries of 34-bit values take
// 39 us instead of 76, 150 entries of 18 bits 10 instead of 29.  A pass costs
// 2.4 us and 1.9 more for every 1024 entries past the first, against ~20 for a
// pass over memory: 8192 entries are where the two are still clear of each other.
// st->sorted receives the length; a list longer than limit (the host may have
// gone by the last cycle's length) is left alone and st->resort set.
constexpr int kSmallSort = 8192, kSmallSortBlock = 1024, kSmallSortBits = 9;
template <int S>
__global__ __launch_bounds__(kSmallSortBlock) void k_sort_small(const uint64_t* __restrict__ kin,
                                                                const int64_t* __restrict__ pin,
                                                                uint64_t* __restrict__ kout,
                                                                int64_t* __restrict__ pout,
                                                                const int64_t* __restrict__ pn, int64_t nb,
                                                                int64_t stride, int fb, int vb, int idx_bits,
                                                                int limit, Stats* __restrict__ st) {
  constexpr int NB = 1 << kSmallSortBits, NW = kSmallSortBlock / 64, R = kSmallSort / kSmallSortBlock;
  __shared__ uint64_t sk[kSmallSort];
  __shared__ uint16_t wc[NW][NB];  // per-wave running digit counts, then the first place of each wave's keys
  __shared__ uint32_t wsh[NW];
  stamp(st, kStSort);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t len = list_len(pn, nb);
  if (len > limit) {  // block-uniform
    if (tid == 0) st->resort = 1;
    return;
  }
  const int n = static_cast<int>(len);
  const int rounds = (n + kSmallSortBlock - 1) / kSmallSortBlock, e0 = wave * rounds * 64 + lane;
  const uint64_t imask = (uint64_t{1} << idx_bits) - 1;
  uint64_t key[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int e = e0 + r * 64;
    key[r] = r < rounds && e < n ? ((kin[e] >> fb) << idx_bits) | static_cast<uint64_t>(e) : 0;
  }
  for (int shift = idx_bits; shift < idx_bits + vb; shift += kSmallSortBits) {
    for (int k = tid; k < NW * NB / 2; k += kSmallSortBlock) reinterpret_cast<uint32_t*>(&wc[0][0])[k] = 0;
    __syncthreads();  // also: the previous pass's reads of sk are done
    // the ballots of all rounds first: only the counts form a chain from round to round
    unsigned long long peers[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (r < rounds)  // block-uniform
        peers[r] = match_digit<kSmallSortBits>(static_cast<uint32_t>(key[r] >> shift) & (NB - 1), e0 + r * 64 < n);
    uint16_t rank[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (r < rounds) {
        const bool valid = e0 + r * 64 < n;
        const uint32_t d = static_cast<uint32_t>(key[r] >> shift) & (NB - 1);
        const uint32_t below = static_cast<uint32_t>(__popcll(peers[r] & ((1ull << lane) - 1)));
        const uint32_t old = valid ? wc[wave][d] : 0;
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0) wc[wave][d] = static_cast<uint16_t>(old + __popcll(peers[r]));
        __builtin_amdgcn_wave_barrier();
        rank[r] = static_cast<uint16_t>(old + below);
      }
    __syncthreads();
    // thread d: digit d's keys in each wave, then the digits before d
    uint32_t x[NW], c = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) x[w] = wc[w][tid & (NB - 1)];
#pragma unroll
    for (int w = 0; w < NW; ++w) c += x[w];
    if (tid >= NB) c = 0;
    uint32_t inc = c;
#pragma unroll
    for (int h = 1; h < 64; h <<= 1) {
      const uint32_t y = __shfl_up(inc, h, 64);
      if (lane >= h) inc += y;
    }
    if (lane == 63) wsh[wave] = inc;
    __syncthreads();
    uint32_t before = inc - c;
#pragma unroll
    for (int w = 0; w < NB / 64; ++w) before += w < wave ? wsh[w] : 0;
    if (tid < NB) {
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        wc[w][tid] = static_cast<uint16_t>(before);
        before += x[w];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r >= rounds) break;
      if (e0 + r * 64 < n) sk[wc[wave][static_cast<uint32_t>(key[r] >> shift) & (NB - 1)] + rank[r]] = key[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r >= rounds) break;
      if (e0 + r * 64 < n) key[r] = sk[e0 + r * 64];
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= rounds) break;
    const int e = e0 + r * 64;
    if (e < n) {
      const int64_t i = static_cast<int64_t>(key[r] & imask);
      kout[e] = kin[i];
#pragma unroll
      for (int q = 0; q < S; ++q) pout[q * stride + e] = pin[q * stride + i];
    }
  }
  if (tid == 0) st->sorted = n;
}

// Sort keys and payload from the spawned list (determinant words, records of
// populations and flag): entry i gets those of entry perm[i] (perm may be
// null: the identity).
__global__ void k_make_keys(KeyPlan kp, int S, const uint64_t* __restrict__ sdet, const int64_t* __restrict__ srec,
                            int W, int64_t ns, int64_t scap, const uint32_t* __restrict__ perm,
                            uint64_t* __restrict__ keys, int64_t* __restrict__ pay) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= ns) return;
  const int64_t src = perm ? static_cast<int64_t>(perm[i]) : i;
  uint64_t f[FQ_MAX_WORDS] = {0, 0};
  FQ_FOR_WORDS(w, W) f[w] = sdet[w * scap + src];
  const int64_t* rec = srec + src * rec_stride(S);
  uint64_t k[2];
  make_key_any(kp, f, W, static_cast<uint64_t>(rec[S]), k);
  for (int w = 0; w < kp.kw; ++w) keys[w * scap + i] = k[w];
  for (int q = 0; q < S; ++q) pay[q * scap + i] = rec[q];
}

// Replay: the reference's quicksort (src/sort.f90:213-396) on an index array,
// one thread; comparisons read the spawned bit strings.
__global__ void k_replay_qsort(const uint64_t* __restrict__ sdet, int64_t ns, int W, int64_t scap,
                               uint32_t* __restrict__ idx, Stats* __restrict__ st) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  stamp(st, kStSort);
  for (int64_t i = 0; i < ns; ++i) idx[i] = static_cast<uint32_t>(i);
  auto gt = [&](uint32_t a, uint32_t b) { return key_cmp(sdet, scap, W, a, b) > 0; };
  auto ge = [&](uint32_t a, uint32_t b) { return key_cmp(sdet, scap, W, a, b) >= 0; };
  // 1-based view of idx
  auto L = [&](int64_t k) -> uint32_t& { return idx[k - 1]; };
  int64_t stack_lo[64], stack_hi[64];
  int nstack = 0;
  int64_t lo = 1, hi = ns;
  while (true) {
    if (hi - lo < 7) {
      for (int64_t j = lo + 1; j <= hi; ++j) {
        const uint32_t tmp = L(j);
        int64_t i;
        for (i = j - 1; i >= 1; --i) {
          if (ge(tmp, L(i))) break;
          L(i + 1) = L(i);
        }
        L(i + 1) = tmp;
      }
      if (nstack == 0) break;
      hi = stack_hi[nstack - 1];
      lo = stack_lo[nstack - 1];
      --nstack;
    } else {
      const int64_t pivot = (lo + hi) / 2;
      uint32_t t = L(pivot);
      L(pivot) = L(lo + 1);
      L(lo + 1) = t;
      if (gt(L(lo), L(hi))) {
        t = L(lo);
        L(lo) = L(hi);
        L(hi) = t;
      }
      if (gt(L(lo + 1), L(hi))) {
        t = L(lo + 1);
        L(lo + 1) = L(hi);
        L(hi) = t;
      }
      if (gt(L(lo), L(lo + 1))) {
        t = L(lo);
        L(lo) = L(lo + 1);
        L(lo + 1) = t;
      }
      int64_t i = lo + 1, j = hi;
      const uint32_t piv = L(lo + 1);
      while (true) {
        ++i;
        while (gt(piv, L(i))) ++i;
        --j;
        while (gt(L(j), piv)) --j;
        if (j < i) break;
        t = L(i);
        L(i) = L(j);
        L(j) = t;
      }
      L(lo + 1) = L(j);
      L(j) = piv;
      ++nstack;
      if (hi - i + 1 >= j - lo) {
        stack_hi[nstack - 1] = hi;
        stack_lo[nstack - 1] = i;
        hi = j - 1;
      } else {
        stack_hi[nstack - 1] = j - 1;
        stack_lo[nstack - 1] = lo;
        lo = i;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Kernels: self-annihilation of the sorted spawned list
// ---------------------------------------------------------------------------
// Equal determinants are adjacent in the sorted keys (equal value fields).
template <int KW>
__device__ __forceinline__ bool same_value(const uint64_t* a, const uint64_t* b, int low_bits) {
  if constexpr (KW == 1) return (a[0] >> low_bits) == (b[0] >> low_bits);
  else return a[1] == b[1] && (a[0] >> low_bits) == (b[0] >> low_bits);
}

// The determinant of a combinatorial rank, in one pass down the orbitals from
// the highest occupied one (a binary search; 7 steps cover 128 orbitals): at
// orbital p with i electrons left, p is occupied iff C(p, i) <= the remaining
// rank, which then drops by C(p, i).  One table read per orbital and no
// nested loop keep a wavefront's lanes together (stepping electron by
// electron lets each lane's gaps serialise the wavefront).  binom: the table
// (in LDS when staged); sat: it holds C(p, i) saturated at 2^64 - 1, one word
// each (ranks below 2^64), instead of (low, high) pairs.
template <bool WIDE>
__device__ __forceinline__ void unrank(const KeyPlan& kp, const uint64_t* __restrict__ binom, bool sat,
                                       unsigned __int128 rank, uint64_t* f) {
  using V = typename std::conditional<WIDE, unsigned __int128, uint64_t>::type;
  const int nel = kp.nel;
  auto C = [&](int p, int i) -> V {
    if constexpr (WIDE) {
      const uint64_t* t = binom + 2 * (p * nel + (i - 1));
      return (static_cast<unsigned __int128>(t[1]) << 64) | t[0];
    } else {
      if (sat) return binom[p * nel + (i - 1)];
      const uint64_t* t = binom + 2 * (p * nel + (i - 1));
      return t[1] ? ~uint64_t{0} : t[0];  // above the 64-bit ranks: larger than any of them
    }
  };
  V r = static_cast<V>(rank);
  int lo = nel - 1, hi = kp.nbasis - 1;
#pragma unroll
  for (int step = 0; step < 7; ++step) {
    const int mid = (lo + hi + 1) >> 1;
    const bool ok = C(mid, nel) <= r;
    const bool live = lo < hi;
    lo = live && ok ? mid : lo;
    hi = live && !ok ? mid - 1 : hi;
  }
  uint64_t f0 = 0, f1 = 0;
  int i = nel;
  for (int p = lo; i > 0 && p >= 0; --p) {
    const V c = C(p, i);
    if (c <= r) {
      if (p < 64)
        f0 |= uint64_t{1} << p;
      else
        f1 |= uint64_t{1} << (p - 64);
      r -= c;
      --i;
    }
  }
  f[0] = f0;
  f[1] = f1;
}

// One sorted entry's share of its run's sums in annihilate_spawn_t_initiator
// (src/spawn_data.F90:937-1101), per space: c[sp] the population; c[S + sp]
// the population if it was spawned from an initiator (flag clear), else 0;
// c[2S + sp] for a flagged (non-initiator) spawn its event count, the sign of
// the population (0 for 0) -- except a run's first entry, which counts the
// sign of its population's low 32 bits read as a default integer.  Every sum
// is additive, so a run's totals may be formed in any grouping.
template <int S>
__device__ __forceinline__ void entry_share(int64_t flags, const int64_t* pop, bool head, int64_t* c) {
#pragma unroll
  for (int sp = 0; sp < S; ++sp) {
    const int64_t v = pop[sp];
    const bool fl = (flags >> sp) & 1;
    c[sp] = v;
    c[S + sp] = fl ? 0 : v;
    int64_t ev = 0;
    if (fl) {
      if (head) {
        const int32_t v32 = static_cast<int32_t>(static_cast<uint32_t>(static_cast<uint64_t>(v) & 0xffffffffULL));
        ev = v32 >= 0 ? 1 : -1;
      } else {
        ev = v < 0 ? -1 : (v > 0 ? 1 : 0);
      }
    }
    c[2 * S + sp] = ev;
  }
}

// Sort values: one 64-bit word, or two as a 128-bit integer.
template <int KW>
using SortValue = typename std::conditional<KW == 1, uint64_t, unsigned __int128>::type;
template <int KW>
__device__ __forceinline__ SortValue<KW> load_value(const uint64_t* __restrict__ v, int64_t stride, int64_t i) {
  if constexpr (KW == 1) return v[i];
  else return (static_cast<unsigned __int128>(v[stride + i]) << 64) | v[i];
}
template <int KW>
__device__ __forceinline__ uint64_t value_word(SortValue<KW> v, int w) {
  if constexpr (KW == 1) return v;
  else return static_cast<uint64_t>(v >> (64 * w));
}
// Lower bound of x among the sorted values [0, n) by one whole wavefront: 64
// pivots a step (4 dependent reads for 10^7 values instead of 23).
template <int KW>
__device__ __forceinline__ int64_t wave_lower_bound(const uint64_t* __restrict__ v, int64_t stride, int64_t n,
                                                    SortValue<KW> x, int lane) {
  int64_t lo = 0, hi = n;  // the bound lies in [lo, hi]
  while (hi - lo > 64) {
    const int64_t step = (hi - lo + 63) / 64, q = lo + (lane + 1) * step - 1;
    const int c = __popcll(__ballot(q < hi && load_value<KW>(v, stride, q) < x));  // the first c pivots are below x
    const int64_t nlo = lo + c * step, nhi = lo + (c + 1) * step - 1;
    lo = nlo < hi ? nlo : hi;
    hi = nhi < hi ? nhi : hi;
  }
  return lo + __popcll(__ballot(lo + lane < hi && load_value<KW>(v, stride, lo + lane) < x));
}

// Per tile of kRunTile sorted keys: the number of run heads (first key, or
// value differing from the previous key), the position of the first head (-1
// if none), the sums (entry_share) of the entries before it -- the part of a
// run that began in an earlier tile -- and the main-list position of the
// tile's first value (mrank: the main list's n sort values), which with the
// next tile's bounds the positions of the tile's runs; win[ntiles] is the end
// of the last tile's.
template <int KW, int S>
__global__ __launch_bounds__(kBlock) void k_run_count(const uint64_t* __restrict__ keys,
                                                      const int64_t* __restrict__ pay, const int64_t* __restrict__ pn,
                                                      int64_t nsb, int64_t stride, int fb,
                                                      const uint64_t* __restrict__ mrank, int64_t n, int64_t cap,
                                                      const int64_t* __restrict__ pmain, int64_t ntiles,
                                                      int32_t* __restrict__ tcnt, int32_t* __restrict__ tfirst,
                                                      int64_t* __restrict__ tpre, int64_t* __restrict__ win,
                                                      Stats* __restrict__ st) {
  constexpr int R = kRunTile / kBlock, NV = 3 * S;
  stamp(st, kStRuns);
  const int64_t ns = list_len(pn, nsb);
  __shared__ int64_t wsh[kBlock / 64];
  __shared__ int32_t wfirst[kBlock / 64];
  const int64_t tile = blockIdx.x, t0 = tile * kRunTile;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (t0 >= ns) {  // a grid sized by a bound: an empty tile
    if (threadIdx.x == 0) {
      tcnt[tile] = 0;
      tfirst[tile] = -1;
    }
    return;
  }
  n = list_len(pmain, n);
  int32_t c = 0;
  int first_here = kRunTile;  // this wavefront's first head in the tile
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t i = t0 + r * kBlock + threadIdx.x;
    bool h = false;
    if (i < ns) {
      uint64_t k[KW], prev[KW];
#pragma unroll
      for (int w = 0; w < KW; ++w) {
        k[w] = keys[w * stride + i];
        prev[w] = i > 0 ? keys[w * stride + i - 1] : 0;
      }
      h = i == 0 || !same_value<KW>(k, prev, fb);
    }
    c += h ? 1 : 0;
    const unsigned long long b = __ballot(h);
    if (b && first_here == kRunTile) first_here = r * kBlock + wave * 64 + __builtin_ctzll(b);
  }
  if (lane == 0) wfirst[wave] = first_here;
  if (wave == kBlock / 64 - 1) {
    const int64_t lb = wave_lower_bound<KW>(mrank, cap, n, load_value<KW>(keys, stride, t0) >> fb, lane);
    if (lane == 0) win[tile] = lb;
  }
  const bool last = t0 + kRunTile >= ns;
  if (last && wave == 0) {  // one past the last value's position
    const int64_t lb = wave_lower_bound<KW>(mrank, cap, n, load_value<KW>(keys, stride, ns - 1) >> fb, lane);
    if (lane == 0) win[tile + 1] = lb;
  }
  const int64_t t = block_sum(c, wsh);  // its barriers also publish wfirst
  int first = kRunTile;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) first = wfirst[w] < first ? wfirst[w] : first;
  const uint64_t fmask = (uint64_t{1} << fb) - 1;
  int64_t acc[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) acc[k] = 0;
  if (first > 0) {  // block-uniform
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int j = r * kBlock + static_cast<int>(threadIdx.x);
      const int64_t i = t0 + j;
      if (j < first && i < ns) {
        int64_t pop[S], cv[NV];
#pragma unroll
        for (int q = 0; q < S; ++q) pop[q] = pay[q * stride + i];
        entry_share<S>(static_cast<int64_t>(keys[i] & fmask), pop, false, cv);
#pragma unroll
        for (int k = 0; k < NV; ++k) acc[k] += cv[k];
      }
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] = block_sum(acc[k], wsh);
  }
  if (threadIdx.x == 0) {
    tcnt[tile] = static_cast<int32_t>(t);
    tfirst[tile] = first < kRunTile ? first : -1;
#pragma unroll
    for (int k = 0; k < NV; ++k) tpre[tile * NV + k] = acc[k];
  }
}

// Sum of cnt[0..b) (off, when given, holds it) for the whole block.
__device__ __forceinline__ int64_t tiles_before(const int32_t* __restrict__ cnt, const int64_t* __restrict__ off,
                                                int64_t b, int64_t* wsh) {
  if (off) return off[b];
  int64_t x = 0;
  for (int64_t k = threadIdx.x; k < b; k += kBlock) x += cnt[k];
  return block_sum(x, wsh);
}

// Runs longer than this are reduced by a wavefront each (a queue in LDS), so a
// determinant spawned onto thousands of times does not hold one lane while
// its wavefront idles; shorter ones by one thread each.  16 measured the same
// for one space and 40 us against 35 for pairs (7e5 two-word keys).  (One
// such run after the other by the whole block, with loads waited for one by
// one: k_runs 24 us against 17 with 9e4 walkers on a 14-site ring, 87 against
// 76 for 4.3e6 keys.)
constexpr int kShortRun = 32;

// Inputs and outputs of k_runs.
struct RunArgs {
  const uint64_t* keys;  // sorted keys and payload
  const int64_t* pay;
  int64_t ns;            // list length, or a bound of it with the length at pns
  const int64_t* pns;
  int64_t stride;
  int fb;
  const int32_t* tcnt;   // k_run_count's outputs; toff: exclusive prefix of tcnt, or null
  const int64_t* toff;
  const int32_t* tfirst;
  const int64_t* tpre;
  const int64_t* win;
  int64_t ntiles;
  const uint64_t* mrank;  // the main list's sort values, its length n (or a bound, the length at pmain)
  int64_t n;
  const int64_t* pmain;
  int64_t cap;
  int64_t* pop_new;
  int initiator, real_amps, replay;
  int64_t rf;
  uint64_t seed;
  uint32_t cyc;
  const uint32_t* pcyc;
  uint64_t* nval;  // new determinants of the tile, from slot tile * kRunTile: values, populations, positions
  int64_t* npop;
  int32_t* npos;
  int32_t* ncnt;   // and their number
  Stats* st;
};
constexpr int kRunWin = 2048;  // main-list values a tile stages in LDS (two-word values: half as many)

// annihilate_spawn_t(_initiator), annihilate_main_list(_initiator) and
// round_low_population_spawns (src/spawn_data.F90:859-1101,
// src/annihilation.f90:294-486, 613-675) over the sorted keys and populations,
// one block per tile of kRunTile keys.  The tile's run heads are listed in
// order (wavefront ballots); thread h takes run h and sums its entries' shares
// (entry_share), so every lane has a run whatever the run lengths.  Runs longer
// than kShortRun are queued and reduced by the wavefronts afterwards.  The
// tile's last run adds the head-free prefixes of the following tiles
// (k_run_count) up to the next head.  The run's first entry is its first in
// sorted order: the reference's quicksort order in replay mode, the earliest
// spawned in production (the stable sort of an attempt-ordered list).
// Run totals stay in LDS; each run's value is then looked up among the main
// list's values between the tile's bounds (staged in LDS when they fit) -- a
// hit adds to the post-death populations, a miss is a new determinant if it may
// be one and its rounded populations do not vanish -- and the tile's new
// determinants are listed in order.  Runs are compared by value, so only the
// determinants that are inserted are ever unranked, by the insertion.
// (Before, every run was unranked and written as a record that three further
// kernels read: 253 us for 4.3e6 keys on 2.8e6 determinants (k_runs 165,
// search bounds 26, merge 39, rounding of new 18, their list 5), 76 us now and
// 20 for the ranks k_scatter_main moves and the unranking of the inserted.)
template <int KW, int S>
__global__ __launch_bounds__(kBlock) void k_runs(RunArgs g) {
  using V = SortValue<KW>;
  constexpr int R = kRunTile / kBlock, NV = 3 * S, NW = kBlock / 64, WIN = kRunWin / KW, kAhead = 4;
  __shared__ int32_t wcount[R][NW];
  __shared__ int32_t hpos[kRunTile + 1];  // tile-relative index of each head, in order; then the tile length
  __shared__ int16_t longq[kRunTile];     // runs (by h) left to a whole wavefront
  __shared__ uint8_t rflag[kRunTile];     // a run's flags, bit 7: some population is not zero
  __shared__ int64_t rtot[S][kRunTile];   // a run's populations
  __shared__ V wval[WIN];                 // the main-list values between the tile's bounds when they fit
  __shared__ int32_t nlong;
  __shared__ int64_t wsh[NW];
  const int64_t ns = list_len(g.pns, g.ns);
  const int64_t stride = g.stride;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t tile = blockIdx.x, t0 = tile * kRunTile;
  if (t0 >= ns) {  // block-uniform
    if (tid == 0) g.ncnt[tile] = 0;
    return;
  }
  const int n = static_cast<int>(ns - t0 < kRunTile ? ns - t0 : kRunTile);
  const int fb = g.fb;
  const uint64_t fmask = (uint64_t{1} << fb) - 1;
  // every value of the tile lies in [value(t0), value(t0 + n)], so its lower bound lies in [wlo, whi]
  const int64_t nm = list_len(g.pmain, g.n);
  const int64_t wlo = g.win[tile], wend = g.win[tile + 1] + 1, whi = wend < nm ? wend : nm;
  const bool staged = whi - wlo <= WIN;
  if (staged)
    for (int64_t q = tid; q < whi - wlo; q += kBlock) wval[q] = load_value<KW>(g.mrank, g.cap, wlo + q);
  bool head[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int j = r * kBlock + tid;
    const int64_t i = t0 + j;
    head[r] = false;
    if (j < n) {
      uint64_t k[KW], prev[KW];
#pragma unroll
      for (int w = 0; w < KW; ++w) {
        k[w] = g.keys[w * stride + i];
        prev[w] = i > 0 ? g.keys[w * stride + i - 1] : 0;
      }
      head[r] = i == 0 || !same_value<KW>(k, prev, fb);
    }
  }
  unsigned long long bal[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    bal[r] = __ballot(head[r]);
    if (lane == 0) wcount[r][wave] = __popcll(bal[r]);
  }
  if (tid == 0) nlong = 0;
  const int64_t rbase = tiles_before(g.tcnt, g.toff, tile, wsh);
  __syncthreads();
  int32_t total = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int32_t p = total + __popcll(bal[r] & ((1ull << lane) - 1));
    for (int w = 0; w < NW; ++w) {
      if (w < wave) p += wcount[r][w];
      total += wcount[r][w];
    }
    if (head[r]) hpos[p] = r * kBlock + tid;
  }
  if (tid == 0) {
    hpos[total] = n;
    if (t0 + n >= ns) g.st->nruns = rbase + total;
  }
  __syncthreads();
  // the shares of run h's entries [a, b) of the tile, from index `from` (stride `step`)
  auto shares = [&](int a, int b, int from, int step, int64_t* acc) {
    for (int j = from; j < b; j += kAhead * step) {
      uint64_t key[kAhead];
      int64_t pop[kAhead][S];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {  // loads of kAhead entries in flight
        const int64_t i = t0 + (j + u * step < b ? j + u * step : j);
        key[u] = g.keys[i];
#pragma unroll
        for (int q = 0; q < S; ++q) pop[u][q] = g.pay[q * stride + i];
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        if (j + u * step >= b) break;
        int64_t cv[NV];
        entry_share<S>(static_cast<int64_t>(key[u] & fmask), pop[u], j + u * step == a, cv);
#pragma unroll
        for (int k = 0; k < NV; ++k) acc[k] += cv[k];
      }
    }
  };
  // run h's totals complete: the continuation of the tile's last run and the initiator rules
  auto finish = [&](int h, int64_t* acc) {
    if (h == total - 1 && t0 + n < ns && g.tfirst[tile + 1] != 0) {
      for (int64_t u = tile + 1; u < g.ntiles && u * kRunTile < ns; ++u) {
#pragma unroll
        for (int k = 0; k < NV; ++k) acc[k] += g.tpre[u * NV + k];
        if (g.tfirst[u] >= 0) break;
      }
    }
    int fl = 0;
#pragma unroll
    for (int sp = 0; sp < S; ++sp) {
      const int64_t tot = acc[sp], init = acc[S + sp], evs = acc[2 * S + sp];
      if (tot != 0) fl |= 0x80;
      if (g.initiator) {
        const int st = tot >= 0 ? 1 : -1, si = init >= 0 ? 1 : -1;
        if (!(init != 0 && st == si) && !(evs > 1 || evs < -1)) fl |= 1 << sp;
      }
      rtot[sp][h] = tot;
    }
    rflag[h] = static_cast<uint8_t>(fl);
  };
  for (int h = tid; h < total; h += kBlock) {
    const int a = hpos[h], b = hpos[h + 1];
    if (b - a > kShortRun) {
      longq[atomicAdd(&nlong, 1)] = static_cast<int16_t>(h);
      continue;
    }
    int64_t acc[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] = 0;
    shares(a, b, a, 1, acc);
    finish(h, acc);
  }
  __syncthreads();
  const int nq = nlong;
  for (int q = wave; q < nq; q += NW) {
    const int h = longq[q];
    const int a = hpos[h], b = hpos[h + 1];
    int64_t acc[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] = 0;
    shares(a, b, a + lane, 64, acc);
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] = wave_sum(acc[k]);
    if (lane == 0) finish(h, acc);
  }
  __syncthreads();
  // merge with the main list and list the new determinants, kBlock runs at a time in order
  const uint32_t cyc = cycle_of(g.pcyc, g.cyc);
  int32_t nnew = 0;
  for (int h0 = 0; h0 < total; h0 += kBlock) {  // block-uniform
    const int h = h0 + tid;
    bool isnew = false;
    V val = 0;
    int64_t pop[S], lo = 0;
    if (h < total && (rflag[h] & 0x80)) {
      const int fl = rflag[h] & 0x7f;
      val = load_value<KW>(g.keys, stride, t0 + hpos[h]) >> fb;
      bool hit;
      if (staged) {
        int a = 0, b = static_cast<int>(whi - wlo);
        while (a < b) {
          const int mid = (a + b) >> 1;
          if (wval[mid] < val)
            a = mid + 1;
          else
            b = mid;
        }
        lo = wlo + a;
        hit = a < whi - wlo && wval[a] == val;
      } else {
        int64_t a = wlo, b = whi;
        while (a < b) {
          const int64_t mid = (a + b) >> 1;
          if (load_value<KW>(g.mrank, g.cap, mid) < val)
            a = mid + 1;
          else
            b = mid;
        }
        lo = a;
        hit = lo < nm && load_value<KW>(g.mrank, g.cap, lo) == val;
      }
#pragma unroll
      for (int sp = 0; sp < S; ++sp) pop[sp] = rtot[sp][h];
      if (hit) {
#pragma unroll
        for (int sp = 0; sp < S; ++sp) {
          int64_t& m = g.pop_new[sp * g.cap + lo];
          if (!g.initiator)
            m += pop[sp];
          else if (m != 0)
            m += pop[sp];
          else if (!((fl >> sp) & 1))
            m = pop[sp];
        }
      } else {
        bool keep = !g.initiator;
        if (g.initiator) {
#pragma unroll
          for (int sp = 0; sp < S; ++sp) {
            if ((fl >> sp) & 1)
              pop[sp] = 0;
            else
              keep = true;
          }
        }
        if (keep) {
          if (g.replay) {
            isnew = true;  // the stream's rounding draws follow the main list's
          } else {
            if (g.real_amps) {
              const int64_t r = rbase + h;
              fqd::Philox rng(g.seed, static_cast<uint32_t>(r), static_cast<uint32_t>(r >> 32),
                              cyc ^ (fqd::kDrawRoundSpawn << 24));
#pragma unroll
              for (int sp = 0; sp < S; ++sp) pop[sp] = fqd::stoch_round_pop(rng, pop[sp], g.rf);
            }
#pragma unroll
            for (int sp = 0; sp < S; ++sp) isnew = isnew || pop[sp] != 0;
          }
        }
      }
    }
    const unsigned long long bn = __ballot(isnew);
    if (lane == 0) wcount[0][wave] = __popcll(bn);
    __syncthreads();
    int32_t k = nnew + __popcll(bn & ((1ull << lane) - 1));
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      if (w < wave) k += wcount[0][w];
      nnew += wcount[0][w];
    }
    if (isnew) {
      const int64_t slot = t0 + k;
#pragma unroll
      for (int w = 0; w < KW; ++w) g.nval[w * stride + slot] = value_word<KW>(val, w);
#pragma unroll
      for (int sp = 0; sp < S; ++sp) g.npop[sp * stride + slot] = pop[sp];
      g.npos[slot] = static_cast<int32_t>(lo);
    }
    __syncthreads();  // wcount is rewritten by the next round
  }
  if (tid == 0) g.ncnt[tile] = nnew;
}

// ---------------------------------------------------------------------------
// Kernels: semi-stochastic projection
// ---------------------------------------------------------------------------
// Element (i, j) of the core Hamiltonian as create_determ_hamil stores it
// (src/semi_stoch.F90:533-685): <D_i|H|D_j>, H_ii - H_00 on the diagonal,
// times the quasi-Newton weight (1 here); the transpose (<D_j|H|D_i>) for
// separate annihilation.
__device__ __forceinline__ double determ_elem(const Sys& s, const uint64_t* fi, int64_t i, int64_t j, int transp) {
  uint64_t fj[FQ_MAX_WORDS];
#pragma unroll
  for (int w = 0; w < FQ_MAX_WORDS; ++w) fj[w] = w < s.W ? s.determ[w * s.ndeterm + j] : 0;
  double h = transp ? fqd::hmatel(s, fj, fi) : fqd::hmatel(s, fi, fj);
  if (i == j) h = h - s.H00;
  return 1.0 * h;
}
constexpr double kDetermEps = 1.0e-12;  // depsilon: smaller elements are not stored

// Non-zero elements per core row: one block per row, threads over columns.
__global__ __launch_bounds__(kBlock) void k_determ_count(Sys s, int transp, int64_t* __restrict__ cnt) {
  __shared__ int64_t wsh[kBlock / 64];
  const int64_t i = blockIdx.x;
  uint64_t fi[FQ_MAX_WORDS];
#pragma unroll
  for (int w = 0; w < FQ_MAX_WORDS; ++w) fi[w] = w < s.W ? s.determ[w * s.ndeterm + i] : 0;
  int64_t c = 0;
  for (int64_t j = threadIdx.x; j < s.ndeterm; j += kBlock) c += fabs(determ_elem(s, fi, i, j, transp)) > kDetermEps;
  c = block_sum(c, wsh);
  if (threadIdx.x == 0) cnt[i] = c;
}

// The row's elements in column order from row[i] (block-wide ranks per chunk
// of kBlock columns).
__global__ __launch_bounds__(kBlock) void k_determ_fill(Sys s, int transp, const int64_t* __restrict__ row,
                                                        int32_t* __restrict__ col, double* __restrict__ mat) {
  __shared__ uint32_t wsh[kBlock / 64];
  const int64_t i = blockIdx.x;
  uint64_t fi[FQ_MAX_WORDS];
#pragma unroll
  for (int w = 0; w < FQ_MAX_WORDS; ++w) fi[w] = w < s.W ? s.determ[w * s.ndeterm + i] : 0;
  int64_t base = row[i];
  for (int64_t j0 = 0; j0 < s.ndeterm; j0 += kBlock) {  // block-uniform trip count
    const int64_t j = j0 + threadIdx.x;
    double h = 0.0;
    bool keep = false;
    if (j < s.ndeterm) {
      h = determ_elem(s, fi, i, j, transp);
      keep = fabs(h) > kDetermEps;
    }
    uint32_t tot;
    const uint32_t off = block_exclusive_u32(keep ? 1u : 0u, wsh, tot);
    if (keep) {
      col[base + off] = static_cast<int32_t>(j);
      mat[base + off] = h;
    }
    base += tot;
  }
}

// sum + a term of each stored element of row `row` in order, the terms being
// scale * H * v (separate) or H * v (combined), by one wavefront: its lanes
// evaluate 64 terms at a time (coalesced reads of the row, the next chunk's in
// flight) and park them in LDS, and every lane then adds them in the row's
// order, so the sum is the one thread's sum bit for bit.
__device__ __forceinline__ double determ_row_sum(const DetermDev& dd, int S, int64_t row, int sp, double sum,
                                                 bool scaled, double scale, int lane, double* __restrict__ term) {
  const int64_t k0 = dd.row[row], k1 = dd.row[row + 1];
  auto value = [&](int64_t k) {
    if (k >= k1) return 0.0;
    const double m = dd.mat[k], v = dd.vec[dd.col[k] * S + sp];
    return scaled ? scale * m * v : m * v;
  };
  double next = value(k0 + lane);
  for (int64_t k = k0; k < k1; k += 64) {
    __builtin_amdgcn_wave_barrier();  // the previous chunk's reads come first (LDS is in order within a wavefront)
    term[lane] = next;
    __builtin_amdgcn_wave_barrier();
    next = value(k + 64 + lane);
    if (k1 - k >= 64) {
#pragma unroll 16
      for (int q = 0; q < 64; ++q) sum = sum + term[q];
    } else {
      for (int q = 0; q < static_cast<int>(k1 - k); ++q) sum = sum + term[q];
    }
  }
  return sum;
}

// Production deterministic projection, one wavefront per core determinant and
// space, each with its own draw keyed (row, space, cycle).  Combined
// annihilation writes the encoded amplitude to the spawned list after the
// stochastic spawns (key and payload, as an initiator's spawn; the count is
// added by k_add_nspawn); separate annihilation adds it to the core
// determinant's post-death population.  (One thread per row read its row
// uncoalesced, one element per trip to memory: 239 us with a 1000-determinant
// core of a 26-orbital molecule, 13 now.)
__global__ __launch_bounds__(kBlock) void k_determ_proj(Sys s, KeyPlan kp, DetermDev dd, double tau, double sh0,
                                                        double sh1, double e0, double e1, uint64_t seed, uint32_t cyc,
                                                        int64_t cap, int64_t* __restrict__ pop_new,
                                                        uint64_t* __restrict__ keys, int64_t* __restrict__ pay,
                                                        int64_t scap, Stats* __restrict__ st) {
  __shared__ double term[kBlock / 64][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * (kBlock / 64) + wave;
  if (t >= dd.nd * s.S) return;  // whole wavefront; no block barriers below
  const int64_t row = t / s.S;
  const int sp = static_cast<int>(t - row * s.S);
  const double shift = sp == 0 ? sh0 : sh1, eold = sp == 0 ? e0 : e1;
  const double v = dd.vec[row * s.S + sp];
  // the expressions of determ_separate and determ_combined
  double amp;
  if (dd.separate) {
    amp = determ_row_sum(dd, s.S, row, sp, -(tau * (eold * (1.0 - 1.0) - shift * 1.0)) * v, true, -1.0 * tau, lane,
                         term[wave]);
  } else {
    const double out = determ_row_sum(dd, s.S, row, sp, 0.0, false, 0.0, lane, term[wave]);
    amp = -tau * (out + (eold * (1.0 - 1.0) - 1.0 * shift) * v);
  }
  if (lane != 0) return;
  fqd::Philox rng(seed, static_cast<uint32_t>(row), static_cast<uint32_t>(sp) << 28, cyc ^ (fqd::kDrawDeterm << 24));
  const int64_t k = fqd::stoch_encode(rng, amp, s.rf);
  if (dd.separate) {
    pop_new[sp * cap + dd.pos[row]] += k;
    return;
  }
  const int64_t slot = st->nspawn + t;
  if (slot >= scap) {
    st->spawn_overflow = 1;
    return;
  }
  for (int q = 0; q < s.S; ++q) pay[q * scap + slot] = q == sp ? k : 0;
  uint64_t f[FQ_MAX_WORDS];
#pragma unroll
  for (int w = 0; w < FQ_MAX_WORDS; ++w) f[w] = w < s.W ? s.determ[w * dd.nd + row] : 0;
  uint64_t key[2];
  make_key_any(kp, f, s.W, 0, key);
  for (int w = 0; w < kp.kw; ++w) keys[w * scap + slot] = key[w];
}
__global__ void k_add_nspawn(Stats* __restrict__ st, int64_t m) { st->nspawn += m; }

// ---------------------------------------------------------------------------
// Kernels: merge with the main list, rounding, insertion
// ---------------------------------------------------------------------------
// Number of rounding draws an entry needs: spaces with 0 < |pop| < rf.
__device__ __forceinline__ int round_draws(const int64_t* p, int64_t stride, int64_t i, int S, int64_t rf) {
  int c = 0;
  for (int sp = 0; sp < S; ++sp) {
    const int64_t v = p[sp * stride + i];
    const int64_t av = v < 0 ? -v : v;
    if (av < rf && v != 0) ++c;
  }
  return c;
}

// A main-list entry of the semi-stochastic core (kept whatever its
// population, never rounded: remove_unoccupied_dets, src/annihilation.f90:537-600).
__device__ __forceinline__ bool is_core_entry(const Sys& s, const uint64_t* __restrict__ det, int64_t cap,
                                              int64_t i) {
  if (s.ndeterm == 0) return false;
  uint64_t f[FQ_MAX_WORDS];
#pragma unroll
  for (int w = 0; w < FQ_MAX_WORDS; ++w) f[w] = w < s.W ? det[w * cap + i] : 0;
  return fqd::core_index(s, f) >= 0;
}

__global__ void k_count_round_main(Sys s, int64_t n, int64_t cap, const int64_t* __restrict__ pop_new,
                                   const uint64_t* __restrict__ det, int64_t* __restrict__ mdraw) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  mdraw[i] = (s.real_amps && !is_core_entry(s, det, cap, i)) ? round_draws(pop_new, cap, i, s.S, s.rf) : 0;
}
// Replay: rounding draws of a run tile's candidates, then (one block per tile)
// the rounding itself at the tile's place in the stream, keeping the candidates
// that survive at the front of the tile's slots.
__global__ __launch_bounds__(kBlock) void k_count_round_new(Sys s, const int32_t* __restrict__ ncnt,
                                                            const int64_t* __restrict__ npop, int64_t stride,
                                                            int64_t* __restrict__ ndraw) {
  __shared__ int64_t wsh[kBlock / 64];
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kRunTile;
  const int cnt = ncnt[blockIdx.x];
  int64_t c = 0;
  if (s.real_amps)
    for (int j = threadIdx.x; j < cnt; j += kBlock) c += round_draws(npop, stride, t0 + j, s.S, s.rf);
  c = block_sum(c, wsh);
  if (threadIdx.x == 0) ndraw[blockIdx.x] = c;
}
__global__ __launch_bounds__(kBlock) void k_replay_round_new(Sys s, int KW, int32_t* __restrict__ ncnt,
                                                             uint64_t* __restrict__ nval, int64_t* __restrict__ npop,
                                                             int32_t* __restrict__ npos, int64_t stride,
                                                             const double* __restrict__ rbuf, int64_t rbase,
                                                             const int64_t* __restrict__ ndraw_off) {
  __shared__ uint32_t wsh[kBlock / 64];
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kRunTile;
  const int cnt = ncnt[blockIdx.x];
  int64_t drawn = ndraw_off[blockIdx.x];
  uint32_t kept = 0;
  for (int j0 = 0; j0 < cnt; j0 += kBlock) {  // block-uniform; slots before j0 are free to overwrite
    const int j = j0 + static_cast<int>(threadIdx.x);
    const bool in = j < cnt;
    int64_t pop[FQ_MAX_SPACES] = {0, 0};
    uint64_t val[2] = {0, 0};
    int32_t pos = 0;
    const uint32_t nd = in && s.real_amps ? round_draws(npop, stride, t0 + j, s.S, s.rf) : 0;
    uint32_t all;
    const int64_t at = rbase + drawn + block_exclusive_u32(nd, wsh, all);
    bool alive = false;
    if (in) {
      fqd::ReplayRng rng{rbuf, at, at + nd, false};
      for (int sp = 0; sp < s.S; ++sp) {
        pop[sp] = npop[sp * stride + t0 + j];
        if (s.real_amps) pop[sp] = fqd::stoch_round_pop(rng, pop[sp], s.rf);
        alive = alive || pop[sp] != 0;
      }
      for (int w = 0; w < KW; ++w) val[w] = nval[w * stride + t0 + j];
      pos = npos[t0 + j];
    }
    drawn += all;
    const uint32_t k = kept + block_exclusive_u32(alive ? 1u : 0u, wsh, all);  // its barriers follow every read above
    kept += all;
    if (alive) {
      for (int w = 0; w < KW; ++w) nval[w * stride + t0 + k] = val[w];
      for (int sp = 0; sp < s.S; ++sp) npop[sp * stride + t0 + k] = pop[sp];
      npos[t0 + k] = pos;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) ncnt[blockIdx.x] = static_cast<int32_t>(kept);
}

// Survivor flags are kept as bits, one ballot word per 64 consecutive entries,
// with the survivors of its tile before each word (mpre) and per tile (mcnt,
// prefixed in moff): an entry's rank among the survivors is moff + mpre + the
// word's bits below it.
//
// Blocks [0, mtiles): remove_unoccupied_dets over a tile of the main list --
// round small real populations, mark survivors.  The other blocks: run tile
// b's new determinants go to their places in one list (a tile's place is the
// count of those before it; noff, when given, holds it).  The two have nothing
// to do with each other and share a launch.
struct RoundArgs {
  Sys s;
  int64_t n;  // main-list length, or a bound of it with the length at pn
  const int64_t* pn;
  int64_t cap, mtiles;
  const uint64_t* det;
  int64_t* pop_new;
  int replay;
  const double* rbuf;
  int64_t rbase;
  const int64_t* mdraw_off;
  uint64_t seed;
  uint32_t cyc;
  const uint32_t* pcyc;
  uint64_t* mmask;
  uint16_t* mpre;
  int32_t* mcnt;
  int KW;
  int64_t scap, ntiles;
  const int32_t* ncnt;
  const int64_t* noff;
  const uint64_t* nval;
  const int64_t* npop;
  const int32_t* npos;
  uint64_t* lval;
  int64_t* lpop;
  int32_t* lpos;
  Stats* st;
};
__global__ __launch_bounds__(kBlock) void k_round(RoundArgs g) {
  constexpr int R = kMainTile / kBlock, NW = kBlock / 64;
  __shared__ int64_t wsh[NW];
  __shared__ int32_t wc[R * NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int S = g.s.S;
  if (g.st->resort) return;  // the list has yet to be sorted
  stamp(g.st, kStRound);
  if (blockIdx.x >= g.mtiles) {
    const int64_t b = blockIdx.x - g.mtiles;
    const int32_t cnt = g.ncnt[b];
    if (cnt == 0 && b != g.ntiles - 1) return;  // block-uniform
    const int64_t k0 = tiles_before(g.ncnt, g.noff, b, wsh), t0 = b * kRunTile;
    for (int j = tid; j < cnt; j += kBlock) {
      for (int w = 0; w < g.KW; ++w) g.lval[w * g.scap + k0 + j] = g.nval[w * g.scap + t0 + j];
      for (int sp = 0; sp < S; ++sp) g.lpop[sp * g.scap + k0 + j] = g.npop[sp * g.scap + t0 + j];
      g.lpos[k0 + j] = g.npos[t0 + j];
    }
    if (tid == 0 && b == g.ntiles - 1) g.st->nnew = k0 + cnt;
    return;
  }
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kMainTile;
  const int64_t nl = list_len(g.pn, g.n);  // entries past it (up to the bound n) are marked dead
  const uint32_t cyc = cycle_of(g.pcyc, g.cyc);
  unsigned long long bal[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t i = t0 + r * kBlock + tid;
    bool alive = false;
    if (i < nl) {
      if (is_core_entry(g.s, g.det, g.cap, i)) {
        alive = true;
      } else {
        int64_t p[FQ_MAX_SPACES];
#pragma unroll
        for (int sp = 0; sp < FQ_MAX_SPACES; ++sp) p[sp] = sp < S ? g.pop_new[sp * g.cap + i] : 0;
        if (g.s.real_amps) {
          bool small = false;  // some population is rounded (draws only matter then)
#pragma unroll
          for (int sp = 0; sp < FQ_MAX_SPACES; ++sp) small = small || (p[sp] != 0 && p[sp] < g.s.rf && p[sp] > -g.s.rf);
          if (small) {
            if (g.replay) {
              fqd::ReplayRng rng{g.rbuf, g.rbase + g.mdraw_off[i], g.rbase + g.mdraw_off[i + 1], false};
              for (int sp = 0; sp < S; ++sp) p[sp] = fqd::stoch_round_pop(rng, p[sp], g.s.rf);
            } else {
              fqd::Philox rng(g.seed, static_cast<uint32_t>(i), static_cast<uint32_t>(i >> 32),
                              cyc ^ (fqd::kDrawRoundMain << 24));
              for (int sp = 0; sp < S; ++sp) p[sp] = fqd::stoch_round_pop(rng, p[sp], g.s.rf);
            }
            for (int sp = 0; sp < S; ++sp) g.pop_new[sp * g.cap + i] = p[sp];
          }
        }
        alive = p[0] != 0 || p[1] != 0;
      }
    }
    bal[r] = __ballot(alive);
    if (lane == 0) wc[r * NW + wave] = __popcll(bal[r]);
  }
  __syncthreads();
  int32_t before = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      if (lane == 0 && w == wave) {
        const int64_t word = (t0 >> 6) + r * NW + w;
        g.mmask[word] = bal[r];
        g.mpre[word] = static_cast<uint16_t>(before);
      }
      before += wc[r * NW + w];
    }
  }
  if (tid == 0) g.mcnt[blockIdx.x] = before;
}

// Insertion of the surviving main entries.  An entry moves up by its rank among
// the survivors plus the number of new determinants inserted at or before it:
// lpos lists their positions, non-decreasing because the runs are sorted, so
// each tile bounds its part of the list (two wavefronts' searches), stages it
// in LDS when it fits and every thread searches only there.  Insertion is
// skipped when the main list would overflow (insert_new_walkers' psip_list%error
// path).  Also written: the survivors before each tile (moff), the new length,
// and the tile's sums of |N|.
struct InsertArgs {
  Sys s;
  int64_t n;
  const int64_t* pn;
  int64_t cap, mtiles;
  const uint64_t* det;
  const uint64_t* rank;  // the list's sort values (rank_words of them; 0: the determinant itself)
  int rank_words;
  const int64_t* pop_new;
  const double* kii;
  const uint64_t* mmask;
  const uint16_t* mpre;
  const int32_t* mcnt;
  const int64_t* moff_in;  // exclusive prefix of mcnt, or null
  int64_t* moff;
  const int32_t* lpos;
  const uint64_t* lval;
  const int64_t* lpop;
  int64_t scap;
  Stats* st;
  uint64_t* det_out;
  uint64_t* rank_out;
  int64_t* pop_out;
  double* kii_out;
  int64_t* abs_part;  // [S][abs_ld]: the tiles', then k_scatter_new's blocks'
  int64_t abs_ld;
};
constexpr int kInsWin = 2048;
// First k in [0, n) with v[k] >= x, by one wavefront.
__device__ __forceinline__ int64_t wave_lower_bound32(const int32_t* __restrict__ v, int64_t n, int64_t x, int lane) {
  int64_t lo = 0, hi = n;
  while (hi - lo > 64) {
    const int64_t step = (hi - lo + 63) / 64, q = lo + (lane + 1) * step - 1;
    const int c = __popcll(__ballot(q < hi && v[q] < x));
    const int64_t nlo = lo + c * step, nhi = lo + (c + 1) * step - 1;
    lo = nlo < hi ? nlo : hi;
    hi = nhi < hi ? nhi : hi;
  }
  return lo + __popcll(__ballot(lo + lane < hi && v[lo + lane] < x));
}
__global__ __launch_bounds__(kBlock) void k_scatter_main(InsertArgs g) {
  constexpr int R = kMainTile / kBlock, NW = kBlock / 64;
  __shared__ int32_t win[kInsWin];
  __shared__ int64_t wsh[NW], bounds[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (g.st->resort) return;
  const int64_t n = list_len(g.pn, g.n), tile = blockIdx.x, t0 = tile * kMainTile;
  const int64_t nnew = g.st->nnew;
  // survivors before the tile, and of the whole list
  int64_t off, total;
  if (g.moff_in) {
    off = g.moff_in[tile];
    total = g.moff_in[g.mtiles];
  } else {
    int64_t pre = 0, all = 0;
    for (int64_t k = tid; k < g.mtiles; k += kBlock) {
      const int64_t c = g.mcnt[k];
      all += c;
      if (k < tile) pre += c;
    }
    off = block_sum(pre, wsh);
    total = block_sum(all, wsh);
  }
  const bool ovf = total + nnew > g.cap;
  if (tid == 0) {
    g.moff[tile] = off;
    if (tile == g.mtiles - 1) {
      g.moff[g.mtiles] = total;
      g.st->nmain = total;
      g.st->main_overflow = ovf ? 1 : 0;
      g.st->new_n = ovf ? total : total + nnew;
    }
  }
  int64_t sum[FQ_MAX_SPACES] = {0, 0};
  if (t0 < n) {  // block-uniform
    if (wave < 2) {
      const int64_t b = ovf ? 0 : wave_lower_bound32(g.lpos, nnew, wave == 0 ? t0 : t0 + kMainTile, lane);
      if (lane == 0) bounds[wave] = b;
    }
    __syncthreads();
    const int64_t c0 = bounds[0], c1 = bounds[1];
    const bool staged = c1 - c0 <= kInsWin;
    if (staged)
      for (int64_t q = tid; q < c1 - c0; q += kBlock) win[q] = g.lpos[c0 + q];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t i = t0 + r * kBlock + tid;
      const int64_t word = i >> 6;  // the wavefront's 64 entries
      const uint64_t m = t0 + r * kBlock + wave * 64 < n ? g.mmask[word] : 0;
      if (!((m >> lane) & 1)) continue;
      int64_t shift;
      if (staged) {
        int a = 0, b = static_cast<int>(c1 - c0);
        while (a < b) {
          const int mid = (a + b) >> 1;
          if (win[mid] <= i)
            a = mid + 1;
          else
            b = mid;
        }
        shift = c0 + a;
      } else {
        int64_t a = c0, b = c1;
        while (a < b) {
          const int64_t mid = (a + b) >> 1;
          if (g.lpos[mid] <= i)
            a = mid + 1;
          else
            b = mid;
        }
        shift = a;
      }
      const int64_t o = off + g.mpre[word] + __popcll(m & ((1ull << lane) - 1)) + shift;
      for (int w = 0; w < g.s.W; ++w) g.det_out[w * g.cap + o] = g.det[w * g.cap + i];
      for (int w = 0; w < g.rank_words; ++w) g.rank_out[w * g.cap + o] = g.rank[w * g.cap + i];
#pragma unroll
      for (int sp = 0; sp < FQ_MAX_SPACES; ++sp)
        if (sp < g.s.S) {
          const int64_t p = g.pop_new[sp * g.cap + i];
          g.pop_out[sp * g.cap + o] = p;
          sum[sp] += p < 0 ? -p : p;
        }
      g.kii_out[o] = g.kii[i];
    }
  }
  for (int sp = 0; sp < g.s.S; ++sp) {
    const int64_t x = block_sum(sp == 0 ? sum[0] : sum[1], wsh);
    if (tid == 0) g.abs_part[sp * g.abs_ld + tile] = x;
  }
}

// Insertion of the new determinants (grid-stride, list order = rank order):
// the determinant unranked from its sort value, K_ii from the diagonal rule.
// A molecular system's dense pair tables (2 norb^2 doubles) and the binomial
// table are staged in LDS when jk_lds / kp.binom_lds say so.
template <bool WIDE>
__global__ __launch_bounds__(kBlock) void k_scatter_new(InsertArgs g, KeyPlan kp, const Sys* __restrict__ sys_arr,
                                                        int jk_lds) {
  extern __shared__ double dyn[];
  __shared__ int64_t wsh[kBlock / 64];
  const Sys& s = g.s;
  const int64_t nnew = g.st->main_overflow ? 0 : g.st->nnew;
  const int64_t n = list_len(g.pn, g.n), nmain = g.st->nmain;
  const int64_t k0 = static_cast<int64_t>(blockIdx.x) * kBlock;
  int64_t sum[FQ_MAX_SPACES] = {0, 0};
  if (k0 < nnew) {  // block-uniform
    double* jk = dyn;
    const int nn = s.norb * s.norb;
    uint64_t* binom = reinterpret_cast<uint64_t*>(dyn + (jk_lds ? 2 * nn : 0));
    if (jk_lds)
      for (int q = threadIdx.x; q < nn; q += kBlock) {
        jk[q] = s.jmat[q];
        jk[nn + q] = s.kmat[q];
      }
    if (kp.rank && kp.binom_lds) {  // one-word ranks: the table saturated at 2^64 - 1, one word per entry
      const int nv = kp.nbasis * kp.nel;
      for (int k = threadIdx.x; k < nv; k += kBlock) {
        if constexpr (WIDE) {
          binom[2 * k] = kp.binom[2 * k];
          binom[2 * k + 1] = kp.binom[2 * k + 1];
        } else {
          binom[k] = kp.binom[2 * k + 1] ? ~uint64_t{0} : kp.binom[2 * k];
        }
      }
    }
    __syncthreads();
    for (int64_t k = k0 + threadIdx.x; k < nnew; k += static_cast<int64_t>(gridDim.x) * kBlock) {
      const int64_t p = g.lpos[k];
      int64_t o = k + nmain;
      if (p < n) {  // survivors before entry p
        const uint64_t m = g.mmask[p >> 6];
        o = k + g.moff[p / kMainTile] + g.mpre[p >> 6] + __popcll(m & ((1ull << (p & 63)) - 1));
      }
      uint64_t f[FQ_MAX_WORDS] = {0, 0};
      const uint64_t v0 = g.lval[k];
      if (!kp.rank) {
        f[0] = v0;  // the word is its own value (batched instances: with the instance index)
      } else {
        const unsigned __int128 v = WIDE ? (static_cast<unsigned __int128>(g.lval[g.scap + k]) << 64) | v0 : v0;
        if (kp.binom_lds)
          unrank<WIDE>(kp, binom, !WIDE, v, f);
        else
          unrank<WIDE>(kp, kp.binom, false, v, f);
      }
      FQ_FOR_WORDS(w, s.W) g.det_out[w * g.cap + o] = f[w];
      for (int w = 0; w < g.rank_words; ++w) g.rank_out[w * g.cap + o] = g.lval[w * g.scap + k];
#pragma unroll
      for (int sp = 0; sp < FQ_MAX_SPACES; ++sp)
        if (sp < s.S) {
          const int64_t x = g.lpop[sp * g.scap + k];
          g.pop_out[sp * g.cap + o] = x;
          sum[sp] += x < 0 ? -x : x;
        }
      if (sys_arr) {  // batched: the instance's diagonal
        const Sys& si = sys_arr[f[0] >> kInstShift];
        f[0] &= kOrbMask;
        g.kii_out[o] = fqd::diagonal(si, f) - si.H00;
      } else if (jk_lds) {
        g.kii_out[o] = fqd::diagonal_mol(s, f, jk, jk + nn) - s.H00;
      } else {
        g.kii_out[o] = fqd::diagonal(s, f) - s.H00;
      }
    }
  }
  for (int sp = 0; sp < s.S; ++sp) {
    const int64_t x = block_sum(sp == 0 ? sum[0] : sum[1], wsh);
    if (threadIdx.x == 0) g.abs_part[sp * g.abs_ld + g.mtiles + blockIdx.x] = x;
  }
}

// Sort values of the main list (a loaded list; the insertion keeps them up).
__global__ void k_rank_list(KeyPlan kp, int W, int64_t n, int64_t cap, const uint64_t* __restrict__ det,
                            uint64_t* __restrict__ rank) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint64_t f[FQ_MAX_WORDS] = {0, 0}, key[2];
  FQ_FOR_WORDS(w, W) f[w] = det[w * cap + i];
  kp.flag_bits = 0;
  make_key_any(kp, f, W, 0, key);
  for (int w = 0; w < kp.kw; ++w) rank[w * cap + i] = key[w];
}

__global__ void k_zero(int64_t* __restrict__ p, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------------------
// Host helpers
// ---------------------------------------------------------------------------
// Make room for `extra` more draws after the live part [rng_pos, rng_end),
// moving the live part to the front of a (possibly larger) buffer.
int reserve_rng(fq_engine* e, int64_t extra) {
  if (e->rng_end + extra <= e->rng_cap) return FQ_OK;
  const int64_t live = e->rng_end - e->rng_pos;
  const int64_t cap = std::max<int64_t>(live + extra, 2 * e->rng_cap);
  double* nb = nullptr;
  if (dalloc(&nb, cap) != FQ_OK) return FQ_ERR_NOMEM;
  if (live > 0)
    FQ_HIP(hipMemcpyAsync(nb, e->rng_buf + e->rng_pos, sizeof(double) * live, hipMemcpyDeviceToDevice, e->stream));
  FQ_HIP(hipStreamSynchronize(e->stream));
  dfree(e->rng_buf);
  e->rng_buf = nb;
  e->rng_cap = cap;
  e->rng_end = live;
  e->rng_pos = 0;
  return FQ_OK;
}

int sync_stats(fq_engine* e) {
  FQ_HIP(hipMemcpyAsync(&e->h_stats, e->d_stats, sizeof(Stats), hipMemcpyDeviceToHost, e->stream));
  FQ_HIP(hipStreamSynchronize(e->stream));
  return FQ_OK;
}

KeyPlan key_plan(const fq_engine* e) {
  KeyPlan kp{};
  kp.kw = e->sort_kw;
  kp.flag_bits = e->flag_bits;
  kp.rank = e->rank_words ? 1 : 0;
  kp.nel = e->sys.nel;
  kp.nbasis = e->sys.nbasis;
  kp.binom = e->d_binom;
  return kp;
}

// Bytes of the rank table, and whether kernels may stage it in LDS.
size_t binom_bytes(const fq_engine* e) {
  return e->rank_words ? sizeof(uint64_t) * 2 * e->sys.nbasis * e->sys.nel : 0;
}
constexpr size_t kBinomLdsMax = 48 * 1024;

// Digits of the sort: the fewest passes of 8- or 9-bit digits covering the
// key's value field (bits flag_bits .. flag_bits + value_bits - 1).
DigitPlan digit_plan(const fq_engine* e) {
  DigitPlan dp{};
  const int bits = e->value_bits;
  const int passes = e->digit8 ? std::max(1, (bits + 7) / 8) : std::max(1, (bits + 8) / 9);
  const int n9 = e->digit8 ? 0 : std::max(0, std::min(passes, bits - 8 * passes));
  int shift = e->flag_bits;
  for (int p = 0; p < passes; ++p) {
    dp.shift[p] = shift;
    dp.bits[p] = p < n9 ? 9 : 8;
    shift += dp.bits[p];
  }
  dp.np = passes;
  return dp;
}

// Key layout and sort buffers for the engine's value width.
int setup_sort(fq_engine* e) {
  const int vb = e->rank_words ? e->rank_bits : e->key_bits;
  const int fb = e->S;
  if (vb + fb > 128) return FQ_ERR_ARG;
  const int kw = vb + fb > 64 ? 2 : 1;
  if (e->batched && kw != 1) return FQ_ERR_ARG;  // the instance bounds read one key word
  const int64_t scap = e->scap;
  e->value_bits = vb;
  e->flag_bits = fb;
  int rc = FQ_OK;
  // The spawned list as determinant words and records (sdet, srec) is only
  // read before the sort (replay walk, caller-supplied lists, rank exchange);
  // it shares the memory of the sort's second buffers.
  const bool new_kw = kw != e->sort_kw || !e->kbuf[0];
  if (new_kw) {
    for (int b = 0; b < 2; ++b) {
      dfree(e->kbuf[b]);
      rc |= dalloc(&e->kbuf[b], (b == 0 ? kw : std::max(kw, e->W)) * scap);
    }
  }
  e->sort_kw = kw;
  for (int b = 0; b < 2; ++b)
    if (!e->pbuf[b]) rc |= dalloc(&e->pbuf[b], (b == 0 ? e->S : std::max(e->S, rec_stride(e->S))) * scap);
  e->sdet = e->kbuf[1];
  e->srec = e->pbuf[1];
  if (!e->perm && e->par.rng_mode == FQ_RNG_REPLAY) rc |= dalloc(&e->perm, scap);
  if (!e->pass_cnt) rc |= dalloc(&e->pass_cnt, 512 * kSortBlocks);
  if (!e->pass_off) rc |= dalloc(&e->pass_off, 512 * kSortBlocks + 1);
  const int64_t rtiles = ceil_div(scap, kRunTile) + 2;
  if (!e->run_tcnt) rc |= dalloc(&e->run_tcnt, rtiles);
  if (!e->run_toff) rc |= dalloc(&e->run_toff, rtiles);
  if (!e->run_tfirst) rc |= dalloc(&e->run_tfirst, rtiles);
  if (!e->run_tpre) rc |= dalloc(&e->run_tpre, 3 * e->S * rtiles);
  if (!e->run_win) rc |= dalloc(&e->run_win, rtiles);
  if (!e->new_cnt) rc |= dalloc(&e->new_cnt, rtiles);
  if (!e->new_off) rc |= dalloc(&e->new_off, rtiles);
  for (int b = 0; b < 2; ++b)
    if (!e->new_pos[b]) rc |= dalloc(&e->new_pos[b], scap);
  if (!e->new_pop) rc |= dalloc(&e->new_pop, e->S * scap);
  if (new_kw) {
    dfree(e->new_val);
    rc |= dalloc(&e->new_val, kw * scap);
  }
  // the main list's sort values (a determinant that is its own value needs none)
  if (new_kw || !e->rank_words)
    for (int b = 0; b < 2; ++b) dfree(e->mrank[b]);
  for (int b = 0; b < 2 && e->rank_words; ++b)
    if (!e->mrank[b]) rc |= dalloc(&e->mrank[b], kw * e->cap + 1);
  // (batched instances, whose sort values are one word, read them to the cycle's end)
  if (!e->att_off && !(kw == 2 && e->rank_words)) rc |= dalloc(&e->att_off, e->S * e->cap + 1);
  return rc == FQ_OK ? FQ_OK : FQ_ERR_NOMEM;
}

// Sort keys and payload made from the spawned list's determinants and records
// (when the spawning pass did not make them): perm (may be null) gives the order.
void launch_make_keys(fq_engine* e, int64_t ns, const uint32_t* perm) {
  hipLaunchKernelGGL(k_make_keys, dim3(grid_for(ns)), dim3(kBlock), 0, e->stream, key_plan(e), e->S, e->sdet, e->srec,
                     e->W, ns, e->scap, perm, e->kbuf[0], e->pbuf[0]);
}

// One radix pass from buffer `src` to the other.
// ns: the list length, or a bound of it when pns (the device count) is given.
template <int KW, int S, int DB, int R>
int sort_pass(fq_engine* e, int src, int64_t ns, const int64_t* pns, int shift) {
  constexpr int T = kBlock * R;
  const int64_t nb = std::min<int64_t>(ceil_div(ns, T), kSortBlocks);
  hipLaunchKernelGGL((k_pass_count<KW, S, DB, R>), dim3(static_cast<unsigned>(nb)), dim3(kBlock), 0, e->stream,
                     e->kbuf[src], pns, ns, e->scap, shift, e->pass_cnt, e->radix_passes == 0 ? e->d_stats : nullptr);
  hipLaunchKernelGGL(k_pass_rowscan, dim3(1u << DB), dim3(kSortBlocks), 0, e->stream, static_cast<int>(nb),
                     e->pass_cnt, e->pass_off);
  hipLaunchKernelGGL((k_pass_scatter<KW, S, DB, R>), dim3(static_cast<unsigned>(nb)), dim3(kBlock), 0, e->stream,
                     e->kbuf[src], e->pbuf[src], e->kbuf[1 - src], e->pbuf[1 - src], pns, ns, e->scap, shift,
                     e->pass_cnt, e->pass_off);
  return FQ_OK;
}
template <int KW, int S>
int sort_pass_db(fq_engine* e, int src, int64_t ns, const int64_t* pns, int shift, int db, bool small) {
  constexpr int R = sort_items(KW, S), Q = kSmallSortItems;
  if (small)
    return db == 9 ? sort_pass<KW, S, 9, Q>(e, src, ns, pns, shift) : sort_pass<KW, S, 8, Q>(e, src, ns, pns, shift);
  return db == 9 ? sort_pass<KW, S, 9, R>(e, src, ns, pns, shift) : sort_pass<KW, S, 8, R>(e, src, ns, pns, shift);
}

// Spawned lists bounded by this many entries run the whole annihilation in
// launches sized by the bound, reading the length on the device: the blocks past
// the length (the bound is the attempts, two to ten times the spawned entries)
// cost less than a stop of the host for the exact length (~20 us).
constexpr int64_t kNoWaitMax = int64_t{1} << 21;

// The main list's sort values in buffer c.
const uint64_t* main_values(const fq_engine* e, int c) { return e->rank_words ? e->mrank[c] : e->det[c]; }
constexpr int64_t kNewBlocks = 1024;  // most blocks of the new determinants' insertion
constexpr size_t kInsertLdsMax = 120 * 1024;  // LDS of their tables (set_insert_lds raises the default 64 KB)

// Index bits of k_sort_small beside the value, and the list length it takes (0: none).
int small_sort_idx_bits(const fq_engine* e) { return std::min(13, 64 - e->value_bits); }
int small_sort_limit(const fq_engine* e) {
  static_assert(kSmallSort == 1 << 13, "indexes of 13 bits");
  return e->sort_kw == 1 && small_sort_idx_bits(e) >= 8 ? 1 << small_sort_idx_bits(e) : 0;
}

// Sort the spawned list, reduce its runs and merge them with the main list;
// leaves the tiles' new determinants in the sort's idle buffers (new_src) and
// the number of run tiles in run_tiles.  The list holds ns entries, or, when
// pns is given (production, no host wait for the length), *pns entries with ns
// a bound of them.  no_small: not by k_sort_small unless the bound is short.
int sort_and_reduce(fq_engine* e, int64_t ns, const int64_t* pns, bool replay, uint32_t cyc, bool no_small) {
  const bool keys_ready = e->keys_ready;  // made by the spawning pass for this spawned list
  e->keys_ready = false;
  const int64_t scap = e->scap;
  const int kw = e->sort_kw, S = e->S;
  hipStream_t st = e->stream;
  int src = 0;
  bool small = false;
  e->radix_passes = 0;
  if (ns > 0) {
    if (replay) {
      hipLaunchKernelGGL(k_replay_qsort, dim3(1), dim3(1), 0, st, e->sdet, ns, e->W, scap, e->perm, e->d_stats);
      launch_make_keys(e, ns, e->perm);
    } else {
      if (!keys_ready) launch_make_keys(e, ns, nullptr);
      const DigitPlan dp = digit_plan(e);
      const int limit = small_sort_limit(e);
      // in LDS when the list is short, by its bound or, if not, by the last cycle's length
      small = ns <= limit || (pns && !e->capturing && ns <= kNoWaitMax && !no_small && e->last_ns >= 0 &&
                              e->last_ns + e->last_ns / 4 + 256 <= limit);
      if (small) {
        hipLaunchKernelGGL(S == 1 ? k_sort_small<1> : k_sort_small<2>, dim3(1), dim3(kSmallSortBlock), 0, st,
                           e->kbuf[0], e->pbuf[0], e->kbuf[1], e->pbuf[1], pns, ns, scap, e->flag_bits, e->value_bits,
                           small_sort_idx_bits(e), limit, e->d_stats);
        src = 1;
        e->radix_passes = ceil_div(e->value_bits, kSmallSortBits);
        pns = &e->d_stats->sorted;
      }
      // tile size by the last cycle's length where this one's is only bounded
      const int64_t like = pns && !e->capturing && e->last_ns >= 0 ? std::min(e->last_ns, ns) : ns;
      const bool st_small = like <= int64_t{kSortBlocks} * kBlock * kSmallSortItems;
      for (int p = 0; p < dp.np && !small; ++p) {
        int rc;
        if (kw == 1)
          rc = S == 1 ? sort_pass_db<1, 1>(e, src, ns, pns, dp.shift[p], dp.bits[p], st_small)
                      : sort_pass_db<1, 2>(e, src, ns, pns, dp.shift[p], dp.bits[p], st_small);
        else
          rc = S == 1 ? sort_pass_db<2, 1>(e, src, ns, pns, dp.shift[p], dp.bits[p], st_small)
                      : sort_pass_db<2, 2>(e, src, ns, pns, dp.shift[p], dp.bits[p], st_small);
        if (rc != FQ_OK) return rc;
        src = 1 - src;
        ++e->radix_passes;
      }
    }
  }
  if (pns && !e->capturing && !small && ns > kNoWaitMax) {  // the passes are queued: now the exact length (copied before them)
    FQ_HIP(hipEventSynchronize(e->ev_len));
    // the attempts cannot exceed the bound the spawning launches covered (every
    // entry makes at most floor(|N|) + 1 of them, |N| for integer populations)
    if (e->h_len[2] > e->spawn_bound) return FQ_ERR_DEVICE;
    ns = std::min<int64_t>(e->h_len[0], e->scap);
    pns = nullptr;
  }
  // Runs: totals, merge with the main list, the tiles' new determinants.
  const int64_t nt = ceil_div(ns, kRunTile);
  e->run_tiles = nt;
  e->new_src = 1 - src;
  if (ns > 0) {
    const int64_t* dn = e->capturing ? e->dn : nullptr;
    const uint64_t* mrank = main_values(e, e->cur);
    auto cnt = kw == 1 ? (S == 1 ? k_run_count<1, 1> : k_run_count<1, 2>)
                       : (S == 1 ? k_run_count<2, 1> : k_run_count<2, 2>);
    hipLaunchKernelGGL(cnt, dim3(static_cast<unsigned>(nt)), dim3(kBlock), 0, st, e->kbuf[src], e->pbuf[src], pns, ns,
                       scap, e->flag_bits, mrank, e->n, e->cap, dn, nt, e->run_tcnt, e->run_tfirst, e->run_tpre,
                       e->run_win, e->d_stats);
    if (nt > e->prefix_runs) {
      const int rc = scan_exclusive(e, e->run_tcnt, e->run_toff, nt);
      if (rc != FQ_OK) return rc;
    }
    RunArgs g{};
    g.keys = e->kbuf[src];
    g.pay = e->pbuf[src];
    g.ns = ns;
    g.pns = pns;
    g.stride = scap;
    g.fb = e->flag_bits;
    g.tcnt = e->run_tcnt;
    g.toff = nt > e->prefix_runs ? e->run_toff : nullptr;
    g.tfirst = e->run_tfirst;
    g.tpre = e->run_tpre;
    g.win = e->run_win;
    g.ntiles = nt;
    g.mrank = mrank;
    g.n = e->n;
    g.pmain = dn;
    g.cap = e->cap;
    g.pop_new = e->pop_new;
    g.initiator = e->sys.initiator;
    g.real_amps = e->sys.real_amps;
    g.replay = replay ? 1 : 0;
    g.rf = e->sys.rf;
    g.seed = e->par.philox_seed;
    g.cyc = cyc;
    g.pcyc = e->capturing ? e->dcyc : nullptr;
    g.nval = e->kbuf[1 - src];
    g.npop = e->pbuf[1 - src];
    g.npos = e->new_pos[0];
    g.ncnt = e->new_cnt;
    g.st = e->d_stats;
    auto kern = kw == 1 ? (S == 1 ? k_runs<1, 1> : k_runs<1, 2>) : (S == 1 ? k_runs<2, 1> : k_runs<2, 2>);
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(nt)), dim3(kBlock), 0, st, g);
  }
  return FQ_OK;
}

// Annihilation proper: merge runs, round, compact, insert.  ns spawned
// entries are in the spawned list; pop_new holds the post-death populations.
// est_blocks: blocks of this cycle's k_det_pass, whose partials k_finish adds
// (0: the estimators are in the stats, or there are none).
int annihilate(fq_engine* e, int64_t ns, const int64_t* pns, bool replay, uint32_t cyc, int64_t& rng_pos,
               int est_blocks = 0, bool no_small = false) {
  int rc = sort_and_reduce(e, ns, pns, replay, cyc, no_small);
  if (rc != FQ_OK) return rc;
  const int64_t ntiles = e->run_tiles;
  // a graph-captured cycle: n is a bound of the list's length, read on the device from dn
  const int64_t n = e->n, cap = e->cap, scap = e->scap;
  const int64_t* dn = e->capturing ? e->dn : nullptr;
  const uint32_t* dcyc = e->capturing ? e->dcyc : nullptr;
  const int c = e->cur, o = 1 - c, kw = e->sort_kw;
  hipStream_t st = e->stream;
  uint64_t* nval = e->kbuf[e->new_src];
  int64_t* npop = e->pbuf[e->new_src];
  // Rounding draws (replay: main list first, then new candidates, in order).
  int64_t main_draws = 0, new_draws = 0;
  if (replay) {
    if (e->sys.real_amps) {
      hipLaunchKernelGGL(k_count_round_main, dim3(grid_for(n)), dim3(kBlock), 0, st, e->sys, n, cap, e->pop_new,
                         e->det[c], e->mdraw);
      rc = scan_exclusive(e, e->mdraw, e->mdraw_off, n);
      if (rc != FQ_OK) return rc;
    }
    if (ntiles > 0) {
      hipLaunchKernelGGL(k_count_round_new, dim3(static_cast<unsigned>(ntiles)), dim3(kBlock), 0, st, e->sys,
                         e->new_cnt, npop, scap, e->ndraw);
      rc = scan_exclusive(e, e->ndraw, e->ndraw_off, ntiles);
      if (rc != FQ_OK) return rc;
    }
    if (e->sys.real_amps) {
      FQ_HIP(hipMemcpyAsync(&main_draws, e->mdraw_off + n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
      if (ntiles > 0)
        FQ_HIP(hipMemcpyAsync(&new_draws, e->ndraw_off + ntiles, sizeof(int64_t), hipMemcpyDeviceToHost, st));
      FQ_HIP(hipStreamSynchronize(st));
      if (rng_pos + main_draws + new_draws > e->rng_end) return FQ_ERR_RNG_EXHAUSTED;
    }
    if (ntiles > 0)
      hipLaunchKernelGGL(k_replay_round_new, dim3(static_cast<unsigned>(ntiles)), dim3(kBlock), 0, st, e->sys, kw,
                         e->new_cnt, nval, npop, e->new_pos[0], scap, e->rng_buf, rng_pos + main_draws, e->ndraw_off);
  }
  const int64_t mtiles = std::max<int64_t>(1, ceil_div(n, kMainTile));
  if (ntiles > e->prefix_runs) {
    rc = scan_exclusive(e, e->new_cnt, e->new_off, ntiles);
    if (rc != FQ_OK) return rc;
  }
  RoundArgs r{};
  r.s = e->sys;
  r.n = n;
  r.pn = dn;
  r.cap = cap;
  r.mtiles = mtiles;
  r.det = e->det[c];
  r.pop_new = e->pop_new;
  r.replay = replay ? 1 : 0;
  r.rbuf = e->rng_buf;
  r.rbase = rng_pos;
  r.mdraw_off = e->mdraw_off;
  r.seed = e->par.philox_seed;
  r.cyc = cyc;
  r.pcyc = dcyc;
  r.mmask = e->mmask;
  r.mpre = e->mpre;
  r.mcnt = e->mcnt;
  r.KW = kw;
  r.scap = scap;
  r.ntiles = ntiles;
  r.ncnt = e->new_cnt;
  r.noff = ntiles > e->prefix_runs ? e->new_off : nullptr;
  r.nval = nval;
  r.npop = npop;
  r.npos = e->new_pos[0];
  r.lval = e->new_val;
  r.lpop = e->new_pop;
  r.lpos = e->new_pos[1];
  r.st = e->d_stats;
  hipLaunchKernelGGL(k_round, dim3(static_cast<unsigned>(mtiles + ntiles)), dim3(kBlock), 0, st, r);
  rng_pos += main_draws + new_draws;
  if (mtiles > e->prefix_main) {  // offsets first: every tile's block would add too many counts
    rc = scan_exclusive(e, e->mcnt, e->moff, mtiles);
    if (rc != FQ_OK) return rc;
  }
  InsertArgs g{};
  g.s = e->sys;
  g.n = n;
  g.pn = dn;
  g.cap = cap;
  g.mtiles = mtiles;
  g.det = e->det[c];
  g.rank = e->mrank[c];
  g.rank_words = e->rank_words ? kw : 0;
  g.pop_new = e->pop_new;
  g.kii = e->kii[c];
  g.mmask = e->mmask;
  g.mpre = e->mpre;
  g.mcnt = e->mcnt;
  g.moff_in = mtiles > e->prefix_main ? e->moff : nullptr;
  g.moff = e->moff;
  g.lpos = e->new_pos[1];
  g.lval = e->new_val;
  g.lpop = e->new_pop;
  g.scap = scap;
  g.st = e->d_stats;
  g.det_out = e->det[o];
  g.rank_out = e->mrank[o];
  g.pop_out = e->pop;
  g.kii_out = e->kii[o];
  g.abs_part = e->abs_part;
  g.abs_ld = cap / kMainTile + 2 + kNewBlocks;
  hipLaunchKernelGGL(k_scatter_main, dim3(static_cast<unsigned>(mtiles)), dim3(kBlock), 0, st, g);
  int64_t nblk = mtiles;
  if (ns > 0) {
    // dense pair tables in LDS for the diagonal (up to 64 orbitals: 64 KB), the binomial table when it fits beside
    // them: both are read in chains (60 orbitals, 20 electrons in pairs: 78 us from L2, 59 from LDS)
    const size_t jk = e->sys.system == FQ_SYS_READ_IN && !e->batched
                          ? 2 * sizeof(double) * static_cast<size_t>(e->sys.norb) * e->sys.norb
                          : 0;
    const bool use_jk = jk > 0 && jk <= 65536;
    KeyPlan kp = key_plan(e);
    const size_t tab = binom_bytes(e) / (kw == 1 ? 2 : 1);
    kp.binom_lds = tab > 0 && tab + (use_jk ? jk : 0) <= kInsertLdsMax;
    const unsigned nb = static_cast<unsigned>(std::min<int64_t>(ceil_div(ns, kBlock), kNewBlocks));
    hipLaunchKernelGGL(kw == 1 ? k_scatter_new<false> : k_scatter_new<true>, dim3(nb), dim3(kBlock),
                       (use_jk ? jk : 0) + (kp.binom_lds ? tab : 0), st, g, kp, e->batched ? e->d_sys_arr : nullptr,
                       use_jk ? 1 : 0);
    nblk += nb;
  }
  hipLaunchKernelGGL(e->S == 1 ? k_finish<1> : k_finish<2>, dim3(1), dim3(kFinishBlock), 0, st, e->part_d, e->part_i,
                     est_blocks, e->abs_part, g.abs_ld, nblk, e->d_stats, e->h_pin);
  if (e->capturing) return FQ_OK;  // the caller reads the stats when the graph has run
  FQ_HIP(hipStreamSynchronize(st));
  e->h_stats = *e->h_pin;
  if (e->h_stats.resort) {  // longer than k_sort_small takes: its keys and the populations are as they were
    hipLaunchKernelGGL(k_zero, dim3(1), dim3(kBlock), 0, st, &e->d_stats->resort, int64_t{1});
    e->keys_ready = true;
    ++e->resorts;
    return annihilate(e, std::min<int64_t>(e->h_stats.nspawn, scap), nullptr, replay, cyc, rng_pos, est_blocks, true);
  }
  e->last_ns = pns ? std::min<int64_t>(e->h_stats.nspawn, scap) : ns;  // a caller's list is not counted on the device
  e->cur = o;
  e->n = e->h_stats.new_n;
  e->att_bound = -1;
  return FQ_OK;
}

// The cycle's times from its stamps (a phase without kernels: none) and its
// sizes: n determinants before it, ns spawned entries.
void fill_profile(fq_engine* e, int64_t n, int64_t ns) {
  int64_t t[kStamps];
  int64_t later = e->h_stats.stamp[kStEnd];
  for (int k = kStamps - 1; k >= 0; --k) {  // a phase that did not run starts where the next one does
    if (e->h_stats.stamp[k] != 0) later = e->h_stats.stamp[k];
    t[k] = later;
  }
  auto ms = [&](int from, int to) { return static_cast<double>(t[to] - t[from]) * e->ms_per_tick; };
  e->t_spawn = static_cast<float>(ms(kStBegin, kStSort));
  e->t_annih = static_cast<float>(ms(kStSort, kStEnd));
  e->t_total = static_cast<float>(ms(kStBegin, kStEnd));
  fq_profile_out& pr = e->prof;
  pr.det_pass_ms = ms(kStBegin, kStProposal);
  pr.proposal_ms = e->par.excit_gen == FQ_EXCIT_LEARNED ? ms(kStProposal, kStSpawn) : 0.0;
  pr.spawn_ms = ms(kStSpawn, kStSort);
  pr.sort_ms = ms(kStSort, kStRuns);
  pr.reduce_ms = ms(kStRuns, kStRound);
  pr.merge_ms = ms(kStRound, kStFinish);
  pr.total_ms = ms(kStBegin, kStFinish);
  pr.spawn_kernel_ms = static_cast<double>(e->h_stats.spawn_ticks) * e->ms_per_tick;
  pr.spawn_launches = e->spawn_launches;
  pr.nstates_in = n;
  pr.nattempts = e->h_stats.total_attempts;
  pr.nspawned = ns;
  pr.nruns = e->h_stats.nruns;
  pr.nstates_out = e->n;
  pr.radix_passes = e->radix_passes;
}

void fill_out(fq_engine* e, fq_cycle_out* out, int64_t rng_used) {
  std::memset(out, 0, sizeof(*out));
  const Stats& s = e->h_stats;
  const double rf = static_cast<double>(e->sys.rf);
  for (int sp = 0; sp < e->S; ++sp) {
    out->proj_energy[sp] = s.proj[sp];
    out->D0_population[sp] = s.d0[sp];
    out->nparticles[sp] = static_cast<double>(s.abs_pop[sp]) / rf;
  }
  out->nstates = e->n;
  out->nspawn_events = std::min<int64_t>(s.nspawn, e->scap);
  out->ndeath = s.ndeath;
  out->nattempts = s.total_attempts;
  out->rng_consumed = rng_used;
  out->spawn_overflow = s.spawn_overflow ? 1 : 0;
  out->main_overflow = s.main_overflow ? 1 : 0;
}

// ---- heat-bath tables: init_excit_mol_heat_bath (src/excit_gen_heat_bath_mol.F90:14-248)
// The reference's loops (i, j, a, b in that nesting) run in serial order per
// table entry: every sum below adds its terms in the reference's order.

// One thread per (i, j, a): the b loop; weights(b,a,j,i), weights_tot(a,j,i)
// and hb_ija%weights(a,j,i) (the same sum: invalid b contribute +0.0).
__global__ void k_hb_ijab(Sys s, double* __restrict__ ijab_w, double* __restrict__ ijab_tot,
                          double* __restrict__ ija_w) {
  const int nb = s.nbasis;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= static_cast<int64_t>(nb) * nb * nb) return;
  const int i = static_cast<int>(t / (static_cast<int64_t>(nb) * nb)) + 1;
  const int j = static_cast<int>((t / nb) % nb) + 1;
  const int a = static_cast<int>(t % nb) + 1;
  double* w = ijab_w + t * nb;
  double tot = 0.0;
  if (i != j && a != i && a != j) {
    const int it = i < j ? i : j, jt = i < j ? j : i;
    const int isymb = s.orb_sym[it - 1] ^ s.orb_sym[jt - 1] ^ s.orb_sym[a - 1];
    for (int b = 1; b <= nb; ++b) {
      double wb = 0.0;
      const bool spin_ok = (fqd::ms_of(it) == fqd::ms_of(a) && fqd::ms_of(jt) == fqd::ms_of(b)) ||
                           (fqd::ms_of(it) == fqd::ms_of(b) && fqd::ms_of(jt) == fqd::ms_of(a));
      if (spin_ok && s.orb_sym[b - 1] == isymb && b != a && b != i && b != j)
        wb = wb + fabs(fqd::sc2_excit(s, it, jt, a < b ? a : b, a < b ? b : a, false));
      w[b - 1] = wb;
      tot = tot + wb;
    }
  } else {
    for (int b = 0; b < nb; ++b) w[b] = 0.0;
  }
  ijab_tot[t] = tot;
  ija_w[t] = tot;
}

// One thread per (i, j): ij_weights(j,i) as the flat (a, b) sum and
// hb_ija%weights_tot(j,i) as the sum over a of the per-a totals.
__global__ void k_hb_ij(Sys s, const double* __restrict__ ijab_w, const double* __restrict__ ija_w,
                        double* __restrict__ ij_w, double* __restrict__ ija_tot) {
  const int nb = s.nbasis;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= static_cast<int64_t>(nb) * nb) return;
  double flat = 0.0, tot = 0.0;
  if (t / nb != t % nb) {
    const double* w = ijab_w + t * nb * nb;
    for (int64_t ab = 0; ab < static_cast<int64_t>(nb) * nb; ++ab) flat = flat + w[ab];
    for (int a = 0; a < nb; ++a) tot = tot + ija_w[t * nb + a];
  }
  ij_w[t] = flat;
  ija_tot[t] = tot;
}

// One thread per i: i_weights(i) = sum over j of ij_weights(j,i), and the
// reference's bias test (src/excit_gen_heat_bath_mol.F90:185-202) per i.
__global__ void k_hb_i(Sys s, const double* __restrict__ ij_w, const double* __restrict__ ija_w,
                       double* __restrict__ i_w, int* __restrict__ bias) {
  const int nb = s.nbasis;
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x) + 1;
  if (i > nb) return;
  double iw = 0.0;
  for (int j = 1; j <= nb; ++j) iw = iw + ij_w[static_cast<int64_t>(i - 1) * nb + (j - 1)];
  i_w[i - 1] = iw;
  int biased = 0;
  for (int a = 1; a <= nb; ++a) {
    int nz = 0;
    for (int j = 1; j <= nb; ++j)
      if (ija_w[(static_cast<int64_t>(i - 1) * nb + (j - 1)) * nb + (a - 1)] > fqd::kDepsilon) ++nz;
    if (nz < nb - s.nel && i != a && s.orb_sym[a - 1] == s.orb_sym[i - 1] && fqd::ms_of(a) == fqd::ms_of(i))
      biased = 1;
  }
  bias[i - 1] = biased;
}

// generate_alias_tables (lib/local/alias.f90:101-184) for ntab tables of n
// entries, one thread per table; table t is built when gate[t / gate_div] and
// tot[t] are nonzero (the reference builds no table otherwise).
__global__ void k_hb_alias(int64_t ntab, int n, const double* __restrict__ w, const double* __restrict__ tot,
                           const double* __restrict__ gate, int64_t gate_div, double* __restrict__ u,
                           int* __restrict__ k) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= ntab) return;
  if (!(fabs(gate[t / gate_div]) > 0.0) || !(fabs(tot[t]) > 0.0)) return;
  fqd::build_alias(n, w + t * n, tot[t], u + t * n, k + t * n);
}

int build_heat_bath(fq_engine* e) {
  Sys& s = e->sys;
  const int64_t nb = s.nbasis, n2 = nb * nb, n3 = n2 * nb, n4 = n3 * nb;
  int rc = FQ_OK;
  rc |= dalloc(&e->d_hb_i, nb);
  rc |= dalloc(&e->d_hb_ij, n2);
  rc |= dalloc(&e->d_hb_ija_tot, n2);
  rc |= dalloc(&e->d_hb_ija, n3);
  rc |= dalloc(&e->d_hb_ija_u, n3);
  rc |= dalloc(&e->d_hb_ija_k, n3);
  rc |= dalloc(&e->d_hb_ijab_tot, n3);
  rc |= dalloc(&e->d_hb_ijab, n4);
  rc |= dalloc(&e->d_hb_ijab_u, n4);
  rc |= dalloc(&e->d_hb_ijab_k, n4);
  rc |= dalloc(&e->d_hb_bias, nb);
  if (rc != FQ_OK) return FQ_ERR_NOMEM;
  hipStream_t st = e->stream;
  FQ_HIP(hipMemsetAsync(e->d_hb_ija_u, 0, sizeof(double) * n3, st));
  FQ_HIP(hipMemsetAsync(e->d_hb_ija_k, 0, sizeof(int) * n3, st));
  FQ_HIP(hipMemsetAsync(e->d_hb_ijab_u, 0, sizeof(double) * n4, st));
  FQ_HIP(hipMemsetAsync(e->d_hb_ijab_k, 0, sizeof(int) * n4, st));
  hipLaunchKernelGGL(k_hb_ijab, dim3(static_cast<unsigned>(ceil_div(n3, kBlock))), dim3(kBlock), 0, st, s,
                     e->d_hb_ijab, e->d_hb_ijab_tot, e->d_hb_ija);
  hipLaunchKernelGGL(k_hb_ij, dim3(static_cast<unsigned>(ceil_div(n2, kBlock))), dim3(kBlock), 0, st, s,
                     e->d_hb_ijab, e->d_hb_ija, e->d_hb_ij, e->d_hb_ija_tot);
  hipLaunchKernelGGL(k_hb_i, dim3(static_cast<unsigned>(ceil_div(nb, kBlock))), dim3(kBlock), 0, st, s, e->d_hb_ij,
                     e->d_hb_ija, e->d_hb_i, e->d_hb_bias);
  hipLaunchKernelGGL(k_hb_alias, dim3(static_cast<unsigned>(ceil_div(n2, kBlock))), dim3(kBlock), 0, st, n2,
                     static_cast<int>(nb), e->d_hb_ija, e->d_hb_ija_tot, e->d_hb_ija_tot, int64_t{1}, e->d_hb_ija_u,
                     e->d_hb_ija_k);
  hipLaunchKernelGGL(k_hb_alias, dim3(static_cast<unsigned>(ceil_div(n3, kBlock))), dim3(kBlock), 0, st, n3,
                     static_cast<int>(nb), e->d_hb_ijab, e->d_hb_ijab_tot, e->d_hb_ija_tot, nb, e->d_hb_ijab_u,
                     e->d_hb_ijab_k);
  FQ_HIP(hipGetLastError());
  std::vector<int> bias(static_cast<size_t>(nb));
  FQ_HIP(hipMemcpyAsync(bias.data(), e->d_hb_bias, sizeof(int) * nb, hipMemcpyDeviceToHost, st));
  FQ_HIP(hipStreamSynchronize(st));
  for (int v : bias)
    if (v) return FQ_ERR_BIASED;
  s.hb_i = e->d_hb_i;
  s.hb_ij = e->d_hb_ij;
  s.hb_ija = e->d_hb_ija;
  s.hb_ija_tot = e->d_hb_ija_tot;
  s.hb_ija_u = e->d_hb_ija_u;
  s.hb_ija_k = e->d_hb_ija_k;
  s.hb_ijab = e->d_hb_ijab;
  s.hb_ijab_tot = e->d_hb_ijab_tot;
  s.hb_ijab_u = e->d_hb_ijab_u;
  s.hb_ijab_k = e->d_hb_ijab_k;
  return FQ_OK;
}

template <class T>
int upload(T** dst, const T* src, int64_t count, hipStream_t st);

constexpr int sort_passes(int bits) { return bits < 9 ? 1 : (bits + 8) / 9; }  // 8- or 9-bit digits

// Binomial table and value width of the sort keys (combinatorial ranks).
int setup_rank_keys(fq_engine* e) {
  const int nb = e->sys.nbasis, nel = e->sys.nel;
  if (nel < 1 || nel > nb) return FQ_OK;
  // Pascal's triangle up to row nb in 128-bit integers (C(128, 64) < 2^128)
  std::vector<unsigned __int128> row(static_cast<size_t>(nel) + 1, 0), prev;
  std::vector<uint64_t> tab(static_cast<size_t>(2) * nb * nel, 0);
  row[0] = 1;
  for (int p = 0; p <= nb; ++p) {
    if (p > 0) {
      prev = row;
      for (int i = 1; i <= nel; ++i) row[i] = prev[i] + prev[i - 1];
    }
    if (p < nb)
      for (int i = 1; i <= nel; ++i) {
        tab[2 * (static_cast<size_t>(p) * nel + (i - 1))] = static_cast<uint64_t>(row[i]);
        tab[2 * (static_cast<size_t>(p) * nel + (i - 1)) + 1] = static_cast<uint64_t>(row[i] >> 64);
      }
  }
  unsigned __int128 top = row[nel] - 1;  // largest rank: C(nb, nel) - 1
  int bits = 1;
  while (bits < 128 && (top >> bits) != 0) ++bits;
  // A one-word determinant that sorts in as many passes as its rank is its own
  // sort value: no ranks are kept beside the main list and nothing is unranked.
  // (18 electrons in 36 spin orbitals, 3e6 determinants: k_scatter_main 46 -> 38
  // us without the 16 bytes of ranks per entry, k_scatter_new 26 -> 14 us.)
  if (e->W == 1 && nb + e->S <= 64 && sort_passes(nb) <= sort_passes(bits)) return FQ_OK;
  e->rank_bits = bits;
  e->rank_words = bits > 64 ? 2 : 1;
  return upload(&e->d_binom, tab.data(), static_cast<int64_t>(tab.size()), e->stream);
}

constexpr int64_t kTrainBatchMax = 16384;  // heat-bath samples per training step

int setup_learned(fq_engine* e) {
  Sys& s = e->sys;
  int rc = fqm::mlp_alloc(e->mlp, s.nbasis, s.W, kTrainBatchMax);
  if (rc != FQ_OK) return rc;
  rc = fqm::mlp_set_classes(e->mlp, s.nbss, s.ssbf, s.nsym_pg, s.max_sym_spin);
  if (rc != FQ_OK) return rc;
  rc = fqm::mlp_init(e->mlp, e->par.philox_seed, e->stream);
  if (rc != FQ_OK) return rc;
  e->mlp_tab_rows = std::min<int64_t>(e->cap, int64_t{1} << 16);
  if (dalloc(&e->mlp_tab, e->mlp_tab_rows * e->mlp.d_out) != FQ_OK || dalloc(&e->mlp_row, e->cap) != FQ_OK ||
      dalloc(&e->mlp_idx, e->cap) != FQ_OK)
    return FQ_ERR_NOMEM;
  s.mlp_tab = e->mlp_tab;
  s.mlp_aff = e->mlp.aff;
  s.mlp_rs = e->mlp.rs;
  s.mlp_crs = e->mlp.crs;
  s.mlp_cmask = e->mlp.cmask;
  s.mlp_au = e->mlp.au;
  s.mlp_ak = e->mlp.ak;
  s.mlp_cu = e->mlp.cu;
  s.mlp_ck = e->mlp.ck;
  {
    const std::vector<float> ones(2 * static_cast<size_t>(s.nbasis), 1.0f);
    if (dalloc(&e->mlp_flat, 2 * static_cast<int64_t>(s.nbasis)) != FQ_OK) return FQ_ERR_NOMEM;
    FQ_HIP(hipMemcpy(e->mlp_flat, ones.data(), sizeof(float) * ones.size(), hipMemcpyHostToDevice));
  }
  s.mlp_flat = e->mlp_flat;
  s.mlp_ld = e->mlp.d_out;
  s.mlp_row = e->mlp_row;
  s.mix = e->par.proposal_mix > 0.0 ? e->par.proposal_mix : 0.1;
  s.cls_sorted = e->cls_sorted;
  return FQ_OK;
}

// The insertion's dynamic LDS limit on the current device.
int set_insert_lds() {
  for (const void* f : {reinterpret_cast<const void*>(&k_scatter_new<false>),
                        reinterpret_cast<const void*>(&k_scatter_new<true>)})
    FQ_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kInsertLdsMax)));
  return FQ_OK;
}

// Determinants with at least min_att spawning attempts this cycle get a
// network row: k_mlp_mark counts them per tile of kMainTile entries, k_mlp_rows
// numbers them in list order (row[i], -1: none) and lists them (idx), adding up
// the counts of the tiles before its own (off, when given, holds them); the
// number of rows goes to the stats, where the inference reads it.  No row is
// numbered lim or above (lim: a bound of their number).
constexpr int64_t kProposalTable = int64_t{1} << 28;  // bytes the weight table may take for a bound of its rows
__device__ __forceinline__ bool gets_row(const int32_t* __restrict__ nat, int S, int64_t i, int64_t min_att) {
  int64_t a = 0;
  for (int sp = 0; sp < S; ++sp) a += nat[i * S + sp];
  return a >= min_att;
}
__global__ __launch_bounds__(kBlock) void k_mlp_mark(int64_t n, int S, const int32_t* __restrict__ nat,
                                                     int64_t min_att, int32_t* __restrict__ cnt,
                                                     Stats* __restrict__ st) {
  __shared__ int64_t wsh[kBlock / 64];
  stamp(st, kStProposal);
  int64_t c = 0;
  for (int r = 0; r < kMainTile / kBlock; ++r) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kMainTile + r * kBlock + threadIdx.x;
    c += i < n && gets_row(nat, S, i, min_att) ? 1 : 0;
  }
  c = block_sum(c, wsh);
  if (threadIdx.x == 0) cnt[blockIdx.x] = static_cast<int32_t>(c);
}
__global__ __launch_bounds__(kBlock) void k_mlp_rows(int64_t n, int S, const int32_t* __restrict__ nat,
                                                     int64_t min_att, int64_t lim, const int32_t* __restrict__ cnt,
                                                     const int64_t* __restrict__ off, int32_t* __restrict__ row,
                                                     int64_t* __restrict__ idx, Stats* __restrict__ st) {
  __shared__ int64_t wsh[kBlock / 64];
  __shared__ uint32_t wsh32[kBlock / 64];
  const int64_t before = tiles_before(cnt, off, blockIdx.x, wsh);
  uint32_t at = static_cast<uint32_t>(before);
  for (int r = 0; r < kMainTile / kBlock; ++r) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kMainTile + r * kBlock + threadIdx.x;
    bool on = i < n && gets_row(nat, S, i, min_att);
    uint32_t all;
    const uint32_t k = at + block_exclusive_u32(on ? 1u : 0u, wsh32, all);
    on = on && k < lim;
    if (i < n) row[i] = on ? static_cast<int32_t>(k) : -1;
    if (on) idx[k] = i;
    at += all;
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) st->mlp_rows = at < lim ? at : lim;
}

// A weight table of `rows` rows (the list's capacity at most).  keep: the old one
// stays where there is no memory for the new one beside it.
int grow_proposal_table(fq_engine* e, int64_t rows, bool keep) {
  rows = std::min(e->cap, rows);
  FQ_HIP(hipStreamSynchronize(e->stream));
  if (!keep) {
    dfree(e->mlp_tab);
    e->mlp_tab_rows = 0;
  }
  float* tab = nullptr;
  if (dalloc(&tab, rows * e->mlp.d_out) != FQ_OK) return FQ_ERR_NOMEM;
  dfree(e->mlp_tab);
  e->mlp_tab = tab;
  e->mlp_tab_rows = rows;
  e->sys.mlp_tab = tab;
  e->sys_dirty = true;
  return FQ_OK;
}

int scan_cb(void* ctx, const int64_t* in, int64_t* out, int64_t n) {
  return scan_exclusive(static_cast<fq_engine*>(ctx), in, out, n);
}

// One generator call per thread from determinant f (the excitation probe).
__global__ void k_probe(Sys s, uint64_t f0, uint64_t f1, const float* __restrict__ wrow, int64_t n, uint64_t seed,
                        int32_t* __restrict__ exc, double* __restrict__ pgen, double* __restrict__ hmat) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const uint64_t f[FQ_MAX_WORDS] = {f0, f1};
  fqd::Philox rng(seed, static_cast<uint32_t>(t), static_cast<uint32_t>(t >> 32), fqd::kDrawProbe << 24);
  fqd::Excit conn;
  double h = 0.0, pg = 1.0;
  const bool ok = fqd::generate_any(s, rng, f, wrow, conn, h, pg);
  exc[6 * t] = ok ? 1 : 0;
  exc[6 * t + 1] = ok ? conn.nexcit : 0;
  exc[6 * t + 2] = conn.from[0];
  exc[6 * t + 3] = conn.from[1];
  exc[6 * t + 4] = conn.to[0];
  exc[6 * t + 5] = conn.to[1];
  pgen[t] = pg;
  hmat[t] = h;
}


// Upload the system descriptor to its device copy when it has changed.
int sync_sysp(fq_engine* e) {
  if (!e->sys_dirty) return FQ_OK;
  FQ_HIP(hipMemcpyAsync(e->d_sysp, &e->sys, sizeof(Sys), hipMemcpyHostToDevice, e->stream));
  e->sys_dirty = false;
  return FQ_OK;
}

// Dynamic LDS of the heat-bath spawning kernel: nel weights per thread.
size_t hb_lds_bytes(int nel) { return static_cast<size_t>(nel) * kBlock * sizeof(double); }
// Whether that LDS, with the kernel's static LDS, fits a workgroup here.
bool hb_lds_fits(int device, int nel) {
  hipFuncAttributes fa;
  int maxlds = 0;
  if (hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(&k_spawn<fqd::kGenHeatBath, false, kSpawnTile>)) != hipSuccess ||
      hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess)
    return false;
  return fa.sharedSizeBytes + hb_lds_bytes(nel) <= static_cast<size_t>(maxlds);
}

// Dynamic LDS of the learned spawning kernel: the tile's parked child
// determinants, the affinity table and the flat weight row.
size_t learned_lds_bytes(int W, int nbasis, int tile = kSpawnTile) {
  const size_t nb = static_cast<size_t>(nbasis);
  return sizeof(uint64_t) * W * tile + sizeof(float) * (nb * nb + 2 * nb);
}
bool learned_lds_fits(int device, int W, int nbasis) {
  hipFuncAttributes fa;
  int maxlds = 0;
  if (hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(&k_spawn<fqd::kGenLearned, false, kSpawnTile>)) != hipSuccess ||
      hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess)
    return false;
  return fa.sharedSizeBytes + learned_lds_bytes(W, nbasis) <= static_cast<size_t>(maxlds);
}

// Attempt offsets of the nent entries from k_det_pass's attempts, and the parent
// windows of the spawning tiles of the first `attempts` attempts.
int scan_attempts(fq_engine* e, int64_t nent, int64_t attempts, int tile) {
  if (nent == 0) {
    hipLaunchKernelGGL(k_set_zero_total, dim3(1), dim3(1), 0, e->stream, att_offsets(e));
    return FQ_OK;
  }
  const int64_t nblk = ceil_div(nent, static_cast<int64_t>(kBlock) * e->S);
  const bool prefix = nblk <= e->prefix_attempts;
  if (!prefix) {
    const int rc = scan_exclusive(e, e->blk_att, e->blk_off, nblk);
    if (rc != FQ_OK) return rc;
  }
  hipLaunchKernelGGL(k_att_scan, dim3(grid_for(nent, kScanTile)), dim3(kBlock), 0, e->stream, att_counts(e), nent, e->blk_att,
                     nblk, kBlock * e->S, prefix ? nullptr : e->blk_off, att_offsets(e), e->tile_win,
                     ceil_div(attempts, tile), 31 - __builtin_clz(static_cast<unsigned>(tile)), e->d_stats);
  return FQ_OK;
}

// Pack the spawned entries of a batch of nbt attempts (tiles of `tile`); first:
// the cycle's only batch.  ptot: the attempt total on the device (recorded in
// the stats); tlim as in k_pack_tiles.
void pack_spawned(fq_engine* e, int64_t nbt, int tile, bool first, const int64_t* ptot, int64_t tlim = -1) {
  const int64_t nt = ceil_div(nbt, tile);
  KeyPlan kp = key_plan(e);
  const size_t tab = binom_bytes(e) / (e->sort_kw == 1 ? 2 : 1);
  kp.binom_lds = tab > 0 && tab <= kBinomLdsMax;
  hipLaunchKernelGGL(e->sort_kw == 1 ? k_pack_tiles<1> : k_pack_tiles<2>, dim3(static_cast<unsigned>(std::min<int64_t>(nt, 2048))), dim3(kBlock),
                     kp.binom_lds ? tab : 0, e->stream, e->W, e->S, nt, tile, e->tile_cnt, e->st_det, e->st_pop,
                     e->st_ent, e->bcap, e->scap, kp, e->kbuf[0], e->pbuf[0], e->d_stats, first ? 1 : 0, ptot, tlim);
  if (!first)
    hipLaunchKernelGGL(k_add_spawned, dim3(1), dim3(kBlock), 0, e->stream, e->tile_cnt, nt, ptot, e->d_stats);
}

// Attempts per tile of a cycle with at most `attempts` attempts of generator
// gen.  The learned generator's affinity table leaves LDS for two blocks of
// 1024-attempt tiles on a CU, four of 256-attempt ones, and its attempts are
// chains of table reads that need the wavefronts (9.5e5 attempts on 40 orbitals:
// 486 -> 322 us).
int spawn_tile(int gen, int64_t attempts) {
  return attempts <= kSmallTileMax || gen == fqd::kGenLearned ? kSmallTile : kSpawnTile;
}
// Most blocks of a spawning launch: as many as are resident for the learned
// generator, whose blocks each stage the affinity table once, else one per tile.
int64_t spawn_grid(int gen, int64_t tiles) { return std::min<int64_t>(tiles, gen == fqd::kGenLearned ? 1024 : 1 << 20); }
template <bool B, int T>
auto spawn_kernel(int gen) {
  if constexpr (B) {
    return gen == fqd::kGenHubK ? k_spawn<fqd::kGenHubK, true, T> : k_spawn<fqd::kGenMolRenorm, true, T>;
  } else {
    return gen == fqd::kGenHubK       ? k_spawn<fqd::kGenHubK, false, T>
           : gen == fqd::kGenHeatBath ? k_spawn<fqd::kGenHeatBath, false, T>
           : gen == fqd::kGenLearned  ? k_spawn<fqd::kGenLearned, false, T>
                                      : k_spawn<fqd::kGenMolRenorm, false, T>;
  }
}

int alloc_engine(fq_engine* e) {
  const int64_t cap = e->cap, scap = e->scap;
  const int W = e->W, S = e->S;
  int rc = FQ_OK;
  for (int b = 0; b < 2; ++b) {
    rc |= dalloc(&e->det[b], W * cap);
    rc |= dalloc(&e->kii[b], cap);
  }
  rc |= dalloc(&e->pop, S * cap);
  rc |= dalloc(&e->pop_new, S * cap);
  const int64_t mtiles = cap / kMainTile + 2;
  rc |= dalloc(&e->mmask, mtiles * (kMainTile / 64));
  rc |= dalloc(&e->mpre, mtiles * (kMainTile / 64));
  rc |= dalloc(&e->mcnt, mtiles);
  rc |= dalloc(&e->moff, mtiles);
  rc |= dalloc(&e->abs_part, S * (mtiles + kNewBlocks));
  const bool replay = e->par.rng_mode == FQ_RNG_REPLAY;
  if (replay) {  // rounding-draw counts of the replay stream
    rc |= dalloc(&e->mdraw, cap + 1);
    rc |= dalloc(&e->mdraw_off, cap + 1);
  }
  rc |= dalloc(&e->part_d, 4 * (cap / kBlock + 2));
  rc |= dalloc(&e->part_i, 2 * (cap / kBlock + 2));
  // spawning attempts are staged in batches of at most bcap (one slot each)
  e->bcap = std::min<int64_t>(scap, int64_t{1} << 26);
  rc |= dalloc(&e->st_det, W * e->bcap);
  rc |= dalloc(&e->st_pop, e->bcap);
  rc |= dalloc(&e->st_ent, e->bcap);
  rc |= dalloc(&e->tile_cnt, e->bcap / kSmallTile + 2);
  rc |= dalloc(&e->tile_win, 2 * (e->bcap / kSmallTile + 2));
  rc |= dalloc(&e->blk_att, cap / kBlock + 2);
  rc |= dalloc(&e->blk_off, cap / kBlock + 2);
  rc |= dalloc(&e->d_sysp, 1);
  if (replay) {
    rc |= dalloc(&e->ndraw, scap / kRunTile + 2);
    rc |= dalloc(&e->ndraw_off, scap / kRunTile + 2);
  }
  rc |= dalloc(&e->d_stats, 1);
  return rc == FQ_OK ? FQ_OK : FQ_ERR_NOMEM;
}

template <class T>
int upload(T** dst, const T* src, int64_t count, hipStream_t st) {
  if (!src || count <= 0) {
    *dst = nullptr;
    return FQ_OK;
  }
  if (dalloc(dst, count) != FQ_OK) return FQ_ERR_NOMEM;
  FQ_HIP(hipMemcpyAsync(*dst, src, sizeof(T) * count, hipMemcpyHostToDevice, st));
  return FQ_OK;
}

}  // namespace

// ---------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------
extern "C" {

int fq_create(const fq_system* sys, const fq_params* params, fq_engine** out) {
  if (!sys || !params || !out) return FQ_ERR_ARG;
  if (sys->nwords < 1 || sys->nwords > FQ_MAX_WORDS || params->nspaces < 1 || params->nspaces > FQ_MAX_SPACES)
    return FQ_ERR_ARG;
  if (sys->system == FQ_SYS_READ_IN && sys->nsym_pg > 8) return FQ_ERR_ARG;
  if (params->excit_gen < FQ_EXCIT_RENORM || params->excit_gen > FQ_EXCIT_LEARNED) return FQ_ERR_ARG;
  if ((params->excit_gen == FQ_EXCIT_HEAT_BATH || params->excit_gen == FQ_EXCIT_LEARNED) &&
      (sys->system != FQ_SYS_READ_IN || sys->nel > fqd::kHbMaxNel))
    return FQ_ERR_ARG;
  if (params->excit_gen == FQ_EXCIT_LEARNED && (params->rng_mode != FQ_RNG_PHILOX || params->proposal_mix < 0.0 ||
                                                 params->proposal_mix > 1.0 || params->proposal_min_attempts < 0))
    return FQ_ERR_ARG;
  if (sys->system == FQ_SYS_READ_IN && params->excit_gen == FQ_EXCIT_NO_RENORM) return FQ_ERR_ARG;
  if (params->main_capacity < 1 || params->spawn_capacity < 1) return FQ_ERR_ARG;
  // (determinant, space) entries are addressed relative to a window in 32 bits
  if (params->main_capacity * params->nspaces >= (int64_t{1} << 31)) return FQ_ERR_ARG;
  if (params->spawn_capacity > 0xffffffffLL) return FQ_ERR_ARG;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= params->device) return FQ_ERR_NO_DEVICE;
  auto* e = new fq_engine();
  e->device = params->device;
  if (hipSetDevice(e->device) != hipSuccess) {
    delete e;
    return FQ_ERR_NO_DEVICE;
  }
  if (params->excit_gen == FQ_EXCIT_HEAT_BATH && !hb_lds_fits(e->device, sys->nel)) {
    delete e;
    return FQ_ERR_ARG;
  }
  if (params->excit_gen == FQ_EXCIT_LEARNED && !learned_lds_fits(e->device, sys->nwords, sys->nbasis)) {
    delete e;
    return FQ_ERR_ARG;
  }
  if (hipStreamCreate(&e->stream) != hipSuccess) {
    delete e;
    return FQ_ERR_DEVICE;
  }
  e->fixed_scratch = fixed_scratch_address(e->device);
  e->par = *params;
  e->W = sys->nwords;
  e->S = params->nspaces;
  e->key_bits = sys->nbasis;
  e->cap = params->main_capacity;
  e->scap = params->spawn_capacity;
  Sys& s = e->sys;
  s.system = sys->system;
  s.nbasis = sys->nbasis;
  s.nel = sys->nel;
  s.nalpha = sys->nalpha;
  s.nbeta = sys->nbeta;
  s.nvirt = sys->nvirt;
  s.nvirt_alpha = sys->nvirt_alpha;
  s.nvirt_beta = sys->nvirt_beta;
  s.W = sys->nwords;
  s.S = params->nspaces;
  for (int w = 0; w < FQ_MAX_WORDS; ++w) {
    s.f0[w] = w < sys->nwords ? sys->f0[w] : 0;
    const int bits = std::max(0, std::min(64, sys->nbasis - 64 * w));
    s.valid[w] = bits == 64 ? ~uint64_t{0} : ((uint64_t{1} << bits) - 1);
  }
  s.H00 = sys->H00;
  s.coulomb_k = sys->coulomb_k;
  s.nsym = sys->nsym;
  s.norb = sys->norb;
  s.nsym_pg = sys->nsym_pg;
  s.max_sym_spin = sys->max_sym_spin;
  s.ecore = sys->ecore;
  s.psingle = sys->pattempt_single;
  s.pdouble = sys->pattempt_double;
  s.initiator = params->initiator;
  s.quadrature = params->quadrature_initiator;
  s.real_amps = params->real_amplitudes;
  s.excit_gen = params->excit_gen;
  s.initiator_pop = params->initiator_pop;
  s.rf = int64_t{1} << params->pop_bit_shift;
  s.spawn_cutoff = params->spawn_cutoff;
  int rc = FQ_OK;
  rc |= upload(&e->d_sp_eigv, sys->sp_eigv, sys->nbasis, e->stream);
  if (sys->system == FQ_SYS_HUB_K) {
    rc |= upload(&e->d_sym_table, sys->sym_table, static_cast<int64_t>(sys->nsym) * sys->nsym, e->stream);
    rc |= upload(&e->d_inv_sym, sys->inv_sym, sys->nsym, e->stream);
    std::vector<uint8_t> diff;
    if (sys->nsym <= 255 && sys->sym_table && sys->inv_sym) {  // labels in a byte: at most 64 of them
      diff.resize(static_cast<size_t>(sys->nsym) * sys->nsym);
      for (int c = 0; c < sys->nsym; ++c)
        for (int p = 0; p < sys->nsym; ++p) {
          const int inv = sys->inv_sym[p];
          diff[c * sys->nsym + p] =
              inv >= 1 && inv <= sys->nsym ? static_cast<uint8_t>(sys->sym_table[c * sys->nsym + inv - 1]) : 0;
        }
    }
    if (rc == FQ_OK) rc = upload(&e->d_sym_diff, diff.data(), static_cast<int64_t>(diff.size()), e->stream);
    if (rc == FQ_OK) FQ_HIP(hipStreamSynchronize(e->stream));
  } else {
    rc |= upload(&e->d_orb_sym, sys->orb_sym, sys->nbasis, e->stream);
    rc |= upload(&e->d_nbss, sys->nbasis_sym_spin, 2 * sys->nsym_pg, e->stream);
    rc |= upload(&e->d_ssbf, sys->sym_spin_basis_fns, 2 * sys->nsym_pg * sys->max_sym_spin, e->stream);
    e->cls_sorted = sys->sym_spin_basis_fns && sys->nbasis_sym_spin ? 1 : 0;
    for (int c = 0; e->cls_sorted && c < 2 * sys->nsym_pg; ++c)
      for (int k = 1; k < sys->nbasis_sym_spin[c]; ++k)
        if (sys->sym_spin_basis_fns[c * sys->max_sym_spin + k] <= sys->sym_spin_basis_fns[c * sys->max_sym_spin + k - 1])
          e->cls_sorted = 0;
    rc |= upload(&e->d_h1, sys->h1, static_cast<int64_t>(sys->norb) * sys->norb, e->stream);
    rc |= upload(&e->d_eri, sys->eri, sys->n_eri, e->stream);
    // Dense Coulomb/exchange pair tables for the diagonal rule: entries copied
    // from the packed store (same values, no re-computation).
    const int no = sys->norb;
    std::vector<double> J(static_cast<size_t>(no) * no), K(static_cast<size_t>(no) * no);
    auto tri = [](int64_t i, int64_t j) { return (i * (i - 1)) / 2 + j; };
    auto idx = [&](int p, int q, int r, int t) {  // (pq|rt) packed, 1-based spatial
      const int64_t a = p >= q ? tri(p, q) : tri(q, p), b = r >= t ? tri(r, t) : tri(t, r);
      return (a >= b ? tri(a, b) : tri(b, a)) - 1;
    };
    for (int pp = 1; pp <= no; ++pp)
      for (int qq = 1; qq <= no; ++qq) {
        J[(pp - 1) * no + (qq - 1)] = sys->eri[idx(pp, pp, qq, qq)];  // <ij|ij> = (ii|jj)
        K[(pp - 1) * no + (qq - 1)] = sys->eri[idx(pp, qq, qq, pp)];  // <ij|ji> = (ij|ji)
      }
    // Single-excitation tables: (pa|oo) and (po|oa) for every spatial p, a, o.
    std::vector<double> S1J(static_cast<size_t>(no) * no * no), S1K(S1J.size());
    for (int pp = 1; pp <= no; ++pp)
      for (int aa = 1; aa <= no; ++aa)
        for (int oo = 1; oo <= no; ++oo) {
          const size_t t = (static_cast<size_t>(pp - 1) * no + (aa - 1)) * no + (oo - 1);
          S1J[t] = sys->eri[idx(pp, aa, oo, oo)];
          S1K[t] = sys->eri[idx(pp, oo, oo, aa)];
        }
    if (rc == FQ_OK) rc = upload(&e->d_jmat, J.data(), static_cast<int64_t>(J.size()), e->stream);
    if (rc == FQ_OK) rc = upload(&e->d_kmat, K.data(), static_cast<int64_t>(K.size()), e->stream);
    if (rc == FQ_OK) rc = upload(&e->d_s1j, S1J.data(), static_cast<int64_t>(S1J.size()), e->stream);
    if (rc == FQ_OK) rc = upload(&e->d_s1k, S1K.data(), static_cast<int64_t>(S1K.size()), e->stream);
    // Host-evaluated divisions and square roots of the generators' integer
    // arguments (IEEE division and sqrt are correctly rounded on both sides).
    std::vector<double> R(kRecipN, 0.0);
    for (int k = 1; k < kRecipN; ++k) R[k] = 1.0 / static_cast<double>(k);
    const int npairs = sys->nel * (sys->nel - 1) / 2;
    std::vector<int> JP(static_cast<size_t>(npairs) + 2, 0);
    for (int ind = 1; ind <= npairs + 1; ++ind) JP[ind] = static_cast<int>(1.50 + std::sqrt(2 * ind - 1.750));
    if (rc == FQ_OK) rc = upload(&e->d_recip, R.data(), kRecipN, e->stream);
    if (rc == FQ_OK) rc = upload(&e->d_jpair, JP.data(), static_cast<int64_t>(JP.size()), e->stream);
    if (rc == FQ_OK) FQ_HIP(hipStreamSynchronize(e->stream));
  }
  s.sp_eigv = e->d_sp_eigv;
  s.sym_table = e->d_sym_table;
  s.inv_sym = e->d_inv_sym;
  s.sym_diff = e->d_sym_diff;
  s.orb_sym = e->d_orb_sym;
  s.nbss = e->d_nbss;
  s.ssbf = e->d_ssbf;
  s.h1 = e->d_h1;
  s.eri = e->d_eri;
  s.jmat = e->d_jmat;
  s.kmat = e->d_kmat;
  s.s1j = e->d_s1j;
  s.s1k = e->d_s1k;
  s.recip = e->d_recip;
  s.nrecip = e->d_recip ? kRecipN : 0;
  s.jpair = e->d_jpair;
  if (rc == FQ_OK) rc = setup_rank_keys(e);
  if (rc == FQ_OK && (params->excit_gen == FQ_EXCIT_HEAT_BATH || params->excit_gen == FQ_EXCIT_LEARNED))
    rc = build_heat_bath(e);
  if (rc == FQ_OK && params->excit_gen == FQ_EXCIT_LEARNED) rc = setup_learned(e);
  if (rc == FQ_OK) rc = set_insert_lds();
  if (rc == FQ_OK) rc = alloc_engine(e);
  if (rc == FQ_OK) rc = setup_sort(e);
  if (int khz = 0; rc == FQ_OK && hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, e->device) == hipSuccess &&
                   khz > 0)
    e->ms_per_tick = 1.0 / khz;
  if (rc == FQ_OK && hipEventCreateWithFlags(&e->ev_len, hipEventDisableTiming) != hipSuccess) rc = FQ_ERR_DEVICE;
  if (rc == FQ_OK && hipHostMalloc(reinterpret_cast<void**>(&e->h_len), 4 * sizeof(int64_t)) != hipSuccess)
    rc = FQ_ERR_NOMEM;
  if (rc == FQ_OK && hipHostMalloc(reinterpret_cast<void**>(&e->h_pin), sizeof(Stats)) != hipSuccess)
    rc = FQ_ERR_NOMEM;
  if (rc != FQ_OK) {
    fq_destroy(e);
    return rc;
  }
  if (hipStreamSynchronize(e->stream) != hipSuccess) {
    fq_destroy(e);
    return FQ_ERR_DEVICE;
  }
  *out = e;
  return FQ_OK;
}

DetermDev determ_dev(const fq_engine* e) {
  return DetermDev{e->d_drow, e->d_dcol, e->d_dmat, e->d_dvec, e->d_dpos, e->ndeterm, e->determ_separate};
}

void release_determ(fq_engine* e) {
  dfree(e->d_determ);
  dfree(e->d_drow);
  dfree(e->d_dcol);
  dfree(e->d_dmat);
  dfree(e->d_dvec);
  dfree(e->d_dpos);
  if (e->sys.ndeterm > 0) e->sys_dirty = true;
  e->ndeterm = 0;
  e->determ_nnz = 0;
  e->sys.determ = nullptr;
  e->sys.ndeterm = 0;
}

int fq_load(fq_engine* e, const uint64_t* states, const int64_t* pops, const double* dat, int64_t n) {
  if (!e || n < 0 || (n > 0 && (!states || !pops || !dat))) return FQ_ERR_ARG;
  if (n > e->cap) return FQ_ERR_CAPACITY;
  FQ_HIP(hipSetDevice(e->device));
  const int W = e->W, S = e->S;
  std::vector<uint64_t> dw(static_cast<size_t>(W) * n);
  std::vector<int64_t> dp(static_cast<size_t>(S) * n);
  for (int64_t i = 0; i < n; ++i) {
    for (int w = 0; w < W; ++w) dw[w * n + i] = states[i * W + w];
    for (int s = 0; s < S; ++s) dp[s * n + i] = pops[i * S + s];
  }
  e->cur = 0;
  for (int w = 0; w < W && n > 0; ++w)
    FQ_HIP(hipMemcpyAsync(e->det[0] + w * e->cap, dw.data() + w * n, 8 * n, hipMemcpyHostToDevice, e->stream));
  for (int s = 0; s < S && n > 0; ++s)
    FQ_HIP(hipMemcpyAsync(e->pop + s * e->cap, dp.data() + s * n, 8 * n, hipMemcpyHostToDevice, e->stream));
  if (n > 0) FQ_HIP(hipMemcpyAsync(e->kii[0], dat, 8 * n, hipMemcpyHostToDevice, e->stream));
  if (n > 0 && e->rank_words)
    hipLaunchKernelGGL(k_rank_list, dim3(grid_for(n)), dim3(kBlock), 0, e->stream, key_plan(e), W, n, e->cap,
                       e->det[0], e->mrank[0]);
  FQ_HIP(hipStreamSynchronize(e->stream));
  e->n = n;
  e->att_bound = -1;
  e->last_ns = -1;
  release_determ(e);  // a new list: no semi-stochastic core until fq_semi_stoch_init
  return FQ_OK;
}

// init_semi_stoch_t with space "high" (src/semi_stoch.F90:134-377,
// create_high_pop_space :1198-1316, find_most_populated_dets :1318-1385):
// the target_size most populated entries of the current list (sum over
// spaces of |N|).  The reference keeps them with a replace-the-minimum scan
// (a later entry replaces the first smallest kept one when strictly larger);
// a min-heap ordered by (population, slot) replaces the same entries.  The
// core is kept sorted as the main list (every core determinant is in it, so
// add_determ_dets_to_psip_list inserts nothing) and its Hamiltonian is built
// on the device (create_determ_hamil :533-685).
int fq_semi_stoch_init(fq_engine* e, int64_t target_size, int separate) {
  if (!e || target_size < 0 || e->batched || e->pending) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  FQ_HIP(hipStreamSynchronize(e->stream));
  release_determ(e);
  const int64_t n = e->n, nd = std::min(target_size, n);
  if (nd == 0) return FQ_OK;
  if (nd > INT32_MAX) return FQ_ERR_ARG;  // column indices are 32-bit
  const int W = e->W, S = e->S, c = e->cur;
  hipStream_t st = e->stream;
  std::vector<int64_t> pw(static_cast<size_t>(S) * n);
  std::vector<uint64_t> dw(static_cast<size_t>(W) * n);
  for (int sp = 0; sp < S; ++sp)
    FQ_HIP(hipMemcpyAsync(pw.data() + sp * n, e->pop + sp * e->cap, 8 * n, hipMemcpyDeviceToHost, st));
  for (int w = 0; w < W; ++w)
    FQ_HIP(hipMemcpyAsync(dw.data() + w * n, e->det[c] + w * e->cap, 8 * n, hipMemcpyDeviceToHost, st));
  FQ_HIP(hipStreamSynchronize(st));
  auto absum = [&](int64_t i) {
    int64_t t = 0;
    for (int sp = 0; sp < S; ++sp) t += std::llabs(pw[sp * n + i]);
    return t;
  };
  using Slot = std::pair<int64_t, int64_t>;  // (population, slot)
  std::priority_queue<Slot, std::vector<Slot>, std::greater<Slot>> heap;
  std::vector<int64_t> idx(nd);
  for (int64_t i = 0; i < nd; ++i) {
    idx[i] = i;
    heap.push({absum(i), i});
  }
  for (int64_t i = nd; i < n; ++i) {
    const int64_t a = absum(i);
    if (a > heap.top().first) {
      const int64_t slot = heap.top().second;
      heap.pop();
      idx[slot] = i;
      heap.push({a, slot});
    }
  }
  std::sort(idx.begin(), idx.end());  // list order
  std::vector<uint64_t> core(static_cast<size_t>(W) * nd);
  for (int w = 0; w < W; ++w)
    for (int64_t k = 0; k < nd; ++k) core[w * nd + k] = dw[w * n + idx[k]];
  int rc = dalloc(&e->d_determ, W * nd);
  rc |= dalloc(&e->d_drow, nd + 1);
  rc |= dalloc(&e->d_dvec, 2 * nd * S);  // populations, then (separate) the projected amplitudes
  rc |= dalloc(&e->d_dpos, nd);
  int64_t* cnt = nullptr;
  rc |= dalloc(&cnt, nd);
  if (rc != FQ_OK) {
    dfree(cnt);
    release_determ(e);
    return FQ_ERR_NOMEM;
  }
  FQ_HIP(hipMemcpyAsync(e->d_determ, core.data(), 8 * W * nd, hipMemcpyHostToDevice, st));
  e->sys.determ = e->d_determ;
  e->sys.ndeterm = nd;
  e->sys_dirty = true;
  const int transp = separate ? 1 : 0;
  hipLaunchKernelGGL(k_determ_count, dim3(static_cast<unsigned>(nd)), dim3(kBlock), 0, st, e->sys, transp, cnt);
  rc = scan_exclusive(e, cnt, e->d_drow, nd);
  int64_t nnz = 0;
  if (rc == FQ_OK) {
    FQ_HIP(hipMemcpyAsync(&nnz, e->d_drow + nd, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    FQ_HIP(hipStreamSynchronize(st));
    rc = dalloc(&e->d_dcol, nnz) | dalloc(&e->d_dmat, nnz);
  }
  if (rc == FQ_OK) {
    hipLaunchKernelGGL(k_determ_fill, dim3(static_cast<unsigned>(nd)), dim3(kBlock), 0, st, e->sys, transp,
                       e->d_drow, e->d_dcol, e->d_dmat);
    if (hipStreamSynchronize(st) != hipSuccess) rc = FQ_ERR_DEVICE;
  }
  dfree(cnt);
  if (rc != FQ_OK) {
    release_determ(e);
    return rc == FQ_ERR_DEVICE ? rc : FQ_ERR_NOMEM;
  }
  e->ndeterm = nd;
  e->determ_nnz = nnz;
  e->determ_separate = transp;
  return FQ_OK;
}

int fq_semi_stoch_info(fq_engine* e, int64_t* ndeterm, int64_t* nnz, uint64_t* states, int64_t capacity) {
  if (!e || !ndeterm) return FQ_ERR_ARG;
  *ndeterm = e->ndeterm;
  if (nnz) *nnz = e->determ_nnz;
  if (!states || e->ndeterm == 0) return FQ_OK;
  if (capacity < e->ndeterm) return FQ_ERR_CAPACITY;
  FQ_HIP(hipSetDevice(e->device));
  std::vector<uint64_t> dw(static_cast<size_t>(e->W) * e->ndeterm);
  FQ_HIP(hipMemcpyAsync(dw.data(), e->d_determ, 8 * dw.size(), hipMemcpyDeviceToHost, e->stream));
  FQ_HIP(hipStreamSynchronize(e->stream));
  for (int64_t k = 0; k < e->ndeterm; ++k)
    for (int w = 0; w < e->W; ++w) states[k * e->W + w] = dw[w * e->ndeterm + k];
  return FQ_OK;
}

int fq_push_rng(fq_engine* e, const double* draws, int64_t n) {
  if (!e || n < 0 || (n > 0 && !draws)) return FQ_ERR_ARG;
  if (n == 0) return FQ_OK;
  FQ_HIP(hipSetDevice(e->device));
  int rc = reserve_rng(e, n);
  if (rc != FQ_OK) return rc;
  FQ_HIP(hipMemcpyAsync(e->rng_buf + e->rng_end, draws, sizeof(double) * n, hipMemcpyHostToDevice, e->stream));
  FQ_HIP(hipStreamSynchronize(e->stream));
  e->rng_end += n;
  return FQ_OK;
}

int fq_rng_available(fq_engine* e, int64_t* n) {
  if (!e || !n) return FQ_ERR_ARG;
  *n = e->rng_end - e->rng_pos;
  return FQ_OK;
}

static int cycle_body(fq_engine* e, const double* shift, const double* eproj_old, double tau, fq_cycle_out* out) {
  if (!e || !shift || !eproj_old || !out || e->batched) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  const bool replay = e->par.rng_mode == FQ_RNG_REPLAY;
  const int64_t n = e->n, cap = e->cap;
  const int c = e->cur;
  hipStream_t st = e->stream;
  const uint32_t cyc = static_cast<uint32_t>(e->cycle_index++);
  const double sh1 = e->S > 1 ? shift[1] : 0.0, e1 = e->S > 1 ? eproj_old[1] : 0.0;
  if (replay)  // production: the determinant pass clears the counters
    hipLaunchKernelGGL(k_zero, dim3(1), dim3(kBlock), 0, st, reinterpret_cast<int64_t*>(e->d_stats),
                       static_cast<int64_t>(sizeof(Stats) / sizeof(int64_t)));
  int64_t rng_pos = e->rng_pos;
  int64_t ns = 0;
  int est_blocks = 0;
  if (replay) {
    hipLaunchKernelGGL(k_replay_walk, dim3(1), dim3(1), 0, st, e->sys, n, cap, e->det[c], e->pop, e->kii[c],
                       e->pop_new, tau, shift[0], sh1, eproj_old[0], e1, e->rng_buf, e->rng_pos, e->rng_end, e->scap,
                       e->sdet, e->srec, e->d_stats, determ_dev(e));
    int rc = sync_stats(e);
    if (rc != FQ_OK) return rc;
    if (e->h_stats.rng_failed) return FQ_ERR_RNG_EXHAUSTED;
    rng_pos = e->h_stats.rng_pos;
    ns = e->h_stats.nspawn;
  } else {
    if (e->online_every > 0 && n > 0 && cyc % static_cast<uint32_t>(e->online_every) == 0) {
      // online training from the current list: this cycle already uses the update
      fqm::Mlp& m = e->mlp;
      for (int32_t k = 0; k < e->online_steps; ++k) {
        int trc = fqm::mlp_sample(m, e->sys, e->det[c], e->pop, cap, n, e->online_batch,
                                  static_cast<int64_t>(e->par.proposal_min_attempts),
                                  e->par.philox_seed ^ 0x6a09e667f3bcc908ull, static_cast<uint32_t>(m.adam_t), st,
                                  scan_cb, e);
        if (trc == FQ_OK) trc = fqm::mlp_train_step(m, e->sys, e->online_batch, e->online_lr, true, st);
        if (trc != FQ_OK) return trc;
      }
      ++e->online_runs;
    }
    const unsigned nb = grid_for(n);
    hipLaunchKernelGGL(e->S == 1 ? k_det_pass<1> : k_det_pass<2>, dim3(nb), dim3(kBlock), 0, st, e->sys, n, cap, e->det[c], e->pop, e->kii[c],
                       e->pop_new, att_counts(e), parent_flags(e), tau, shift[0], sh1, eproj_old[0], e1, e->par.philox_seed, cyc,
                       e->part_d, e->part_i, e->d_dvec, e->d_dpos, e->blk_att, e->d_stats);
    est_blocks = static_cast<int>(nb);
    if (e->par.excit_gen == FQ_EXCIT_LEARNED && n > 0) {
      const int64_t min_att = e->par.proposal_min_attempts, mt = ceil_div(n, kMainTile);
      // A bound of the rows: every determinant without a threshold; else at most
      // one per min_att of the attempts, where these are bounded (see the
      // spawning below), so that the host need not wait for the count (the
      // wait and the three kernels of its scan took 50 us of a cycle with 1e6
      // walkers, the two kernels here take 10).  It waits where the attempts are
      // unknown, or the table would have to grow past kProposalTable for the
      // bound alone or finds no memory to: then it follows the rows present.
      const int64_t bound_rows = kProposalTable / (static_cast<int64_t>(sizeof(float)) * e->mlp.d_out);
      int64_t rows = n;
      bool count = false;
      if (min_att > 0) {
        if (e->att_bound > 0) rows = std::min(n, e->att_bound / min_att);
        count = e->att_bound <= 0 || (rows > e->mlp_tab_rows && rows > bound_rows);
      }
      hipLaunchKernelGGL(k_mlp_mark, dim3(static_cast<unsigned>(mt)), dim3(kBlock), 0, st, n, e->S, att_counts(e), min_att,
                         e->mcnt, e->d_stats);
      if (mt > e->prefix_runs) {
        const int mrc = scan_exclusive(e, e->mcnt, e->moff, mt);
        if (mrc != FQ_OK) return mrc;
      }
      hipLaunchKernelGGL(k_mlp_rows, dim3(static_cast<unsigned>(mt)), dim3(kBlock), 0, st, n, e->S, att_counts(e), min_att,
                         rows, e->mcnt, mt > e->prefix_runs ? e->moff : nullptr, e->mlp_row, e->mlp_idx, e->d_stats);
      if (min_att > 0 && !count && rows > e->mlp_tab_rows)
        count = grow_proposal_table(e, std::max(rows, std::min(2 * e->mlp_tab_rows, bound_rows)), true) != FQ_OK;
      if (count) {
        FQ_HIP(hipMemcpyAsync(&rows, &e->d_stats->mlp_rows, sizeof(int64_t), hipMemcpyDeviceToHost, st));
        FQ_HIP(hipStreamSynchronize(st));
      }
      if (rows > e->mlp_tab_rows) {  // rare: rows follow the inferred determinants
        const int grc = grow_proposal_table(e, std::max(rows, 2 * e->mlp_tab_rows), false);
        if (grc != FQ_OK) return grc;
      }
      const int mrc = fqm::mlp_infer(e->mlp, e->sys, e->det[c], cap, rows, e->mlp_tab, st, e->mlp_idx,
                                     &e->d_stats->mlp_rows, e->prof.proposal_rows);
      if (mrc != FQ_OK) return mrc;
    }
    // Attempt offsets over the n*S (det, space) entries.
    const int64_t nent = e->S * n;
    // The spawning launches cover attempts [0, bound): after a production
    // cycle the host holds a bound of this cycle's total (every entry makes at
    // most floor(|N|) + 1 attempts, |N| for integer populations), so it need
    // not wait for the prefix sum; otherwise it reads the total.  The kernels
    // clamp to the total on the device.
    int64_t bound = e->att_bound;
    const int gen = fqd::gen_of(e->sys.system, e->sys.excit_gen);
    const int tile = bound > 0 && bound <= e->bcap ? spawn_tile(gen, bound) : kSpawnTile;  // batches: k_tile_bounds' tiles
    int rc = scan_attempts(e, nent, bound > 0 ? std::min(bound, e->bcap) : e->bcap, tile);
    if (rc != FQ_OK) return rc;
    if (bound <= 0) {  // unknown (or an empty list): the exact total
      FQ_HIP(hipMemcpyAsync(&bound, att_offsets(e) + nent, sizeof(int64_t), hipMemcpyDeviceToHost, st));
      FQ_HIP(hipStreamSynchronize(st));
    }
    e->spawn_launches = 0;
    if (int rs = sync_sysp(e); rs != FQ_OK) return rs;
    const bool one_batch = bound <= e->bcap;
    auto kern = tile == kSmallTile ? spawn_kernel<false, kSmallTile>(gen) : spawn_kernel<false, kSpawnTile>(gen);
    const size_t lds = gen == fqd::kGenHeatBath    ? hb_lds_bytes(e->sys.nel)
                       : gen == fqd::kGenMolRenorm ? sizeof(uint64_t) * e->W * tile
                       : gen == fqd::kGenLearned   ? learned_lds_bytes(e->W, e->sys.nbasis, tile)
                                                   : 0;
    for (int64_t tb = 0; tb < bound; tb += e->bcap) {
      const int64_t te = std::min(bound, tb + e->bcap);
      const int64_t nt = ceil_div(te - tb, tile);
      ++e->spawn_launches;
      if (!one_batch)
        hipLaunchKernelGGL(k_tile_bounds, dim3(grid_for(nt)), dim3(kBlock), 0, st, nent, att_offsets(e), tb, te,
                           e->tile_win);
      hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(spawn_grid(gen, nt))), dim3(kBlock), lds, st,
                         e->d_sysp, nent, cap, tb, te, att_offsets(e), e->det[c], e->pop, tau, e->par.philox_seed, cyc,
                         e->bcap, e->st_det, e->st_pop, e->st_ent, e->tile_cnt, e->tile_win, parent_flags(e), nullptr,
                         nullptr, nullptr, nullptr, e->d_stats);
      pack_spawned(e, te - tb, tile, one_batch, att_offsets(e) + nent);
    }
    int64_t ndet_entries = 0;  // the deterministic projection's spawned entries (combined annihilation)
    if (e->ndeterm > 0) {
      const int64_t m = e->ndeterm * e->S;
      hipLaunchKernelGGL(k_determ_proj, dim3(grid_for(m, kBlock / 64)), dim3(kBlock), 0, st, e->sys, key_plan(e), determ_dev(e),
                         tau, shift[0], sh1, eproj_old[0], e1, e->par.philox_seed, cyc, cap, e->pop_new,
                         e->kbuf[0], e->pbuf[0], e->scap, e->d_stats);
      if (!e->determ_separate) {
        hipLaunchKernelGGL(k_add_nspawn, dim3(1), dim3(1), 0, st, e->d_stats, m);
        ndet_entries = m;
      }
    }
    e->keys_ready = true;  // the packing kernels wrote the sort keys
    // The spawned-list length and the attempt total are copied to pinned host
    // memory behind the spawning kernels; the radix passes read the length on
    // the device (their grids sized by a bound: successes <= attempts <=
    // bound), so the host waits for the copy only once they are queued, and
    // the device does not idle meanwhile.  Lists bounded by kNoWaitMax are not
    // waited for at all.
    if (bound + ndet_entries > kNoWaitMax) {
      FQ_HIP(hipMemcpyAsync(e->h_len, &e->d_stats->nspawn, 3 * sizeof(int64_t), hipMemcpyDeviceToHost, st));
      FQ_HIP(hipEventRecord(e->ev_len, st));
    }
    e->spawn_bound = bound;
    ns = std::min<int64_t>(bound + ndet_entries, e->scap);
  }
  int rc = annihilate(e, ns, replay ? nullptr : &e->d_stats->nspawn, replay, cyc, rng_pos, est_blocks);
  if (rc != FQ_OK) return rc;
  // the attempts cannot exceed the bound the spawning launches covered (see sort_and_reduce)
  if (!replay && e->h_stats.total_attempts > e->spawn_bound) return FQ_ERR_DEVICE;
  ns = std::min<int64_t>(e->h_stats.nspawn, e->scap);
  if (!replay) {  // next cycle's attempts <= sum floor(|N|) (+1 per entry with real amplitudes)
    unsigned long long sum = 0;
    for (int sp = 0; sp < e->S; ++sp) sum += e->h_stats.abs_pop[sp];
    e->att_bound = static_cast<int64_t>(sum / static_cast<unsigned long long>(e->sys.rf)) +
                   (e->sys.real_amps ? e->n * e->S : 0);
  }
  const int64_t used = rng_pos - e->rng_pos;
  e->rng_pos = rng_pos;
  fill_profile(e, n, ns);
  e->prof.proposal_rows = e->par.excit_gen == FQ_EXCIT_LEARNED && !replay ? e->h_stats.mlp_rows : 0;
  if (replay) e->prof.spawn_launches = 0;
  fill_out(e, out, used);
  return FQ_OK;
}

int fq_cycle(fq_engine* e, const double* shift, const double* eproj_old, double tau, fq_cycle_out* out) {
  if (e && e->pending) return FQ_ERR_ARG;
  return cycle_body(e, shift, eproj_old, tau, out);
}

int fq_cycle_spawn(fq_engine* e, const double* shift, const double* eproj_old, double tau, fq_cycle_out* out) {
  if (!e || !shift || !eproj_old || !out || e->batched || e->pending) return FQ_ERR_ARG;
  if (e->par.rng_mode != FQ_RNG_REPLAY) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  const int c = e->cur;
  hipStream_t st = e->stream;
  const uint32_t cyc = static_cast<uint32_t>(e->cycle_index++);
  const double sh1 = e->S > 1 ? shift[1] : 0.0, e1 = e->S > 1 ? eproj_old[1] : 0.0;
  hipLaunchKernelGGL(k_zero, dim3(1), dim3(kBlock), 0, st, reinterpret_cast<int64_t*>(e->d_stats),
                     static_cast<int64_t>(sizeof(Stats) / sizeof(int64_t)));
  hipLaunchKernelGGL(k_replay_walk, dim3(1), dim3(1), 0, st, e->sys, e->n, e->cap, e->det[c], e->pop, e->kii[c],
                     e->pop_new, tau, shift[0], sh1, eproj_old[0], e1, e->rng_buf, e->rng_pos, e->rng_end, e->scap,
                     e->sdet, e->srec, e->d_stats, determ_dev(e));
  int rc = sync_stats(e);
  if (rc != FQ_OK) return rc;
  if (e->h_stats.rng_failed) return FQ_ERR_RNG_EXHAUSTED;
  e->pending = true;
  e->pend_cyc = cyc;
  e->pend_rng_pos = e->h_stats.rng_pos;
  e->pend_ns = std::min<int64_t>(e->h_stats.nspawn, e->scap);
  e->pend_stats = e->h_stats;
  std::memset(out, 0, sizeof(*out));
  for (int sp = 0; sp < e->S; ++sp) {
    out->proj_energy[sp] = e->h_stats.proj[sp];
    out->D0_population[sp] = e->h_stats.d0[sp];
  }
  out->nspawn_events = e->pend_ns;
  out->ndeath = e->h_stats.ndeath;
  out->nattempts = e->h_stats.total_attempts;
  out->rng_consumed = e->pend_rng_pos - e->rng_pos;
  out->spawn_overflow = e->h_stats.spawn_overflow ? 1 : 0;
  return FQ_OK;
}

int fq_spawned_list(fq_engine* e, uint64_t* states, int64_t* pops, int64_t* flags, int64_t capacity, int64_t* n) {
  if (!e || !n || !e->pending) return FQ_ERR_ARG;
  const int64_t ns = e->pend_ns;
  *n = ns;
  if (capacity < ns) return FQ_ERR_CAPACITY;
  if (ns == 0) return FQ_OK;
  FQ_HIP(hipSetDevice(e->device));
  const int W = e->W, S = e->S, RS = rec_stride(S);
  std::vector<uint64_t> dw(static_cast<size_t>(W) * ns);
  std::vector<int64_t> rec(static_cast<size_t>(RS) * ns);
  for (int w = 0; w < W; ++w)
    FQ_HIP(hipMemcpyAsync(dw.data() + w * ns, e->sdet + w * e->scap, 8 * ns, hipMemcpyDeviceToHost, e->stream));
  FQ_HIP(hipMemcpyAsync(rec.data(), e->srec, 8 * RS * ns, hipMemcpyDeviceToHost, e->stream));
  FQ_HIP(hipStreamSynchronize(e->stream));
  for (int64_t i = 0; i < ns; ++i) {
    if (states)
      for (int w = 0; w < W; ++w) states[i * W + w] = dw[w * ns + i];
    if (pops)
      for (int sp = 0; sp < S; ++sp) pops[i * S + sp] = rec[i * RS + sp];
    if (flags) flags[i] = rec[i * RS + S];
  }
  return FQ_OK;
}

int fq_cycle_finish(fq_engine* e, const uint64_t* sstates, const int64_t* spops, const int64_t* sflags, int64_t ns,
                    fq_cycle_out* out) {
  if (!e || !out || !e->pending || ns < 0 || (ns > 0 && (!sstates || !spops))) return FQ_ERR_ARG;
  if (ns > e->scap) return FQ_ERR_CAPACITY;
  FQ_HIP(hipSetDevice(e->device));
  const int W = e->W, S = e->S, RS = rec_stride(S);
  std::vector<uint64_t> dw(static_cast<size_t>(W) * std::max<int64_t>(ns, 1));
  std::vector<int64_t> rec(static_cast<size_t>(RS) * std::max<int64_t>(ns, 1), 0);
  for (int64_t i = 0; i < ns; ++i) {
    for (int w = 0; w < W; ++w) dw[w * ns + i] = sstates[i * W + w];
    for (int sp = 0; sp < S; ++sp) rec[i * RS + sp] = spops[i * S + sp];
    rec[i * RS + S] = (sflags && e->par.initiator) ? sflags[i] : 0;
  }
  hipStream_t st = e->stream;
  for (int w = 0; w < W && ns > 0; ++w)
    FQ_HIP(hipMemcpyAsync(e->sdet + w * e->scap, dw.data() + w * ns, 8 * ns, hipMemcpyHostToDevice, st));
  if (ns > 0) FQ_HIP(hipMemcpyAsync(e->srec, rec.data(), 8 * RS * ns, hipMemcpyHostToDevice, st));
  e->pending = false;
  int64_t rng_pos = e->pend_rng_pos;
  int rc = annihilate(e, ns, nullptr, true, e->pend_cyc, rng_pos);
  if (rc != FQ_OK) return rc;
  const int64_t used = rng_pos - e->rng_pos;
  e->rng_pos = rng_pos;
  const Stats& k = e->pend_stats;
  for (int sp = 0; sp < S; ++sp) {
    e->h_stats.proj[sp] = k.proj[sp];
    e->h_stats.d0[sp] = k.d0[sp];
  }
  e->h_stats.nspawn = e->pend_ns;
  e->h_stats.ndeath = k.ndeath;
  e->h_stats.total_attempts = k.total_attempts;
  e->h_stats.spawn_overflow = k.spawn_overflow;
  fill_out(e, out, used);
  return FQ_OK;
}

int fq_cycle_noalloc(fq_engine* e, const double* shift, const double* eproj_old, double tau, fq_cycle_out* out) {
  if (!e || !shift || !eproj_old || !out || e->batched) return FQ_ERR_ARG;
  // replay streams and the learned proposal's weight table grow on demand
  if (e->par.rng_mode != FQ_RNG_PHILOX || e->par.excit_gen == FQ_EXCIT_LEARNED) return FQ_ERR_ARG;
  if (!e->fixed_scratch) return FQ_ERR_DEVICE;
  e->noalloc = true;
  e->scratch_short = false;
  const int rc = cycle_body(e, shift, eproj_old, tau, out);
  e->noalloc = false;
  if (e->scratch_short) {
    fprintf(stderr, "fqmc: fq_cycle_noalloc: this cycle needs more scratch than the fixed %lld bytes hold; "
            "the walker list is unchanged\n", static_cast<long long>(sizeof(int64_t) * kScratchElems));
    (void)hipStreamSynchronize(e->stream);
    return FQ_ERR_SCRATCH;
  }
  return rc;
}

int fq_annihilate(fq_engine* e, const uint64_t* sstates, const int64_t* spops, const int64_t* sflags, int64_t ns,
                  fq_cycle_out* out) {
  if (!e || !out || ns < 0 || (ns > 0 && (!sstates || !spops)) || e->pending) return FQ_ERR_ARG;
  if (ns > e->scap) return FQ_ERR_CAPACITY;
  FQ_HIP(hipSetDevice(e->device));
  const bool replay = e->par.rng_mode == FQ_RNG_REPLAY;
  const int W = e->W, S = e->S;
  const int64_t n = e->n, cap = e->cap;
  std::vector<uint64_t> dw(static_cast<size_t>(W) * std::max<int64_t>(ns, 1));
  const int RS = rec_stride(S);
  std::vector<int64_t> rec(static_cast<size_t>(RS) * std::max<int64_t>(ns, 1), 0);
  for (int64_t i = 0; i < ns; ++i) {
    for (int w = 0; w < W; ++w) dw[w * ns + i] = sstates[i * W + w];
    for (int s = 0; s < S; ++s) rec[i * RS + s] = spops[i * S + s];
    rec[i * RS + S] = (sflags && e->par.initiator) ? sflags[i] : 0;
  }
  hipStream_t st = e->stream;
  for (int w = 0; w < W && ns > 0; ++w)
    FQ_HIP(hipMemcpyAsync(e->sdet + w * e->scap, dw.data() + w * ns, 8 * ns, hipMemcpyHostToDevice, st));
  if (ns > 0) FQ_HIP(hipMemcpyAsync(e->srec, rec.data(), 8 * RS * ns, hipMemcpyHostToDevice, st));
  // post-death populations = current populations
  for (int s = 0; s < S && n > 0; ++s)
    FQ_HIP(hipMemcpyAsync(e->pop_new + s * cap, e->pop + s * cap, 8 * n, hipMemcpyDeviceToDevice, st));
  FQ_HIP(hipMemsetAsync(e->d_stats, 0, sizeof(Stats), st));
  FQ_HIP(hipStreamSynchronize(st));
  const uint32_t cyc = static_cast<uint32_t>(e->cycle_index++);
  int64_t rng_pos = e->rng_pos;
  int rc = annihilate(e, ns, nullptr, replay, cyc, rng_pos);
  if (rc != FQ_OK) return rc;
  const int64_t used = rng_pos - e->rng_pos;
  e->rng_pos = rng_pos;
  e->h_stats.nspawn = ns;
  fill_out(e, out, used);
  return FQ_OK;
}

int fq_nstates(fq_engine* e, int64_t* n) {
  if (!e || !n) return FQ_ERR_ARG;
  *n = e->n;
  return FQ_OK;
}

// Rows [r0, r1) of the list to the caller's arrays by way of one pinned slot,
// as many rows at a time as it holds.
static hipError_t copy_rows(fq_engine* e, int slot, int64_t r0, int64_t r1, uint64_t* states, int64_t* pops,
                            double* dat) {
  if (hipError_t err = hipSetDevice(e->device); err != hipSuccess) return err;
  const int W = e->W, S = e->S, c = e->cur;
  const int64_t rows = kListSlotBytes / (8 * (W + S + 1));
  uint64_t* buf = e->list_buf + slot * (kListSlotBytes / 8);
  const int q3 = slot % fq_engine::kListStreams;
  hipStream_t st = q3 == 0 ? e->stream : e->list_stream[q3];  // shared: each thread waits for its own copies only
  for (int64_t i = r0; i < r1; i += rows) {
    const int64_t m = std::min(rows, r1 - i);
    uint64_t* q = buf;
    auto fetch = [&](const void* from) {
      const hipError_t err = hipMemcpyAsync(q, from, 8 * m, hipMemcpyDeviceToHost, st);
      q += m;
      return err;
    };
    hipError_t err = hipSuccess;
    if (states)
      for (int w = 0; w < W && err == hipSuccess; ++w) err = fetch(e->det[c] + w * e->cap + i);
    if (pops)
      for (int sp = 0; sp < S && err == hipSuccess; ++sp) err = fetch(e->pop + sp * e->cap + i);
    if (dat && err == hipSuccess) err = fetch(e->kii[c] + i);
    if (err == hipSuccess) err = hipEventRecord(e->list_ev[slot], st);
    if (err == hipSuccess) err = hipEventSynchronize(e->list_ev[slot]);
    if (err != hipSuccess) return err;
    q = buf;
    auto place = [&](void* to, int n) {  // n arrays of m words, interleaved
      if (n == 1) {
        std::memcpy(static_cast<uint64_t*>(to) + i, q, 8 * m);
      } else {
        uint64_t* d = static_cast<uint64_t*>(to) + n * i;
        for (int64_t k = 0; k < m; ++k)
          for (int w = 0; w < n; ++w) d[n * k + w] = q[w * m + k];
      }
      q += n * m;
    };
    if (states) place(states, W);
    if (pops) place(pops, S);
    if (dat) place(dat, 1);
  }
  return hipSuccess;
}

// The list leaves through pinned slots, one per thread: each thread copies its
// part of the rows a slot at a time, so one thread's transfer runs while the
// others move theirs to the caller's (pageable) arrays.  (Copies to pageable
// temporaries and a second pass over them took 15.8 ms for 2.7e6 one-word
// entries and 8.4 ms for 1.0e6 two-word pairs; 2.3 and 1.7 ms now.)
int fq_download(fq_engine* e, uint64_t* states, int64_t* pops, double* dat, int64_t capacity, int64_t* nout) {
  if (!e || !nout) return FQ_ERR_ARG;
  const int64_t n = e->n;
  *nout = n;
  if (capacity < n) return FQ_ERR_CAPACITY;
  if (n == 0) return FQ_OK;
  std::lock_guard<std::mutex> lock(e->list_mutex);
  FQ_HIP(hipSetDevice(e->device));
  FQ_HIP(hipStreamSynchronize(e->stream));
  const int64_t bytes = 8 * n * (e->W + e->S + 1);
  const int nt = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(fq_engine::kListSlots, bytes / kListSlotBytes)));
  if (e->list_slots < nt) {
    if (e->list_buf) (void)hipHostFree(e->list_buf);
    e->list_buf = nullptr;
    e->list_slots = nt == 1 ? 1 : fq_engine::kListSlots;
    if (hipHostMalloc(reinterpret_cast<void**>(&e->list_buf), e->list_slots * kListSlotBytes) != hipSuccess) {
      e->list_buf = nullptr;
      e->list_slots = 0;
      return FQ_ERR_NOMEM;
    }
  }
  for (int t = 0; t < nt; ++t) {
    if (!e->list_ev[t]) FQ_HIP(hipEventCreateWithFlags(&e->list_ev[t], hipEventDisableTiming));
    const int q = t % fq_engine::kListStreams;
    if (q > 0 && !e->list_stream[q]) FQ_HIP(hipStreamCreateWithFlags(&e->list_stream[q], hipStreamNonBlocking));
  }
  hipError_t err[fq_engine::kListSlots] = {};
  std::thread th[fq_engine::kListSlots];
  auto part = [&](int t) { err[t] = copy_rows(e, t, n * t / nt, n * (t + 1) / nt, states, pops, dat); };
  for (int t = 1; t < nt; ++t) {
    try {
      th[t] = std::thread(part, t);
    } catch (const std::exception&) {  // no thread to be had: this one does the part below
    }
  }
  part(0);
  for (int t = 1; t < nt; ++t) {
    if (th[t].joinable())
      th[t].join();
    else
      part(t);
  }
  for (int t = 0; t < nt; ++t) FQ_HIP(err[t]);
  return FQ_OK;
}

int fq_last_profile(fq_engine* e, fq_profile_out* out) {
  if (!e || !out) return FQ_ERR_ARG;
  *out = e->prof;
  return FQ_OK;
}

int fq_last_timing(fq_engine* e, double* spawn_ms, double* annihilate_ms, double* total_ms) {
  if (!e) return FQ_ERR_ARG;
  if (spawn_ms) *spawn_ms = e->t_spawn;
  if (annihilate_ms) *annihilate_ms = e->t_annih;
  if (total_ms) *total_ms = e->t_total;
  return FQ_OK;
}

// ---- batched independent instances ---------------------------------------------
int fq_create_batch(const fq_system* systems, int32_t ninst, const fq_params* params, fq_engine** out) {
  if (!systems || !params || !out || ninst < 1 || ninst > kMaxInst) return FQ_ERR_ARG;
  if (params->rng_mode != FQ_RNG_PHILOX || params->real_amplitudes) return FQ_ERR_ARG;
  if (params->excit_gen == FQ_EXCIT_HEAT_BATH || params->excit_gen == FQ_EXCIT_LEARNED) return FQ_ERR_ARG;
  for (int k = 0; k < ninst; ++k)
    if (systems[k].nwords != 1 || systems[k].nbasis > kInstShift || systems[k].system != systems[0].system)
      return FQ_ERR_ARG;
  fq_engine* e = nullptr;
  int rc = fq_create(&systems[0], params, &e);
  if (rc != FQ_OK) return rc;
  e->batched = true;
  e->ninst = ninst;
  e->rank_words = 0;  // the instance index is part of the key: sort the encoded words
  int ib = 0;
  while ((1 << ib) < ninst) ++ib;
  e->key_bits = kInstShift + std::max(ib, 1);
  rc = setup_sort(e);
  if (rc != FQ_OK) {
    fq_destroy(e);
    return rc;
  }
  fq_params small = *params;
  small.main_capacity = small.spawn_capacity = 1;
  std::vector<Sys> hs(static_cast<size_t>(ninst));
  for (int k = 0; k < ninst && rc == FQ_OK; ++k) {
    fq_engine* sub = nullptr;
    rc = fq_create(&systems[k], &small, &sub);
    if (rc == FQ_OK) {
      e->subs.push_back(sub);
      hs[k] = sub->sys;
    }
  }
  const int64_t S = e->S;
  if (rc == FQ_OK) rc = upload(&e->d_sys_arr, hs.data(), ninst, e->stream);
  if (rc == FQ_OK) {
    rc |= dalloc(&e->d_ipar, (1 + 2 * S) * ninst);
    rc |= dalloc(&e->d_ibound, 2 * (ninst + 1));
    rc |= dalloc(&e->d_isb, ninst + 1);
    rc |= dalloc(&e->d_iatt, ninst);
    rc |= dalloc(&e->d_cterm, 2 * S * e->cap);
    rc |= dalloc(&e->d_cdeath, e->cap);
    e->ipb = e->cap / kBlock + ninst + 2;
    rc |= dalloc(&e->d_iblk_cnt, ninst + 1);
    rc |= dalloc(&e->d_iblk_off, ninst + 1);
    rc |= dalloc(&e->d_nblk_off, ninst + 1);
    rc |= dalloc(&e->d_ipart_d, 2 * S * e->ipb);
    rc |= dalloc(&e->d_ipart_i, (1 + S) * e->ipb);
    rc |= dalloc(&e->d_iout_d, 2 * S * ninst);
    rc |= dalloc(&e->d_iout_i, (4 + S) * ninst);
    if (rc != FQ_OK) rc = FQ_ERR_NOMEM;
  }
  if (rc == FQ_OK && hipStreamSynchronize(e->stream) != hipSuccess) rc = FQ_ERR_DEVICE;
  if (rc != FQ_OK) {
    fq_destroy(e);
    return rc;
  }
  *out = e;
  return FQ_OK;
}

int fq_load_batch(fq_engine* e, const int32_t* inst, const uint64_t* states, const int64_t* pops, const double* dat,
                  int64_t n) {
  if (!e || !e->batched || n < 0 || (n > 0 && (!inst || !states || !pops || !dat))) return FQ_ERR_ARG;
  const int S = e->S;
  std::vector<int64_t> order(static_cast<size_t>(n));
  std::vector<uint64_t> key(static_cast<size_t>(n));
  for (int64_t i = 0; i < n; ++i) {
    if (inst[i] < 0 || inst[i] >= e->ninst || (states[i] >> kInstShift) != 0) return FQ_ERR_ARG;
    key[i] = states[i] | (static_cast<uint64_t>(inst[i]) << kInstShift);
    order[i] = i;
  }
  std::sort(order.begin(), order.end(), [&](int64_t a, int64_t b) { return key[a] < key[b]; });
  for (int64_t i = 1; i < n; ++i)
    if (key[order[i]] == key[order[i - 1]]) return FQ_ERR_ARG;
  std::vector<uint64_t> st(static_cast<size_t>(n));
  std::vector<int64_t> po(static_cast<size_t>(S) * n);
  std::vector<double> da(static_cast<size_t>(n));
  for (int64_t i = 0; i < n; ++i) {
    st[i] = key[order[i]];
    for (int q = 0; q < S; ++q) po[i * S + q] = pops[order[i] * S + q];
    da[i] = dat[order[i]];
  }
  return fq_load(e, st.data(), po.data(), da.data(), n);  // the encoded, sorted list
}

// Per-instance estimators and counts of a batched cycle (after annihilation;
// old-list bounds ob, new-list bounds nbd, nold and nnew bounds of the two
// lengths, pnew the new list's populations).
static int inst_stats(fq_engine* e, const int64_t* ob, const int64_t* nbd, int64_t nold, int64_t nnew,
                      const int64_t* pnew) {
  const int ninst = e->ninst, S = e->S;
  hipStream_t st = e->stream;
  hipLaunchKernelGGL(k_inst_nblk, dim3(grid_for(ninst)), dim3(kBlock), 0, st, ninst, ob, e->d_iblk_cnt);
  int rc = scan_exclusive(e, e->d_iblk_cnt, e->d_iblk_off, ninst);
  if (rc != FQ_OK) return rc;
  hipLaunchKernelGGL(k_inst_nblk, dim3(grid_for(ninst)), dim3(kBlock), 0, st, ninst, nbd, e->d_iblk_cnt);
  rc = scan_exclusive(e, e->d_iblk_cnt, e->d_nblk_off, ninst);
  if (rc != FQ_OK) return rc;
  // blocks of either list: at most (length / 256) + ninst
  const int64_t nblk = std::min<int64_t>(std::max<int64_t>(nold, nnew) / kBlock + ninst + 1, e->ipb);
  hipLaunchKernelGGL(k_inst_part, dim3(static_cast<unsigned>(nblk)), dim3(kBlock), 0, st, ninst, S, e->cap, ob,
                     e->d_iblk_off, e->d_cterm, e->d_cdeath, nbd, e->d_nblk_off, pnew, e->ipb,
                     e->d_ipart_d, e->d_ipart_i);
  hipLaunchKernelGGL(k_inst_stats, dim3(ninst), dim3(kBlock), 0, st, ninst, S, ob, nbd, e->d_isb, e->d_iblk_off,
                     e->d_nblk_off, e->ipb, e->d_ipart_d, e->d_ipart_i, att_offsets(e), e->d_iout_d, e->d_iout_i);
  return FQ_OK;
}

// Per-instance results of a batched cycle from the k_inst_stats outputs.
static void batch_outputs(const fq_engine* e, bool spawn_ovf, bool main_ovf, const double* od, const int64_t* oi,
                          fq_cycle_out* out) {
  const int S = e->S;
  const double rf = static_cast<double>(e->sys.rf);
  for (int k = 0; k < e->ninst; ++k) {
    fq_cycle_out& r = out[k];
    std::memset(&r, 0, sizeof(r));
    const int64_t* q = oi + k * (4 + S);
    for (int sp = 0; sp < S; ++sp) {
      r.proj_energy[sp] = od[k * 2 * S + 2 * sp];
      r.D0_population[sp] = od[k * 2 * S + 2 * sp + 1];
      r.nparticles[sp] = static_cast<double>(q[4 + sp]) / rf;
    }
    r.ndeath = q[0];
    r.nattempts = q[1];
    r.nspawn_events = q[2];
    r.nstates = q[3];
    r.spawn_overflow = spawn_ovf ? 1 : 0;
    r.main_overflow = main_ovf ? 1 : 0;
  }
}

// ---- graph-captured batched cycles ---------------------------------------------
// Launch bound of a length: the next multiple of a quarter of its octave (at
// most 25% past it), so one graph serves while the length stays in its step.
static int64_t len_step(int64_t x) {
  if (x <= 4096) return 4096;
  const int e = 63 - __builtin_clzll(static_cast<unsigned long long>(x - 1));  // 2^e <= x - 1 < 2^(e+1)
  const int64_t step = int64_t{1} << (e - 2);
  return ceil_div(x, step) * step;
}
// Candidate schedules: (8-bit digits only, spawning grid cap); index 0 is the
// one ordinary cycles use.
constexpr int kNumSched = 6;
constexpr int kSchedDigit8[kNumSched] = {0, 0, 0, 1, 1, 1};
constexpr int kSchedSpawnBlocks[kNumSched] = {0, 2048, 1024, 0, 2048, 1024};
constexpr int kTuneReps = 3;  // timed graph cycles per candidate

static size_t graph_in_bytes(const fq_engine* e) { return 16 + sizeof(double) * (1 + 2 * e->S) * e->ninst; }

// The whole batched cycle for list buffer c, launches sized by nb (main list)
// and tb (attempts), lengths and the cycle index read on the device, inputs
// copied from h_in first and outputs to the pinned buffers last.  Called while
// the stream is captured.
static int enqueue_graph_cycle(fq_engine* e, int64_t nb, int64_t tb) {
  const int ninst = e->ninst, S = e->S;
  const int64_t cap = e->cap;
  const int c = e->cur;
  hipStream_t st = e->stream;
  const int64_t* dn = reinterpret_cast<const int64_t*>(e->d_in);
  const uint32_t* dcyc = reinterpret_cast<const uint32_t*>(e->d_in + 8);
  const double* par = reinterpret_cast<const double*>(e->d_in + 16);
  FQ_HIP(hipMemcpyAsync(e->d_in, e->h_in, graph_in_bytes(e), hipMemcpyHostToDevice, st));
  int64_t* ob = e->d_ibound;
  int64_t* nbd = e->d_ibound + (ninst + 1);
  hipLaunchKernelGGL(k_inst_bounds, dim3(grid_for(ninst + 1)), dim3(kBlock), 0, st, e->det[c], nb, ninst, kInstShift,
                     ob, dn);
  hipLaunchKernelGGL(k_det_pass_batch, dim3(grid_for(nb)), dim3(kBlock), 0, st, e->sys, e->d_sys_arr, ob, par, ninst,
                     nb, cap, e->det[c], e->pop, e->kii[c], e->pop_new, att_counts(e), parent_flags(e), e->par.philox_seed, 0u,
                     e->d_cterm, e->d_cdeath, dn, dcyc, e->blk_att, e->d_stats);
  // entries past the list have no attempts, so att_off[S nb] is the total
  const int64_t nent = S * nb;
  const int gen = fqd::gen_of(e->sys.system, e->sys.excit_gen);
  const int tile = spawn_tile(gen, tb);
  int rc = scan_attempts(e, nent, tb, tile);
  if (rc != FQ_OK) return rc;
  hipLaunchKernelGGL(k_inst_att, dim3(grid_for(ninst)), dim3(kBlock), 0, st, ninst, S, ob, att_offsets(e), e->d_iatt);
  const unsigned g = static_cast<unsigned>(std::min<int64_t>(
      ceil_div(tb, tile), e->spawn_blocks > 0 ? e->spawn_blocks : int64_t{1} << 20));
  auto kern = tile == kSmallTile ? spawn_kernel<true, kSmallTile>(gen) : spawn_kernel<true, kSpawnTile>(gen);
  hipLaunchKernelGGL(kern, dim3(g), dim3(kBlock), 0, st, e->d_sysp, nent, cap, int64_t{0}, tb, att_offsets(e), e->det[c],
                     e->pop, 0.0, e->par.philox_seed, 0u, e->bcap, e->st_det, e->st_pop, e->st_ent, e->tile_cnt,
                     e->tile_win, parent_flags(e), e->d_sys_arr, e->d_iatt, par, dcyc, e->d_stats);
  pack_spawned(e, tb, tile, true, att_offsets(e) + nent, tb);
  e->keys_ready = true;
  const int64_t nsb = std::min<int64_t>(tb, e->scap);
  const int64_t* pns = &e->d_stats->nspawn;
  hipLaunchKernelGGL(k_inst_bounds, dim3(grid_for(ninst + 1)), dim3(kBlock), 0, st, e->kbuf[0], nsb, ninst,
                     kInstShift + e->flag_bits, e->d_isb, pns);
  int64_t rng_pos = e->rng_pos;
  rc = annihilate(e, nsb, pns, false, 0u, rng_pos);
  if (rc != FQ_OK) return rc;
  const int o = 1 - c;
  hipLaunchKernelGGL(k_inst_bounds, dim3(grid_for(ninst + 1)), dim3(kBlock), 0, st, e->det[o],
                     std::min<int64_t>(nb + nsb, cap), ninst, kInstShift, nbd, &e->d_stats->new_n);
  rc = inst_stats(e, ob, nbd, nb, std::min<int64_t>(nb + nsb, cap), e->pop);
  if (rc != FQ_OK) return rc;
  FQ_HIP(hipMemcpyAsync(e->h_god, e->d_iout_d, sizeof(double) * 2 * S * ninst, hipMemcpyDeviceToHost, st));
  FQ_HIP(hipMemcpyAsync(e->h_goi, e->d_iout_i, sizeof(int64_t) * (4 + S) * ninst, hipMemcpyDeviceToHost, st));
  return FQ_OK;
}

// The graph of (list buffer, bounds, schedule), captured on first use.
static int graph_for(fq_engine* e, int64_t nb, int64_t tb, int sched, hipGraphExec_t* out) {
  for (const auto& g : e->graphs)
    if (g.c == e->cur && g.nb == nb && g.tb == tb && g.sched == sched) {
      *out = g.exec;
      return FQ_OK;
    }
  e->digit8 = kSchedDigit8[sched];
  e->spawn_blocks = kSchedSpawnBlocks[sched];
  const int64_t n_keep = e->n;
  e->n = nb;  // annihilation sizes its launches by e->n
  e->dn = reinterpret_cast<const int64_t*>(e->d_in);
  e->dcyc = reinterpret_cast<const uint32_t*>(e->d_in + 8);
  e->capturing = true;
  hipGraph_t graph = nullptr;
  int rc = FQ_OK;
  if (hipStreamBeginCapture(e->stream, hipStreamCaptureModeRelaxed) != hipSuccess) {
    rc = FQ_ERR_DEVICE;
  } else {
    rc = enqueue_graph_cycle(e, nb, tb);
    if (hipStreamEndCapture(e->stream, &graph) != hipSuccess && rc == FQ_OK) rc = FQ_ERR_DEVICE;
  }
  e->capturing = false;
  e->dn = nullptr;
  e->dcyc = nullptr;
  e->n = n_keep;
  e->digit8 = 0;
  e->spawn_blocks = 0;
  hipGraphExec_t exec = nullptr;
  if (rc == FQ_OK && hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess) rc = FQ_ERR_DEVICE;
  if (graph) (void)hipGraphDestroy(graph);
  if (rc != FQ_OK) return rc;
  e->graphs.push_back({e->cur, nb, tb, sched, exec});
  *out = exec;
  return FQ_OK;
}

static float median_of(std::vector<float> v) {
  std::sort(v.begin(), v.end());
  return v.empty() ? 0.0f : v[v.size() / 2];
}

// One batched cycle as a graph launch; *done = false when the cycle must run
// as ordinary launches (attempt bound unknown or past the staging capacity).
static int graph_cycle(fq_engine* e, const double* shift, const double* eproj_old, const double* tau,
                       fq_cycle_out* out, bool* done) {
  *done = false;
  const int ninst = e->ninst, S = e->S;
  if (e->n <= 0 || e->att_bound <= 0) return FQ_OK;
  const int64_t nb = std::min<int64_t>(len_step(e->n), e->cap);
  const int64_t tb = std::min<int64_t>(len_step(e->att_bound), e->bcap);
  if (e->att_bound > tb) return FQ_OK;
  if (int rs = sync_sysp(e); rs != FQ_OK) return rs;
  // the tuner works per octave of the attempt bound (the schedules' relative
  // cost changes with the workload's size): candidates in turn until each has
  // run kTuneReps times, then the fastest by median
  const int oct = 63 - __builtin_clzll(static_cast<unsigned long long>(tb));
  e->last_oct = oct;
  int sched = e->sched[oct];
  if (sched < 0) sched = e->tune_iter[oct] % kNumSched;
  hipGraphExec_t exec = nullptr;
  int rc = graph_for(e, nb, tb, sched, &exec);
  if (rc != FQ_OK) return rc;
  // inputs: the list length, the cycle index, then tau, shift, E_proj per instance
  const uint32_t cyc = static_cast<uint32_t>(e->cycle_index++);
  int64_t* hi = reinterpret_cast<int64_t*>(e->h_in);
  hi[0] = e->n;
  hi[1] = static_cast<int64_t>(cyc);
  double* par = reinterpret_cast<double*>(e->h_in + 16);
  for (int k = 0; k < ninst; ++k) {
    par[k] = tau[k];
    for (int sp = 0; sp < S; ++sp) {
      par[ninst + sp * ninst + k] = shift[k * S + sp];
      par[(1 + S) * ninst + sp * ninst + k] = eproj_old[k * S + sp];
    }
  }
  FQ_HIP(hipEventRecord(e->gev[0], e->stream));
  FQ_HIP(hipGraphLaunch(exec, e->stream));
  FQ_HIP(hipEventRecord(e->gev[1], e->stream));
  FQ_HIP(hipStreamSynchronize(e->stream));
  float ms = 0.0f;
  (void)hipEventElapsedTime(&ms, e->gev[0], e->gev[1]);
  ++e->graph_cycles;
  if (e->sched[oct] < 0) {
    e->tune_ms[oct][sched].push_back(ms);
    if (++e->tune_iter[oct] >= kNumSched * kTuneReps) {
      int best = 0;
      for (int k = 1; k < kNumSched; ++k)
        if (median_of(e->tune_ms[oct][k]) < median_of(e->tune_ms[oct][best])) best = k;
      e->sched[oct] = best;
    }
  }
  e->h_stats = *e->h_pin;
  if (e->h_stats.spawn_overflow && e->h_stats.total_attempts > tb) return FQ_ERR_DEVICE;  // the bound was wrong
  e->cur = 1 - e->cur;
  e->n = e->h_stats.new_n;
  unsigned long long sum = 0;
  for (int sp = 0; sp < S; ++sp) sum += e->h_stats.abs_pop[sp];
  e->att_bound = static_cast<int64_t>(sum / static_cast<unsigned long long>(e->sys.rf));
  e->t_total = ms;
  e->prof = fq_profile_out{};
  e->prof.total_ms = ms;
  e->prof.nattempts = e->h_stats.total_attempts;
  e->prof.nspawned = std::min<int64_t>(e->h_stats.nspawn, e->scap);
  e->prof.nruns = e->h_stats.nruns;
  e->prof.nstates_out = e->n;
  batch_outputs(e, e->h_stats.spawn_overflow != 0, e->h_stats.main_overflow != 0, e->h_god, e->h_goi, out);
  *done = true;
  return FQ_OK;
}

int fq_batch_graph(fq_engine* e, int32_t enable) {
  if (!e || !e->batched) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  if (enable && !e->h_in) {
    // scan scratch for the longest list of counts a cycle of this engine can
    // scan: the determinant pass's blocks, the run and main tiles, the instances
    const int64_t longest = std::max({ceil_div(e->cap, kBlock), ceil_div(e->scap, kRunTile), int64_t{e->ninst}});
    const int64_t ntile = ceil_div(longest, kScanTile);
    if (!scan_scratch(e, 0, ntile) || !scan_scratch(e, 1, ntile + 1)) return FQ_ERR_NOMEM;
    const size_t nin = graph_in_bytes(e);
    if (hipHostMalloc(reinterpret_cast<void**>(&e->h_in), nin) != hipSuccess ||
        hipHostMalloc(reinterpret_cast<void**>(&e->h_god), sizeof(double) * 2 * e->S * e->ninst) != hipSuccess ||
        hipHostMalloc(reinterpret_cast<void**>(&e->h_goi), sizeof(int64_t) * (4 + e->S) * e->ninst) != hipSuccess)
      return FQ_ERR_NOMEM;
    if (dalloc(&e->d_in, static_cast<int64_t>(nin)) != FQ_OK) return FQ_ERR_NOMEM;
    for (int k = 0; k < 2; ++k)
      if (hipEventCreate(&e->gev[k]) != hipSuccess) return FQ_ERR_DEVICE;
    for (int o = 0; o < 64; ++o) {
      e->sched[o] = -1;
      e->tune_iter[o] = 0;
    }
  }
  e->graph_on = enable != 0;
  return FQ_OK;
}

int fq_batch_schedule(fq_engine* e, fq_schedule_out* out) {
  if (!e || !e->batched || !out) return FQ_ERR_ARG;
  std::memset(out, 0, sizeof(*out));
  const int oct = e->last_oct;  // the last graph cycle's octave
  const int ch = oct >= 0 ? e->sched[oct] : -1;
  const int k = ch < 0 ? 0 : ch;
  out->graph = e->graph_on ? 1 : 0;
  out->tuned = ch >= 0 ? 1 : 0;
  out->chosen = ch;
  out->octave = oct;
  for (int o = 0; o < 64; ++o) out->tuned_octaves += e->h_in && e->sched[o] >= 0 ? 1 : 0;
  out->digit_bits = kSchedDigit8[k] ? 8 : 9;
  out->spawn_blocks = kSchedSpawnBlocks[k];
  out->ncand = kNumSched;
  out->graph_cycles = e->graph_cycles;
  out->graphs = static_cast<int64_t>(e->graphs.size());
  out->eager_cycles = e->eager_cycles;
  for (int q = 0; q < kNumSched; ++q) {
    out->cand_ms[q] = oct >= 0 ? median_of(e->tune_ms[oct][q]) : 0.0;
    out->cand_digit_bits[q] = kSchedDigit8[q] ? 8 : 9;
    out->cand_spawn_blocks[q] = kSchedSpawnBlocks[q];
  }
  return FQ_OK;
}

int fq_cycle_batch(fq_engine* e, const double* shift, const double* eproj_old, const double* tau,
                   fq_cycle_out* out) {
  if (!e || !e->batched || !shift || !eproj_old || !tau || !out) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  if (e->graph_on) {
    bool done = false;
    const int grc = graph_cycle(e, shift, eproj_old, tau, out, &done);
    if (grc != FQ_OK || done) return grc;
  }
  ++e->eager_cycles;
  const int ninst = e->ninst, S = e->S;
  const int64_t n = e->n, cap = e->cap;
  const int c = e->cur;
  hipStream_t st = e->stream;
  const uint32_t cyc = static_cast<uint32_t>(e->cycle_index++);
  std::vector<double> par(static_cast<size_t>((1 + 2 * S) * ninst));
  for (int k = 0; k < ninst; ++k) {
    par[k] = tau[k];
    for (int sp = 0; sp < S; ++sp) {
      par[ninst + sp * ninst + k] = shift[k * S + sp];
      par[(1 + S) * ninst + sp * ninst + k] = eproj_old[k * S + sp];
    }
  }
  FQ_HIP(hipMemcpyAsync(e->d_ipar, par.data(), sizeof(double) * par.size(), hipMemcpyHostToDevice, st));
  int64_t* ob = e->d_ibound;
  int64_t* nbd = e->d_ibound + (ninst + 1);
  hipLaunchKernelGGL(k_inst_bounds, dim3(grid_for(ninst + 1)), dim3(kBlock), 0, st, e->det[c], n, ninst, kInstShift, ob,
                     nullptr);
  hipLaunchKernelGGL(k_det_pass_batch, dim3(grid_for(n)), dim3(kBlock), 0, st, e->sys, e->d_sys_arr, ob, e->d_ipar,
                     ninst, n, cap, e->det[c], e->pop, e->kii[c], e->pop_new, att_counts(e), parent_flags(e), e->par.philox_seed,
                     cyc, e->d_cterm, e->d_cdeath, nullptr, nullptr, e->blk_att, e->d_stats);
  const int64_t nent = S * n;
  int rc = scan_attempts(e, nent, e->bcap, kSpawnTile);
  if (rc != FQ_OK) return rc;
  hipLaunchKernelGGL(k_inst_att, dim3(grid_for(ninst)), dim3(kBlock), 0, st, ninst, S, ob, att_offsets(e), e->d_iatt);
  int64_t total = 0;
  FQ_HIP(hipMemcpyAsync(&total, att_offsets(e) + nent, sizeof(int64_t), hipMemcpyDeviceToHost, st));
  FQ_HIP(hipStreamSynchronize(st));
  e->spawn_launches = 0;
  if (int rs = sync_sysp(e); rs != FQ_OK) return rs;
  const bool one_batch = total <= e->bcap;
  auto kern = spawn_kernel<true, kSpawnTile>(fqd::gen_of(e->sys.system, e->sys.excit_gen));
  for (int64_t tb = 0; tb < total; tb += e->bcap) {
    const int64_t te = std::min(total, tb + e->bcap);
    const int64_t nt = ceil_div(te - tb, kSpawnTile);
    ++e->spawn_launches;
    if (!one_batch)
      hipLaunchKernelGGL(k_tile_bounds, dim3(grid_for(nt)), dim3(kBlock), 0, st, nent, att_offsets(e), tb, te,
                         e->tile_win);
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(std::min<int64_t>(nt, 1 << 20))), dim3(kBlock), 0, st,
                       e->d_sysp, nent, cap, tb, te, att_offsets(e), e->det[c], e->pop, 0.0, e->par.philox_seed, cyc,
                       e->bcap, e->st_det, e->st_pop, e->st_ent, e->tile_cnt, e->tile_win, parent_flags(e), e->d_sys_arr,
                       e->d_iatt, e->d_ipar, nullptr, e->d_stats);
    pack_spawned(e, te - tb, kSpawnTile, one_batch, att_offsets(e) + nent);
  }
  e->keys_ready = true;  // the packing kernels wrote the sort keys
  rc = sync_stats(e);
  if (rc != FQ_OK) return rc;
  const int64_t ns = std::min<int64_t>(e->h_stats.nspawn, e->scap);
  // spawned entries are in attempt order, hence grouped by instance
  hipLaunchKernelGGL(k_inst_bounds, dim3(grid_for(ninst + 1)), dim3(kBlock), 0, st, e->kbuf[0], ns, ninst,
                     kInstShift + e->flag_bits, e->d_isb, nullptr);
  const Stats keep = e->h_stats;
  int64_t rng_pos = e->rng_pos;
  rc = annihilate(e, ns, nullptr, false, cyc, rng_pos);
  if (rc != FQ_OK) return rc;
  const int o = e->cur;
  hipLaunchKernelGGL(k_inst_bounds, dim3(grid_for(ninst + 1)), dim3(kBlock), 0, st, e->det[o], e->n, ninst, kInstShift,
                     nbd, nullptr);
  rc = inst_stats(e, ob, nbd, n, e->n, e->pop);
  if (rc != FQ_OK) return rc;
  std::vector<double> od(static_cast<size_t>(2 * S * ninst));
  std::vector<int64_t> oi(static_cast<size_t>((4 + S) * ninst));
  FQ_HIP(hipMemcpyAsync(od.data(), e->d_iout_d, sizeof(double) * od.size(), hipMemcpyDeviceToHost, st));
  FQ_HIP(hipMemcpyAsync(oi.data(), e->d_iout_i, sizeof(int64_t) * oi.size(), hipMemcpyDeviceToHost, st));
  FQ_HIP(hipStreamSynchronize(st));
  fill_profile(e, n, ns);
  batch_outputs(e, keep.spawn_overflow != 0, e->h_stats.main_overflow != 0, od.data(), oi.data(), out);
  // the next cycle's attempt total: sum |N| over the new list (integer populations)
  unsigned long long sum = 0;
  for (int sp = 0; sp < S; ++sp) sum += e->h_stats.abs_pop[sp];
  e->att_bound = static_cast<int64_t>(sum / static_cast<unsigned long long>(e->sys.rf));
  return FQ_OK;
}

// ---- learned proposal ---------------------------------------------------------
int fq_mlp_nparams(fq_engine* e, int64_t* n) {
  if (!e || !n) return FQ_ERR_ARG;
  if (e->par.excit_gen != FQ_EXCIT_LEARNED) return FQ_ERR_ARG;
  *n = e->mlp.nparams;
  return FQ_OK;
}

int fq_mlp_set_params(fq_engine* e, const float* p, int64_t n) {
  if (!e || !p || e->par.excit_gen != FQ_EXCIT_LEARNED || n != e->mlp.nparams) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  return fqm::mlp_set(e->mlp, p, e->stream);
}

int fq_mlp_get_params(fq_engine* e, float* p, int64_t n) {
  if (!e || !p || e->par.excit_gen != FQ_EXCIT_LEARNED || n != e->mlp.nparams) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  FQ_HIP(hipMemcpyAsync(p, e->mlp.p, sizeof(float) * n, hipMemcpyDeviceToHost, e->stream));
  FQ_HIP(hipStreamSynchronize(e->stream));
  return FQ_OK;
}

int fq_mlp_affinity(fq_engine* e, float* out, int64_t n) {
  if (!e || !out || e->par.excit_gen != FQ_EXCIT_LEARNED) return FQ_ERR_ARG;
  if (n != static_cast<int64_t>(e->mlp.nb) * e->mlp.nb) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  FQ_HIP(hipMemcpyAsync(out, e->mlp.aff, sizeof(float) * n, hipMemcpyDeviceToHost, e->stream));
  FQ_HIP(hipStreamSynchronize(e->stream));
  return FQ_OK;
}

int fq_mlp_forward(fq_engine* e, const uint64_t* dets, int64_t n, float* out) {
  if (!e || !dets || !out || n < 1 || e->par.excit_gen != FQ_EXCIT_LEARNED) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  const int W = e->W;
  std::vector<uint64_t> soa(static_cast<size_t>(W) * n);
  for (int64_t i = 0; i < n; ++i)
    for (int w = 0; w < W; ++w) soa[w * n + i] = dets[i * W + w];
  uint64_t* d_det = nullptr;
  float* d_out = nullptr;
  int rc = dalloc(&d_det, W * n);
  rc |= dalloc(&d_out, n * e->mlp.d_out);
  if (rc == FQ_OK) {
    hipStream_t st = e->stream;
    if (hipMemcpyAsync(d_det, soa.data(), sizeof(uint64_t) * W * n, hipMemcpyHostToDevice, st) != hipSuccess)
      rc = FQ_ERR_DEVICE;
    if (rc == FQ_OK) rc = fqm::mlp_infer(e->mlp, e->sys, d_det, n, n, d_out, st);
    if (rc == FQ_OK &&
        hipMemcpyAsync(out, d_out, sizeof(float) * n * e->mlp.d_out, hipMemcpyDeviceToHost, st) != hipSuccess)
      rc = FQ_ERR_DEVICE;
    if (hipStreamSynchronize(st) != hipSuccess) rc = FQ_ERR_DEVICE;
  } else {
    rc = FQ_ERR_NOMEM;
  }
  dfree(d_det);
  dfree(d_out);
  return rc;
}

static int loss_grad(fq_engine* e, const uint64_t* dets, const int32_t* exc, const double* w, const double* habs,
                     const int32_t* flat, int64_t n, double* loss, float* grad) {
  if (!e || !dets || !exc || !w || !loss || n < 1 || e->par.excit_gen != FQ_EXCIT_LEARNED) return FQ_ERR_ARG;
  fqm::Mlp& m = e->mlp;
  if (n > m.bcap) return FQ_ERR_CAPACITY;
  const int W = e->W;
  // every weighted sample: a double i<j (occupied) -> a<b (unoccupied), orbitals in 1..nbasis
  for (int64_t k = 0; k < n; ++k) {
    if (!(w[k] > 0.0)) continue;
    const int32_t* x = exc + 4 * k;
    auto occ = [&](int o) { return (dets[k * W + (o - 1) / 64] >> ((o - 1) % 64)) & 1; };
    for (int q = 0; q < 4; ++q)
      if (x[q] < 1 || x[q] > e->sys.nbasis) return FQ_ERR_ARG;
    if (!(x[0] < x[1] && x[2] < x[3]) || !occ(x[0]) || !occ(x[1]) || occ(x[2]) || occ(x[3])) return FQ_ERR_ARG;
  }
  FQ_HIP(hipSetDevice(e->device));
  hipStream_t st = e->stream;
  std::vector<uint64_t> soa(static_cast<size_t>(W) * n);
  for (int64_t i = 0; i < n; ++i)
    for (int q = 0; q < W; ++q) soa[q * n + i] = dets[i * W + q];
  for (int q = 0; q < W; ++q)
    FQ_HIP(hipMemcpyAsync(m.sdet + q * m.bcap, soa.data() + q * n, sizeof(uint64_t) * n, hipMemcpyHostToDevice, st));
  FQ_HIP(hipMemcpyAsync(m.sexc, exc, sizeof(int32_t) * 4 * n, hipMemcpyHostToDevice, st));
  FQ_HIP(hipMemcpyAsync(m.sw, w, sizeof(double) * n, hipMemcpyHostToDevice, st));
  if (habs) FQ_HIP(hipMemcpyAsync(m.sh, habs, sizeof(double) * n, hipMemcpyHostToDevice, st));
  const std::vector<int32_t> fl = flat ? std::vector<int32_t>(flat, flat + n) : std::vector<int32_t>(n, 0);
  FQ_HIP(hipMemcpyAsync(m.sflat, fl.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, st));
  const int keep = m.objective;
  m.objective = habs ? 1 : 0;
  int rc = fqm::mlp_train_step(m, e->sys, n, 0.0, false, st);
  m.objective = keep;
  if (rc != FQ_OK) return rc;
  double sums[2] = {0.0, 0.0};
  FQ_HIP(hipMemcpyAsync(sums, m.dsum, sizeof(sums), hipMemcpyDeviceToHost, st));
  if (grad) FQ_HIP(hipMemcpyAsync(grad, m.g, sizeof(float) * m.nparams, hipMemcpyDeviceToHost, st));
  FQ_HIP(hipStreamSynchronize(st));
  *loss = sums[1];
  return FQ_OK;
}

int fq_mlp_loss_grad(fq_engine* e, const uint64_t* dets, const int32_t* exc, const double* w, const int32_t* flat,
                     int64_t n, double* loss, float* grad) {
  return loss_grad(e, dets, exc, w, nullptr, flat, n, loss, grad);
}

int fq_mlp_variance_grad(fq_engine* e, const uint64_t* dets, const int32_t* exc, const double* w,
                         const double* habs, const int32_t* flat, int64_t n, double* loss, float* grad) {
  if (!habs) return FQ_ERR_ARG;
  return loss_grad(e, dets, exc, w, habs, flat, n, loss, grad);
}

int fq_mlp_online(fq_engine* e, int32_t every, int32_t steps, int64_t batch, double lr, int32_t objective) {
  if (!e || e->par.excit_gen != FQ_EXCIT_LEARNED || every < 0 || steps < 0 || (objective != 0 && objective != 1))
    return FQ_ERR_ARG;
  if (every > 0 && (batch < 1 || !(lr > 0.0))) return FQ_ERR_ARG;
  if (batch > e->mlp.bcap) return FQ_ERR_CAPACITY;
  e->online_every = every;
  e->online_steps = steps;
  e->online_batch = batch;
  e->online_lr = lr;
  e->mlp.objective = objective;
  return FQ_OK;
}

int fq_mlp_train(fq_engine* e, int64_t batch, int32_t steps, double lr, uint64_t seed, double* losses) {
  if (!e || batch < 1 || steps < 0 || !(lr > 0.0) || e->par.excit_gen != FQ_EXCIT_LEARNED) return FQ_ERR_ARG;
  fqm::Mlp& m = e->mlp;
  if (batch > m.bcap) return FQ_ERR_CAPACITY;
  if (e->n < 1) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  hipStream_t st = e->stream;
  const int c = e->cur;
  for (int32_t k = 0; k < steps; ++k) {
    int rc = fqm::mlp_sample(m, e->sys, e->det[c], e->pop, e->cap, e->n, batch,
                             static_cast<int64_t>(e->par.proposal_min_attempts), seed,
                             static_cast<uint32_t>(m.adam_t), st, scan_cb, e);
    if (rc != FQ_OK) return rc;
    rc = fqm::mlp_train_step(m, e->sys, batch, lr, true, st);
    if (rc != FQ_OK) return rc;
    if (losses) {
      double sums[2] = {0.0, 0.0};
      FQ_HIP(hipMemcpyAsync(sums, m.dsum, sizeof(sums), hipMemcpyDeviceToHost, st));
      FQ_HIP(hipStreamSynchronize(st));
      losses[k] = sums[1];
    }
  }
  FQ_HIP(hipStreamSynchronize(st));
  return FQ_OK;
}

int fq_probe_excitations(fq_engine* e, const uint64_t* det, int64_t n, uint64_t seed, int32_t* exc, double* pgen,
                         double* hmatel) {
  if (!e || !det || !exc || !pgen || !hmatel || n < 1) return FQ_ERR_ARG;
  if (e->sys.system != FQ_SYS_READ_IN) return FQ_ERR_ARG;
  const int W = e->W;
  {  // the determinant must hold nel electrons in orbitals 1..nbasis
    int nel = 0;
    for (int w = 0; w < W; ++w) {
      if (det[w] & ~e->sys.valid[w]) return FQ_ERR_ARG;
      nel += __builtin_popcountll(det[w]);
    }
    if (nel != e->sys.nel) return FQ_ERR_ARG;
  }
  FQ_HIP(hipSetDevice(e->device));
  hipStream_t st = e->stream;
  int32_t* d_exc = nullptr;
  double *d_pg = nullptr, *d_h = nullptr;
  float* d_row = nullptr;
  uint64_t* d_det = nullptr;
  int rc = dalloc(&d_exc, 6 * n);
  rc |= dalloc(&d_pg, n);
  rc |= dalloc(&d_h, n);
  rc |= dalloc(&d_det, W);
  rc |= dalloc(&d_row, 2 * static_cast<int64_t>(e->sys.nbasis));
  if (rc == FQ_OK && hipMemcpyAsync(d_det, det, sizeof(uint64_t) * W, hipMemcpyHostToDevice, st) != hipSuccess)
    rc = FQ_ERR_DEVICE;
  // learned: the network's row, or (proposal_min_attempts > 1, as for a determinant with one
  // attempt in a cycle) none, so that the flat weights are drawn from
  const bool row = e->par.excit_gen == FQ_EXCIT_LEARNED && e->par.proposal_min_attempts <= 1;
  if (rc == FQ_OK && row) rc = fqm::mlp_infer(e->mlp, e->sys, d_det, 1, 1, d_row, st);
  if (rc == FQ_OK) {
    hipLaunchKernelGGL(k_probe, dim3(grid_for(n)), dim3(kBlock), 0, st, e->sys, det[0], W > 1 ? det[1] : 0,
                       row ? d_row : nullptr, n, seed, d_exc, d_pg, d_h);
    if (hipGetLastError() != hipSuccess) rc = FQ_ERR_DEVICE;
  }
  if (rc == FQ_OK) {
    if (hipMemcpyAsync(exc, d_exc, sizeof(int32_t) * 6 * n, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipMemcpyAsync(pgen, d_pg, sizeof(double) * n, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipMemcpyAsync(hmatel, d_h, sizeof(double) * n, hipMemcpyDeviceToHost, st) != hipSuccess)
      rc = FQ_ERR_DEVICE;
  }
  if (hipStreamSynchronize(st) != hipSuccess) rc = FQ_ERR_DEVICE;
  dfree(d_exc);
  dfree(d_pg);
  dfree(d_h);
  dfree(d_det);
  dfree(d_row);
  return rc;
}

void fq_destroy(fq_engine* e) {
  if (!e) return;
  (void)hipSetDevice(e->device);
  if (e->stream) (void)hipStreamSynchronize(e->stream);
  for (int b = 0; b < 2; ++b) {
    dfree(e->det[b]);
    dfree(e->kii[b]);
    dfree(e->kbuf[b]);
    dfree(e->mrank[b]);
    dfree(e->new_pos[b]);
  }
  dfree(e->pop);
  dfree(e->pop_new);
  dfree(e->att_off);
  release_determ(e);
  dfree(e->mmask);
  dfree(e->mpre);
  dfree(e->abs_part);
  dfree(e->run_win);
  dfree(e->new_cnt);
  dfree(e->new_off);
  dfree(e->new_val);
  dfree(e->new_pop);
  dfree(e->mcnt);
  dfree(e->moff);
  dfree(e->mdraw);
  dfree(e->mdraw_off);
  dfree(e->part_d);
  dfree(e->part_i);
  dfree(e->st_det);
  dfree(e->st_pop);
  dfree(e->st_ent);
  dfree(e->tile_cnt);
  dfree(e->blk_att);
  dfree(e->blk_off);
  dfree(e->tile_win);
  e->sdet = nullptr;  // aliases of kbuf[1], pbuf[1]
  e->srec = nullptr;
  dfree(e->perm);
  dfree(e->pbuf[0]);
  dfree(e->pbuf[1]);
  dfree(e->pass_cnt);
  dfree(e->pass_off);
  dfree(e->run_tcnt);
  dfree(e->run_toff);
  dfree(e->run_tfirst);
  dfree(e->run_tpre);
  dfree(e->d_sysp);
  dfree(e->ndraw);
  dfree(e->ndraw_off);
  for (auto*& p : e->scan_tmp) dfree(p);
  dfree(e->rng_buf);
  dfree(e->d_stats);
  dfree(e->d_sp_eigv);
  dfree(e->d_sym_table);
  dfree(e->d_inv_sym);
  dfree(e->d_sym_diff);
  dfree(e->d_orb_sym);
  dfree(e->d_nbss);
  dfree(e->d_ssbf);
  dfree(e->d_h1);
  dfree(e->d_eri);
  dfree(e->d_jmat);
  dfree(e->d_kmat);
  dfree(e->d_s1j);
  dfree(e->d_s1k);
  dfree(e->d_recip);
  dfree(e->d_jpair);
  dfree(e->d_hb_i);
  dfree(e->d_hb_ij);
  dfree(e->d_hb_ija);
  dfree(e->d_hb_ija_tot);
  dfree(e->d_hb_ija_u);
  dfree(e->d_hb_ija_k);
  dfree(e->d_hb_ijab);
  dfree(e->d_hb_ijab_tot);
  dfree(e->d_hb_ijab_u);
  dfree(e->d_hb_ijab_k);
  dfree(e->d_hb_bias);
  fqm::mlp_free(e->mlp);
  dfree(e->mlp_tab);
  dfree(e->mlp_flat);
  dfree(e->mlp_row);
  dfree(e->mlp_idx);
  dfree(e->d_binom);
  dfree(e->d_sys_arr);
  dfree(e->d_ipar);
  dfree(e->d_ibound);
  dfree(e->d_isb);
  dfree(e->d_iatt);
  dfree(e->d_cterm);
  dfree(e->d_cdeath);
  dfree(e->d_iblk_cnt);
  dfree(e->d_iblk_off);
  dfree(e->d_nblk_off);
  dfree(e->d_ipart_d);
  dfree(e->d_ipart_i);
  dfree(e->d_iout_d);
  dfree(e->d_iout_i);
  for (fq_engine* sub : e->subs) fq_destroy(sub);
  e->subs.clear();
  if (e->ev_len) (void)hipEventDestroy(e->ev_len);
  if (e->h_len) (void)hipHostFree(e->h_len);
  if (e->h_pin) (void)hipHostFree(e->h_pin);
  if (e->list_buf) (void)hipHostFree(e->list_buf);
  for (hipEvent_t ev : e->list_ev)
    if (ev) (void)hipEventDestroy(ev);
  for (hipStream_t q : e->list_stream)
    if (q) (void)hipStreamDestroy(q);
  for (auto& g : e->graphs) (void)hipGraphExecDestroy(g.exec);
  for (int k = 0; k < 2; ++k)
    if (e->gev[k]) (void)hipEventDestroy(e->gev[k]);
  if (e->h_in) (void)hipHostFree(e->h_in);
  if (e->h_god) (void)hipHostFree(e->h_god);
  if (e->h_goi) (void)hipHostFree(e->h_goi);
  dfree(e->d_in);
  if (e->stream) (void)hipStreamDestroy(e->stream);
  delete e;
}

// ---- for the tests; not part of the interface in include/fqmc.h ----------------
// The parents (det-major (det, space) entries) of the first and last attempt of
// the last cycle's first ntiles spawning tiles.
int fqt_tile_windows(fq_engine* e, int64_t* out, int64_t ntiles) {
  if (!e || !out || ntiles < 1 || ntiles > e->bcap / kSmallTile + 2) return FQ_ERR_ARG;
  FQ_HIP(hipSetDevice(e->device));
  FQ_HIP(hipMemcpyAsync(out, e->tile_win, sizeof(int64_t) * 2 * ntiles, hipMemcpyDeviceToHost, e->stream));
  FQ_HIP(hipStreamSynchronize(e->stream));
  return FQ_OK;
}

// The longest counts of the attempts' blocks, the run tiles and the main tiles
// that no scan precedes (kPrefixAttempts, ...); results do not depend on them.
// Before graph cycles only.
int fqt_prefix_tiles(fq_engine* e, int64_t attempts, int64_t runs, int64_t main) {
  if (!e || attempts < 0 || runs < 0 || main < 0 || !e->graphs.empty()) return FQ_ERR_ARG;
  e->prefix_attempts = attempts;
  e->prefix_runs = runs;
  e->prefix_main = main;
  return FQ_OK;
}

// Spawned lists so far that were sorted again because the one-block sort could not take them.
int64_t fqt_resorts(fq_engine* e) { return e ? e->resorts : -1; }

// Address and elements of a scan scratch buffer (0 and 0: none).
int fqt_scan_scratch(fq_engine* e, int slot, int64_t* address, int64_t* elements) {
  if (!e || slot < 0 || !address || !elements) return FQ_ERR_ARG;
  const bool have = slot < static_cast<int>(e->scan_tmp.size());
  *address = have ? reinterpret_cast<intptr_t>(e->scan_tmp[slot]) : 0;
  *elements = have ? e->scan_tmp_cap[slot] : 0;
  return FQ_OK;
}

}  // extern "C"

// internal.hpp -- library-internal types of libthrml_hip.so.
//
// Device data layout (HBM):
//   state words  uint64_t [G * P][n_total]   G = ceil(n_chains / 64) chain
//                groups, P = bit planes per node (1 for spins, ceil(log2 q)
//                for categories).  Bit l of word (g*P + b, pos) is bit b of
//                the value of chain 64*g + l at global position pos.  A wave
//                of 64 lanes handles one chain group, lane l = chain 64*g + l,
//                so a node's word is wave-uniform (scalar loads) and the new
//                word of a site is one ballot.
//   positions    the reference's global state order: free blocks then clamped
//                blocks, concatenated (crates/thrml-core/src/blockspec.rs:15-67).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/thrml_hip.h"

namespace thrml {

void set_error(const std::string &msg);
int fail(int code, const std::string &msg);
int hip_fail(hipError_t e, const char *what);

#define THRML_HIP(call)                                   \
  do {                                                    \
    hipError_t e_ = (call);                               \
    if (e_ != hipSuccess) return thrml::hip_fail(e_, #call); \
  } while (0)

enum ProgKind : uint32_t { K_LATTICE = 0, K_CSR = 1, K_POTTS = 2, K_DENSE = 3, K_DISCRETE = 4 };

// Resident runs (k_resident.hip): a piece is a run of sites of one block, a
// part the pieces whose keystream blocks one phase computes.
constexpr uint32_t RES_NONE = 0xffffffffu;
constexpr uint32_t RES_MAX_NODES = 65535;   // 16-bit positions; one LDS byte each beside the keystream
constexpr uint32_t RES_MAX_ENT = 10;        // entries per wave of the register kernel
constexpr int RES_LDS = 160 * 1024;
struct ResPiece {
  uint32_t blk, site0, n;  // block, first block-local site, sites
  uint32_t kb0;            // its first keystream block within the part
  uint32_t row0, slice0;   // global position of its first site, its first slice
};
struct ResPart {
  uint32_t piece0, piece1, kb;  // pieces [piece0, piece1), keystream blocks
};

// Device memory that the objects of one context have let go of, for its next
// objects of about the same size: a training step that builds programs,
// states and moments anew then allocates nothing (a hipMalloc and hipFree pair
// of more than 2 MiB takes 100-200 us).  All work of a context is ordered on
// its stream, so a block may be taken again while the last kernels that use it
// still run.  Bounded by KEEP bytes; emptied with the context, when its
// stream changes (blocks taken before that are then freed, not kept: their
// last use may lie on the old stream) and when an allocation fails.  Beside
// them one block of at most LARGEST bytes for host transfers, which come in any
// size; a transfer that finds it taken by another thread's gets its own.
class DevPool {
 public:
  static constexpr size_t KEEP = 256u << 20, LARGEST = 64u << 20;
  ~DevPool() { clear(); }
  // a block of at least n bytes and at most twice as many (capacity in *cap), or
  // null; *era goes back with the block
  void *take(size_t n, size_t *cap, uint64_t *era) {
    std::lock_guard<std::mutex> lk(mu_);
    *era = era_;
    const auto it = free_.lower_bound(n);
    if (it == free_.end() || it->first > 2 * n + 4096) return nullptr;
    void *p = it->second;
    *cap = it->first;
    held_ -= it->first;
    free_.erase(it);
    return p;
  }
  bool give(void *p, size_t cap, uint64_t era) {
    std::lock_guard<std::mutex> lk(mu_);
    if (era != era_ || cap > LARGEST || held_ + cap > KEEP) return false;
    free_.emplace(cap, p);
    held_ += cap;
    return true;
  }
  // the transfer block if it is free and holds n bytes (a smaller one makes way
  // for the larger that the caller now allocates)
  void *take_transfer(size_t n, size_t *cap, uint64_t *era) {
    std::lock_guard<std::mutex> lk(mu_);
    *era = era_;
    void *p = transfer_;
    transfer_ = nullptr;
    if (p && transfer_cap_ < n) {
      (void)hipFree(p);
      p = nullptr;
    }
    *cap = transfer_cap_;
    return p;
  }
  bool give_transfer(void *p, size_t cap, uint64_t era) {
    std::lock_guard<std::mutex> lk(mu_);
    if (era != era_ || cap > LARGEST || transfer_) return false;
    transfer_ = p;
    transfer_cap_ = cap;
    return true;
  }
  // (at once: a block given back in between would be kept for the new stream)
  void new_stream() {
    std::lock_guard<std::mutex> lk(mu_);
    empty();
    ++era_;
  }
  void clear() {
    std::lock_guard<std::mutex> lk(mu_);
    empty();
  }

 private:
  void empty() {
    for (auto &b : free_) (void)hipFree(b.second);
    free_.clear();
    held_ = 0;
    if (transfer_) (void)hipFree(transfer_);
    transfer_ = nullptr;
  }

  std::mutex mu_;
  std::multimap<size_t, void *> free_;
  void *transfer_ = nullptr;
  size_t held_ = 0, transfer_cap_ = 0;
  uint64_t era_ = 0;
};

// A device allocation that frees itself, from and back to a context's pool
// when it is allocated with one.
struct DevBuf {
  void *p = nullptr;
  size_t bytes = 0;
  DevBuf() = default;
  DevBuf(const DevBuf &) = delete;
  DevBuf &operator=(const DevBuf &) = delete;
  ~DevBuf() { release(); }
  void release() {
    if (p && !(pool_ && (transfer_ ? pool_->give_transfer(p, cap_, era_) : pool_->give(p, cap_, era_))))
      (void)hipFree(p);
    p = nullptr;
    pool_ = nullptr;
    transfer_ = false;
    bytes = cap_ = 0;
  }
  // n bytes, from the pool and back to it
  int alloc(size_t n, DevPool *pool) {
    release();
    if (n == 0) n = 16;
    p = pool->take(n, &cap_, &era_);
    if (!p)
      if (int rc = allocate(n, pool)) return rc;
    pool_ = pool;
    bytes = n;
    return THRML_OK;
  }
  // n bytes for a host transfer
  int alloc_transfer(size_t n, DevPool *pool) {
    release();
    p = pool->take_transfer(n, &cap_, &era_);
    if (!p)
      if (int rc = allocate(std::max<size_t>(n, 1u << 16), pool)) return rc;
    pool_ = pool;
    transfer_ = true;
    bytes = n;
    return THRML_OK;
  }
  // n bytes that go back to the device: for buffers that a context keeps itself
  int alloc_own(size_t n, DevPool *pool) {
    release();
    if (n == 0) n = 16;
    if (int rc = allocate(n, pool)) return rc;
    bytes = n;
    return THRML_OK;
  }
  template <class T>
  T *as() const {
    return reinterpret_cast<T *>(p);
  }

 private:
  int allocate(size_t n, DevPool *pool) {
    hipError_t e = hipMalloc(&p, n);
    if (e != hipSuccess) {  // what the pool holds may be what is missing
      pool->clear();
      e = hipMalloc(&p, n);
      // taken back, or the next launch's check would find the failure
      (void)hipGetLastError();
    }
    if (e != hipSuccess) {
      p = nullptr;
      return fail(THRML_ENOMEM, "device allocation of " + std::to_string(n) + " bytes failed: " +
                                    hipGetErrorString(e));
    }
    cap_ = n;
    return THRML_OK;
  }

  DevPool *pool_ = nullptr;
  bool transfer_ = false;
  size_t cap_ = 0;
  uint64_t era_ = 0;
};

// Declared after host memory that copies queued on a stream read or write: they
// have ended when the scope is left, on whatever path.
class StreamWait {
 public:
  explicit StreamWait(hipStream_t s) : stream_(s) {}
  StreamWait(const StreamWait &) = delete;
  StreamWait &operator=(const StreamWait &) = delete;
  ~StreamWait() {
    if (open_) (void)hipStreamSynchronize(stream_);
  }
  hipError_t now() {
    open_ = false;
    return hipStreamSynchronize(stream_);
  }

 private:
  hipStream_t stream_;
  bool open_ = true;
};

struct TimingSlot {
  std::vector<hipEvent_t> ev;  // pairs
  std::vector<uint64_t> n;     // half-sweeps of each pair's launch
  size_t used = 0;
  hipEvent_t span0 = nullptr;  // span mode: recorded before the first launch
  uint64_t span_n = 0;         // span mode: launches since span0
};

}  // namespace thrml

struct thrml_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  bool own_stream = false;
  int timing = 0;  // 0 off, 1 an event pair per launch, 2 one span of launches
  // per kernel class: recorded (start, stop) event pairs
  thrml::TimingSlot slots[2];
  double acc_ms[2] = {0, 0};
  uint64_t acc_n[2] = {0, 0};
  int cu_count = 256;
  // The expanded stream keys of the run in flight, grown as needed and reused
  // by later runs (calls on one context are ordered on its stream).  run_mu
  // serialises the runs of host threads that share the context.
  thrml::DevBuf keys;
  std::mutex run_mu;
  thrml::DevPool pool;  // what this context's objects have let go of
  int flush_timing(int k);
  int time_begin(int k, hipEvent_t *start);
  int time_end(int k, hipEvent_t start, uint64_t half_sweeps = 1);
};

struct thrml_prog {
  thrml_ctx *ctx = nullptr;
  uint32_t kind = 0;
  uint32_t n_free = 0, n_clamped = 0;
  uint32_t planes = 1;            // bit planes per node
  uint32_t q = 2;                 // categories (2 for spins)
  std::vector<uint64_t> blk_off;  // [n_free + n_clamped + 1]
  uint64_t n_total = 0;
  std::vector<int64_t> node_pos;  // node -> global position (-1: not in any block)
  std::vector<uint32_t> pos_node;
  // Ising parameters (host copies: hinton init and energies)
  float beta = 1.0f;
  std::vector<float> bias_raw;    // [n_nodes]
  std::vector<uint32_t> eu, ev;
  std::vector<float> w_raw;
  uint64_t device_bytes = 0;

  // --- lattice path: one table row of 16 keystream-word thresholds per free
  // position, indexed by the (left, right, up, down) neighbour bits.
  uint32_t L = 0, half = 0;
  uint32_t parity[2] = {0, 0};    // column parity of block b in row 0
  thrml::DevBuf table;            // [n_free_total][16] u32

  // --- CSR path (Ising and Potts): per free position, slots in reference
  // order.  Ising: slot = {tail position, fl(beta*J)}; Potts: u-role slots
  // then v-role slots, slot = {tail position, edge id}.
  thrml::DevBuf row_off;          // [n_free_total + 1] u32 (Ising) / [n_free_total + 1] u32 (Potts u+v)
  thrml::DevBuf slots;            // [n_slots] uint2
  thrml::DevBuf bias_w;           // Ising: [n_free_total] f32 fl(beta*b); Potts: [n_free_total][q]
  thrml::DevBuf uend;             // Potts: [n_free_total] end of the u-role slots
  thrml::DevBuf wts;              // Potts: [E+1][q][q], W[e][a][b] couples x_u = a, x_v = b (edge E: zeros)
  thrml::DevBuf wts_t;            // Potts: [E+1][q][q] transposes (edge E: zeros)
  thrml::DevBuf pslots;           // Potts: [n_free_total][2*pm] uint2, role-padded slots
  uint32_t pm = 0;                // Potts: padded role width (2 or 4), 0 = unpadded kernel
  uint32_t cat_bytes = 1;         // byte-layout programs: bytes per (position, chain), 2 for q > 256
  uint32_t mean_slots = 0;        // Potts, discrete: slots per free position, rounded
  uint64_t n_edges = 0;
  bool intra_block_edges = false;
  // Superblocks (crates/thrml-samplers/src/program.rs:28-64): superblock s
  // holds the free blocks sb_off[s] .. sb_off[s+1]-1, all sampled from the
  // state before it.  A staged block writes its new state into the state's
  // staging buffer, which mirrors positions blk_off[first block of s] ..
  // + stage_width[s] (rows of stage_width[s] positions), and the superblock's
  // staged range is copied into place after its last block.  A block is
  // staged when a later block of its superblock reads the state, or when the
  // program has edges inside a block (it then reads its own positions).
  std::vector<uint32_t> sb_off;       // [n_superblocks + 1]
  std::vector<uint32_t> blk_sb;       // free block -> superblock
  std::vector<uint8_t> staged;        // per free block
  std::vector<uint64_t> stage_width;  // per superblock: positions staged (0: none)
  uint64_t stage_max = 0;             // the largest stage_width
  // Ising CSR: per free block, the most slots in a window of 4, 8, 16, 32
  // sites (windows aligned at multiples of their size)
  std::vector<uint32_t> csr_win[4];
  std::vector<uint32_t> csr_maxdeg;  // largest slot count of a site, per free block

  // --- resident runs of small Ising programs (res_T = 0: not eligible)
  uint32_t res_T = 0;              // threads per workgroup (one chain)
  uint32_t res_parts = 0, res_kb = 0, res_pf = 0;
  uint32_t res_ent = 0;            // register kernel: entries per wave (0: streaming kernel)
  double res_work = 0.0, res_deg = 0.0;  // us per sweep besides the blocks', slots per site
  thrml::DevBuf r_tab;             // its tables and slot data, at r_off
  uint64_t r_off[5] = {};

  // --- dense bipartite path.  Side 0 ("visible") holds the rows of W, side 1
  // ("hidden") its columns; dense_side[b] is the side of block b (blocks are
  // free ++ clamped in any order) and side_off[s] the global offset of side s.
  uint32_t V = 0, H = 0, Vp = 0, Hp = 0;  // sizes, padded to multiples of 256 (row tiles and K slices)
  uint32_t dense_side[2] = {0, 1};
  uint64_t side_off[2] = {0, 0};
  // Each weight is the exact sum of dense_pieces bf16 values (1 for weights
  // that are bf16 already, up to 3 for any f32); the pieces of a row follow
  // each other along K, each padded alike, so a row holds pieces * Kp values.
  uint32_t dense_pieces = 1;
  thrml::DevBuf w_vh;             // bf16 [Vp][pieces * Hp] (K = H contiguous)
  thrml::DevBuf w_hv;             // bf16 [Hp][pieces * Vp]
  thrml::DevBuf dense_bias;       // f32 [Vp + Hp] fl(beta*b): visible at 0, hidden at Vp

  // --- general discrete factor programs.  blk_kind[b] is 0 for a block of
  // spin nodes, 1 for categorical nodes.  Per free position (row_off), slots
  // in the reference's order (groups in order, head positions ascending),
  // each a uint4 {weight offset, first categorical tail's position or
  // DISC_NONE, the spin tail's position (n_sp = 1) or the first spin tail in
  // d_sp, n_sp | group start << 8 | axis << 9};
  // axis 0: entry c of the row, 2: x * q + c (a head-U slot points at the
  // transposed copy of its factor's weights, so every categorical head reads
  // q contiguous floats; axis 1, c * q + x, is not produced).  Energy terms:
  // one per factor row whose nodes all have positions, two uint4
  // {weight row, first spin in d_tsp, n_sp, x0 position | DISC_NONE},
  // {x1 position | DISC_NONE, d2, 0, 0}.
  std::vector<uint8_t> blk_kind;
  thrml::DevBuf d_slots, d_sp, d_w, d_terms, d_tsp;
  uint64_t d_nterms = 0;

  // --- energies (built on the first energy call): endpoint positions of
  // the edges whose endpoints both have a position, raw J, raw b per position
  std::mutex en_mu;
  bool en_ready = false;
  uint64_t en_ne = 0;
  thrml::DevBuf en_pos;           // [en_ne] uint2
  thrml::DevBuf en_w;             // [en_ne] f32 (spin programs)
  thrml::DevBuf en_bias;          // [n_total] f32 (spin programs)
};

struct thrml_state {
  thrml_prog *prog = nullptr;
  thrml_ctx *ctx = nullptr;  // the program's context: destroy needs no program
  uint32_t C = 0;     // chains
  uint32_t G = 0;     // chain groups of 64
  thrml::DevBuf words;  // spin programs: [G * planes][n_total] u64
  thrml::DevBuf cat;    // categorical programs: [n_total][Cp] u8, chains fastest
  uint32_t Cp = 0;      // C rounded up to 4
  thrml::DevBuf scratch;// per-block staging for programs with intra-block edges / dense operands
  thrml::DevBuf flag;   // u32: the first column an import check refuses, or IMPORT_OK
  // CSR spin programs with at most 32 chains and no staged block: [n_total]
  // u32, the low halves of the state words (the high halves are zero).  The
  // sweep kernel gathers neighbour states here, half the footprint of the
  // words, and writes both; each run refreshes it from the words first.
  // low_live: it holds the current spins (set within a run that keeps it).
  thrml::DevBuf low;
  bool low_live = false;
  // resident runs of several chains: [C][ceil(n_total / 64)] u64, the chains'
  // spins at a run's end
  thrml::DevBuf bits;
  // dense path operands: spin-down bits per block, one bit vector per chain
  // (bit k%32 of word k/32 is 1 when the spin at block position k is down)
  uint32_t C_pad = 0;     // chains rounded up to the 256-wide GEMM tile
  thrml::DevBuf dbits_v;  // [C_pad][Vp/32] u32
  thrml::DevBuf dbits_h;  // [C_pad][Hp/32] u32
  uint64_t plane_stride() const { return prog->n_total; }
};

// A moment specification bound to a program (ising_moment_spec +
// MomentAccumulatorObserver::new, crates/thrml-observers/src/moment.rs:52,125-150).
// native: lattice programs count in the sweep kernels' layout (ones per
// global position, diff per block-1 site and direction) and slot1/slot2 map
// the requested nodes/pairs onto those counters; otherwise the moment kernel
// counts per requested entry at the positions npos/ppos.
struct thrml_moments {
  thrml_prog *prog = nullptr;
  thrml_ctx *ctx = nullptr;  // the program's context: destroy needs no program
  bool native = false;
  uint64_t n1 = 0, n2 = 0;      // requested nodes, pairs
  uint64_t len1 = 0, len2 = 0;  // counters
  // one allocation: native, the counter index per requested entry (slot1,
  // slot2), else the positions of nodes and of pair endpoints (npos, ppos);
  // u32 counters of the current fold period, u64 totals
  thrml::DevBuf buf;
  uint32_t *slot1 = nullptr, *slot2 = nullptr, *npos = nullptr, *ppos = nullptr;
  uint32_t *cnt1 = nullptr, *cnt2 = nullptr;
  uint64_t *acc1 = nullptr, *acc2 = nullptr;
  size_t clear_bytes = 0;       // totals and counters, from acc1 on
  thrml::DevBuf out;            // the sums of a run whose outputs lie on the host, from the first one on
};

// A general moment observer (MomentAccumulatorObserver with any spec): row r
// multiplies f(x) over the positions pos[row_off[r] .. row_off[r+1]].
struct thrml_observer {
  thrml_prog *prog = nullptr;
  thrml_ctx *ctx = nullptr;
  uint64_t n_rows = 0;
  bool transform = true;
  double max_row_log2 = 0.0;  // byte states: log2 of the largest |product| a row can take
  thrml::DevBuf row_off;  // [n_rows + 1] u64
  thrml::DevBuf pos;      // positions, u32
  thrml::DevBuf acc;      // [n_rows] int64 sums
};

namespace thrml {
// Allocates buf for v and queues the upload on the context's stream.
template <class T>
int upload_to(thrml_ctx *ctx, DevBuf &buf, const std::vector<T> &v) {
  if (int rc = buf.alloc(v.size() * sizeof(T), &ctx->pool)) return rc;
  if (!v.empty())
    THRML_HIP(hipMemcpyAsync(buf.p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice,
                             ctx->stream));
  return THRML_OK;
}

// A dense bipartite program: W[i][j] couples node side_nodes[0][i] with node
// side_nodes[1][j]; block k of the global state is side block_side[k], and
// the first n_free blocks are free.  Node ids lie below n_nodes.
struct DenseSpec {
  uint32_t n_nodes = 0;
  std::vector<uint32_t> side_nodes[2];
  std::vector<float> w;          // [n0][n1]
  std::vector<float> bias;       // [n_nodes] raw biases
  float beta = 1.0f;
  uint32_t block_side[2] = {0, 1};
  uint32_t n_free = 2;
};
int dense_program_create(thrml_ctx *ctx, const DenseSpec &d, thrml_prog **out);
// The bf16 pieces w = p[0] + p[1] + p[2] (exact; unused pieces 0) of an f32
// weight, each the nearest bf16 to what the earlier pieces leave.  Returns the
// number of pieces needed (0..3), or -1 when w is not finite or a nonzero
// piece would be a subnormal bf16 (the sum could then be inexact).
__host__ __device__ int bf16_pieces(float w, uint16_t p[3]);

constexpr uint32_t DISC_NONE = 0xffffffffu;
// Programs whose state is one byte per (position, chain): [n_total][Cp].
inline bool byte_layout(const thrml_prog *p) { return p->kind == K_POTTS || p->kind == K_DISCRETE; }
// Values a block of a byte-layout program accepts: 2 for spins, else q.
inline uint32_t block_q(const thrml_prog *p, uint32_t b) {
  return (p->kind == K_DISCRETE && !p->blk_kind[b]) ? 2u : p->q;
}

// Superblocks: set_superblocks checks offsets[n_sb + 1] over the free blocks
// (n_sb = 0: one superblock per free block); plan_staging then decides which
// blocks write through the staging buffer (needs intra_block_edges).
int set_superblocks(thrml_prog *p, uint32_t n_sb, const uint32_t *offsets);
void plan_staging(thrml_prog *p);
// Where free block b writes its new state: in place (false), or into the
// staging buffer at position offset *off with rows of *width positions.
inline bool stage_target(const thrml_prog *p, uint32_t b, uint64_t *off, uint64_t *width) {
  if (!p->staged[b]) return false;
  const uint32_t s = p->blk_sb[b];
  *off = p->blk_off[b] - p->blk_off[p->sb_off[s]];
  *width = p->stage_width[s];
  return true;
}
// Copies superblock s's staged range into the state (no-op when none).
int commit_superblock(thrml_prog *p, thrml_state *st, uint32_t s);

// kernels (launchers return THRML_OK or an error)
// Key tree of one run: run_blocks (mode 0) or sample_with_observation
// (mode 1) with n_chains chains of the root key.
struct KeyPlan {
  uint64_t root;
  uint32_t C, C_pad, n_blocks, mode;
  uint64_t n_iters;                       // mode 0
  uint64_t n_warmup, n_samples, steps;    // mode 1
};
int launch_key_schedule(thrml_ctx *ctx, const KeyPlan &kp, uint64_t s0, uint32_t n_sweeps,
                        uint32_t *d_keys);
// Moment counters of lattice programs: ones[pos] per global position,
// diff[i*4 + d] per block-local site i of block 1 and neighbour direction d
// (0 left, 1 right, 2 up, 3 down).
struct LatticeMoments {
  uint32_t *ones;
  uint32_t *diff;
};
int launch_lattice_half(thrml_prog *p, thrml_state *st, uint32_t b, const uint32_t *d_keys,
                        const LatticeMoments *mom);
int launch_lattice_moments(thrml_state *st, const LatticeMoments *mom);
int launch_csr_half(thrml_prog *p, thrml_state *st, uint32_t b, const uint32_t *d_keys);
// refreshes st->low from the state words (CSR programs that keep it)
int launch_pack_low(thrml_state *st);
// Resident runs: tables at program creation, and n_sweeps whole sweeps whose
// expanded keys start at d_keys.
int resident_tables(thrml_prog *p, const std::vector<uint32_t> &row_off, const uint32_t *d_row_off,
                    const uint2 *d_slots, const float *d_bias, std::vector<uint8_t> &keep);
bool resident_pays(const thrml_prog *p, const thrml_state *st, uint64_t n_sweeps, uint64_t n_seg,
                   bool fused);
int launch_resident(thrml_prog *p, thrml_state *st, const uint32_t *d_keys, uint32_t n_sweeps);
void csr_windows(thrml_prog *p, const std::vector<uint32_t> &row_off);
int launch_potts_half(thrml_prog *p, thrml_state *st, uint32_t b, const uint32_t *d_keys);
int launch_discrete_half(thrml_prog *p, thrml_state *st, uint32_t b, const uint32_t *d_keys);
int discrete_energy(thrml_prog *p, thrml_state *st, double *out);
// out[c] = -(sum over rows k < n of part[k * stride + c]) for the state's chains
int reduce_energy(thrml_prog *p, uint32_t C, const double *part, uint32_t n, uint32_t stride,
                  double *out);
// Dense programs: one half-sweep of side `side` (0 rows of W, 1 columns).
int launch_dense_half(thrml_prog *p, thrml_state *st, uint32_t side, const uint32_t *d_keys);
int launch_lattice_table(thrml_prog *p, const uint32_t *d_dir, const uint2 *d_slots, const float *d_bias);
int launch_hinton(thrml_prog *p, thrml_state *st, uint32_t b, const uint32_t *d_key8,
                  const float *d_prob);
// State import and export of positions p0 .. p0 + n - 1 from / to device memory
// that holds one row of `stride` values per chain, at columns col0 .. col0 + n - 1.
// An import writes nothing unless *d_bad is IMPORT_OK (launch_import_check).
int launch_potts_pack(thrml_state *st, uint64_t p0, uint32_t n, const void *d_src, int dtype,
                      uint64_t stride, uint64_t col0, const uint32_t *d_bad);
int launch_potts_unpack(thrml_state *st, uint64_t p0, uint32_t n, void *d_dst, int dtype, uint64_t stride,
                        uint64_t col0);
int launch_pack(thrml_state *st, uint64_t p0, uint32_t n, const void *d_src, int dtype,
                uint64_t stride, uint64_t col0, const uint32_t *d_bad);
int launch_unpack(thrml_state *st, uint64_t p0, uint32_t n, void *d_dst, int dtype, uint64_t stride,
                  uint64_t col0);
int launch_potts_weights(thrml_ctx *ctx, float *w, float *wt, uint64_t n_edges, uint32_t q,
                         uint64_t n_w);
int launch_moments(thrml_state *st, const uint32_t *d_npos, uint64_t n1, const uint32_t *d_ppos,
                   uint64_t n2, uint32_t *d_ones, uint32_t *d_diff);
// Dense programs: recompute side `side`'s spin-down operand bits from the
// state words.
int launch_dense_sync_act(thrml_state *st, uint32_t side);
int launch_fold_counts(thrml_ctx *ctx, uint32_t *cnt, uint64_t *acc, uint64_t n);
// Adds one observation of st to obs->acc.
int launch_observe(thrml_state *st, thrml_observer *obs);
int launch_finalize_moments(thrml_ctx *ctx, const uint32_t *cnt1, const uint64_t *acc1,
                            const uint32_t *slot1, uint64_t n1, const uint32_t *cnt2,
                            const uint64_t *acc2, const uint32_t *slot2, uint64_t n2, int64_t cn,
                            int64_t *out1, int64_t *out2);
// Per-chain energies of a state into host out[C] (spin: lattice, CSR and
// dense programs; categorical programs).
int spin_energy(thrml_prog *p, thrml_state *st, double *out);
int potts_energy(thrml_prog *p, thrml_state *st, double *out);
// Dense programs: the coupling term sum_h s_h sum_v W[v][h] s_v of every
// chain, as f64 partials [Hp/32][C_pad] (one per 32 hidden sites and chain).
int launch_dense_energy(thrml_prog *p, thrml_state *st, double *part);
int launch_sigmoid_bernoulli(thrml_ctx *ctx, const float *g, const float *u, float *o, uint64_t n);
int launch_fast_math_check(thrml_ctx *ctx, float out[3]);
// *d_bad = IMPORT_OK, and lowered to the first column among col0 .. col0 + n - 1
// that holds something else than a state value 0..q-1 in one of C rows.
constexpr uint32_t IMPORT_OK = 0xffffffffu;
int launch_import_reset(thrml_ctx *ctx, uint32_t *d_bad);
int launch_import_check(thrml_ctx *ctx, const void *d_src, int dtype, uint32_t C, uint32_t n,
                        uint64_t stride, uint64_t col0, uint32_t q, uint32_t *d_bad);
// The per-device cached self-check (run at the first call on a device).  With
// ok_out NULL it fails with THRML_EUNSUPPORTED when the bounds do not hold;
// otherwise it reports the values and the verdict.
int fast_math_gate(thrml_ctx *ctx, float *v_out, int *ok_out);
// categories of a categorical node: one byte of state per (position, chain)
constexpr uint32_t POTTS_MAX_Q = 256;       // one byte of state per node
constexpr uint32_t POTTS_WIDE_MAX_Q = 65536;  // Potts programs: two bytes above 256
// Lanes per (site, chain) item of the wide kernels (q > 16): P lanes split a
// site's keystream blocks of 16 categories, nb = (offset of its first word +
// q + 15) / 16 of them, in ceil(nb / P) steps each.  Fitted to launches on
// MI355X (tori of side 16 .. 256 and Erdos-Renyi graphs, q = 17 .. 256, 1 ..
// 128 chains; bias-only blocks of q = 300 .. 16384), in us:
//   2 + steps (1.2 + 0.8 slots) + 1.1 items P steps (17 + 5 slots) / 10^6;
// for P = 1 and 2, which read one and two slots at a time, 1.5 and 1.1 instead
// of 0.8 and 1 instead of 1.1.  The first part is one wave's chain of dependent
// loads, the second the whole chip's issue, to which idle lanes count as much
// as busy ones.
// The rule is taken for each block; a graph's colour blocks differ in size, so
// that it can beat any one P.  us per launch, averaged over the program's blocks,
// with the same P for all of them and by the rule:
//                                          P = 1     2     4     8    16   rule
//   E-R 10007 deg 8, q = 21, 50 chains        37    22    20    30    51     20
//   E-R 10007 deg 8, q = 21, 25 chains        38    21    15    19    30     16
//   E-R 10007 deg 8, q = 21, 100 chains       40    28    30    51    92     26
//   E-R 20000 deg 6, q = 24, 30 chains        35    19    23    35    62     18
//   E-R 10007 deg 8, q = 48, 50 chains        66    39    28    38    60     28
//   E-R 1000 deg 8, q = 100, 8 chains        108    46    20    11    11     11
//   128^2, q = 32, 128 chains                 77    67   121   233   456     67
//   16^2, q = 256, 8 chains                   63    33    17    10   6.7    6.8
inline uint32_t wide_lanes(uint32_t q, uint64_t items, uint32_t slots) {
  uint32_t step = 16u;  // the offsets a site's first word can have: multiples of gcd(q, 16)
  while (q % step) step /= 2u;
  uint32_t best = 1u;
  double best_t = 0.0;
  for (uint32_t P = 1; P <= (q > 256u ? 64u : 16u); P *= P == 16u ? 4u : 2u) {
    if (items * P > (1ull << 32) - 256u) break;  // a launch, whole workgroups, stays below 2^32 threads
    double steps = 0.0;
    for (uint32_t o = 0; o < 16u; o += step) steps += (double)(((o + q + 15u) / 16u + P - 1u) / P);
    steps /= 16u / step;
    const double t = 2.0 + steps * (1.2 + (P == 1u ? 1.5 : P == 2u ? 1.1 : 0.8) * slots) +
                     (P > 2u ? 1.1 : 1.0) * (double)items * P * steps * (17.0 + 5.0 * slots) * 1e-6;
    if (P == 1u || t < best_t) {
      best = P;
      best_t = t;
    }
  }
  return best;
}

// Weight rows may be loaded up to 15 floats past either end (load_chunk16):
// their arrays carry ROW_PAD floats before and after (256 bytes, so that rows
// of 32 floats still lie in one cache line each: 64 bytes cost a 256^2 torus
// of 32 categories 8 %).
constexpr uint32_t ROW_PAD = 64;
inline float *padded(const DevBuf &b) { return b.as<float>() + ROW_PAD; }

constexpr uint32_t BATCH_GATHER_MAX_INDICES = 64;
struct BatchGatherStrides {
  uint32_t s[BATCH_GATHER_MAX_INDICES];
  uint32_t batch_stride;
};
int launch_batch_gather(thrml_ctx *ctx, const float *w, uint64_t n_w, const int32_t *idx,
                        uint64_t batch, uint32_t n_idx, const BatchGatherStrides &st, float *out);
int launch_gumbel_argmax(thrml_ctx *ctx, const float *l, const float *u, int32_t *o, uint64_t n,
                         uint32_t q);
}  // namespace thrml

// k_resident.hip -- whole runs of sweeps of a small Ising program in one
// launch (gfx950).
//
// The per-block kernels (k_ising.hip) launch once per block and sweep, with a
// chain per lane; a small model then spends its time between launches (about
// 3.8 us per half-sweep however little there is to do).  Here a workgroup takes one
// chain and keeps its whole state in LDS for the run: lanes are sites, a
// half-sweep ends with a workgroup barrier instead of a launch, and no other
// workgroup is waited for.  Sites, slots, keystream words and decisions are
// those of the per-block kernels (same sums in the same order, same words,
// spin_decision), so the states are identical.
//
// Bound: instruction issue of one CU (16 waves, one chain): 42 vector
// instructions per 64 sites with the records in registers (683 million for the
// 2000 half-sweeps of 8192 slices of a 64^2 torus with 256 chains), 23 of them
// the keystream.  Measured, per sweep: 64^2 torus, 256 chains 5.1 -> 1.7 us (7.35
// -> 1.80 ms for 1000 sweeps and the read-back); Erdos-Renyi graph of 20011
// nodes, mean degree 7, 200 chains 48 -> 23 us; two 40^2 layers with 13
// neighbours each, one chain 8.0 -> 4.2 us.
//
// Phases.  The keystream depends on nothing but the keys, so it is computed
// ahead: lane t computes the t-th ChaCha8 block of the coming half-sweeps
// (all lanes busy, up to one block per lane) into LDS, and the half-sweeps
// they cover follow.  A program whose sweep takes at most as many blocks as
// the workgroup has lanes runs several sweeps per phase (one part); a larger
// one splits its sweep into several parts.
//
// Tables (built once per program).  The sites of a piece (a block, or the
// part of a block that one phase covers) are sorted by slot count, so that
// the 64 sites of a slice have nearly as many slots each.  Slot records lie
// two per uint4, lane-interleaved (pair g of lane l at 64 g + l); slots past a
// site's last have weight 0 (they add +-0 to a sum that is never -0, as in the
// CSR kernel).  A slice is one or more entries of at most PF pairs; before
// the pairs of its last entry lie the 64 site records {global position | byte offset of
// the site's keystream word << 16, bias}.  Padding sites write to a spare byte.
// A wave's entries form a ring that it walks for the whole run.
#include <algorithm>
#include <cstring>

#include "dev_util.hpp"
#include "internal.hpp"

namespace thrml {

struct ResArgs {
  uint64_t *words;          // state words, group 0; written here for one chain
  uint64_t *bits;           // [C][n_words] new spins of each chain, 64 positions per word
  const uint32_t *keys;     // [n_sweeps][n_blocks][C_pad][KEY_WORDS]
  const ResPiece *pieces;
  const ResPart *parts;
  const uint4 *ents;        // the waves' entries {byte offset of the data, meta, next entry, 0}
  const uint4 *woff;        // [n_parts][waves] {first entry, entries, leading barriers, ring's first entry}
  const uint8_t *data;      // site records and slot pairs {position, weight, position, weight}
  uint32_t n_total, n_words, n_sweeps, n_blocks, C_pad;
  uint32_t n_parts, per_phase;  // sweeps per phase (1 with several parts)
  FastDiv div_kb;           // by the keystream blocks of one sweep (one part)
};

// Wave-uniform tables through the scalar cache.
template <class T>
__device__ __forceinline__ T uload(const T *p, uint32_t i) {
  typedef const __attribute__((address_space(4))) uint32_t cu32;
  cu32 *q = (cu32 *)(uintptr_t)(p + i);
  struct { uint32_t w[sizeof(T) / 4]; } r;
#pragma unroll
  for (uint32_t k = 0; k < sizeof(T) / 4; ++k) r.w[k] = q[k];
  return __builtin_bit_cast(T, r);
}

// LDS written by this wave is visible to the workgroup, and the waves meet.
// Only LDS is shared between waves, so global loads in flight are not waited for.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" : : : "memory");
}

// An entry's meta word: slot pairs, whether it is its slice's last (its sites
// are then decided), and the barriers after it.
__host__ __device__ constexpr uint32_t ent_meta(uint32_t ng, bool last, uint32_t nbar) {
  return ng | (last ? 16u : 0u) | (nbar << 5);
}
constexpr uint32_t RES_SITES = 64u * sizeof(uint2);   // bytes of a slice's site records
constexpr uint32_t RES_PAIRS = 64u * sizeof(uint4);   // bytes of a slot pair of 64 sites
constexpr uint32_t RES_MAX_PF = 8;

// Word of keystream block k of a part (its blocks counted from the sweep's
// first) that holds word j of the block: a block's four 16-byte quarters are
// swapped by its index, so that the 16 lanes of one write pass cover all LDS
// banks.
__host__ __device__ constexpr uint32_t res_word(uint32_t k, uint32_t j) {
  return k * 16u + (j ^ (((k >> 2) & 3u) << 2));
}

// The keystream of one phase: lane t computes its t-th block into LDS.
__device__ __forceinline__ void res_keystream(const ResArgs &a, uint32_t part, uint32_t s0,
                                              uint32_t ns, uint32_t chain, uint8_t *ks) {
  const uint32_t t = threadIdx.x;
  const ResPart pt = uload(a.parts, part);
  if (t < ns * pt.kb) {
    const uint32_t sp = a.n_parts == 1u ? fdiv(t, a.div_kb) : 0u;
    const uint32_t r = t - sp * pt.kb;
    uint32_t blk = 0u, ctr = 0u;
    for (uint32_t q = pt.piece0; q < pt.piece1; ++q) {
      const ResPiece pc = uload(a.pieces, q);
      if (r >= pc.kb0) {
        blk = pc.blk;
        ctr = pc.site0 / 16u + (r - pc.kb0);
      }
    }
    uint32_t key[KEY_WORDS];
    load_keyx(a.keys + (size_t)((s0 + sp) * a.n_blocks + blk) * a.C_pad * KEY_WORDS, chain, key);
    uint32_t x[16];
    chacha_block_pre<8>(key, ctr, x);
    uint8_t *const o = ks + sp * pt.kb * 64u;
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q)
      *reinterpret_cast<uint4 *>(o + res_word(r, 4u * q) * 4u) =
          make_uint4(x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]);
  }
}

// A chain's spins from the state words into LDS: f(position, 1 for up).
template <class F>
__device__ __forceinline__ void res_load_state(const ResArgs &a, uint32_t chain, F &&f) {
  const uint32_t *w32 = reinterpret_cast<const uint32_t *>(a.words + (size_t)(chain >> 6) * a.n_total) +
                        ((chain >> 5) & 1u);
  for (uint32_t p = threadIdx.x; p < a.n_total; p += blockDim.x)
    f(p, (w32[2u * p] >> (chain & 31u)) & 1u);
}

// The chain's spins, 64 positions per word; up(position) tells a spin.  A single
// chain's state words hold nothing else, and no other workgroup writes them:
// they are written at once, which saves resident_commit_kernel's launch (one
// chain of a 10^2 torus, 20 observed states: 238 -> 190 us; of two 40^2 layers,
// a training step of 20 observations: 1750 -> 1668 us).
template <class F>
__device__ __forceinline__ void res_store_bits(const ResArgs &a, uint32_t chain, F &&up) {
  const uint32_t lane = threadIdx.x & 63u;
  if (gridDim.x == 1u) {
    for (uint32_t p = threadIdx.x; p < a.n_total; p += blockDim.x) a.words[p] = up(p) ? 1ull : 0ull;
    return;
  }
  for (uint32_t p0 = threadIdx.x & ~63u; p0 < a.n_total; p0 += blockDim.x) {
    const uint32_t p = p0 + lane;
    const uint64_t m = __builtin_amdgcn_ballot_w64(p < a.n_total && up(p));
    if (lane == 0u) a.bits[(size_t)chain * a.n_words + p0 / 64u] = m;
  }
}

// fl(acc + (+-w)) with w negated where the neighbour (a state byte, read
// sign-extended) is down
__device__ __forceinline__ float res_add(float acc, uint32_t w, int32_t d) {
  return acc + bitsf(w ^ ((uint32_t)d & 0x80000000u));
}

// Decides the site of record sb, whose slots sum to acc.
__device__ __forceinline__ void res_decide(int8_t *st, const uint8_t *kss, uint32_t sb, float bias,
                                           float acc) {
  const uint32_t wd = *reinterpret_cast<const uint32_t *>(kss + (sb >> 16));
  const uint64_t up = spin_decision_mask((0.0f + bias) + acc, wd);
  st[sb & 0xffffu] = lane_bit(up) ? 0 : -128;
}

// State: one LDS byte per position, 0x80 for a down spin, and a spare one.
__device__ __forceinline__ uint32_t res_state_bytes(uint32_t n_total) { return (n_total + 16u) & ~15u; }

// Register kernel (one part, at most NE entries per wave, at most 4 slots per
// site): every lane keeps its sites' slot records in registers for the whole
// run, so a half-sweep reads nothing but LDS.
template <int NE>
__global__ __launch_bounds__(1024) void resident_reg_kernel(ResArgs a) {
  extern __shared__ __align__(16) uint8_t rlds[];
  int8_t *const st = reinterpret_cast<int8_t *>(rlds);
  uint8_t *const ks = rlds + res_state_bytes(a.n_total);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t chain = blockIdx.x;
  res_load_state(a, chain, [&](uint32_t p, uint32_t up) { st[p] = up ? 0 : -128; });
  const uint4 wo = uload(a.woff, wave);

  uint32_t site[NE];
  float bias[NE];
  uint32_t pos[NE][2];  // two 16-bit positions per word
  uint32_t w[NE][4];
  uint32_t nbar[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    uint2 sb = make_uint2(a.n_total, 0u);
    uint4 r0 = make_uint4(0u, 0u, 0u, 0u), r1 = r0;
    nbar[e] = 0u;
    if ((uint32_t)e < wo.y) {
      const uint4 en = uload(a.ents, wo.x + e);
      const uint32_t ng = en.y & 15u;
      nbar[e] = en.y >> 5;
      const uint8_t *d = a.data + en.x;
      sb = reinterpret_cast<const uint2 *>(d)[lane];
      if (ng > 0u) r0 = reinterpret_cast<const uint4 *>(d + RES_SITES)[lane];
      if (ng > 1u) r1 = reinterpret_cast<const uint4 *>(d + RES_SITES + RES_PAIRS)[lane];
    }
    site[e] = sb.x;
    bias[e] = bitsf(sb.y);
    pos[e][0] = r0.x | (r0.z << 16);
    pos[e][1] = r1.x | (r1.z << 16);
    w[e][0] = r0.y;
    w[e][1] = r0.w;
    w[e][2] = r1.y;
    w[e][3] = r1.w;
  }
  const uint32_t kb_sweep = uload(a.parts, 0u).kb;
  lds_barrier();
  for (uint32_t s0 = 0; s0 < a.n_sweeps; s0 += a.per_phase) {
    const uint32_t ns = min(a.per_phase, a.n_sweeps - s0);
    res_keystream(a, 0u, s0, ns, chain, ks);
    lds_barrier();
    for (uint32_t ss = 0; ss < ns; ++ss) {
      const uint8_t *const kss = ks + ss * kb_sweep * 64u;
      for (uint32_t j = 0; j < wo.z; ++j) lds_barrier();
      static_for<NE>([&](auto e_c) {
        constexpr int e = decltype(e_c)::value;
        if ((uint32_t)e < wo.y) {
          if constexpr (NE > 4) {
            // unpacked here: kept unpacked, the entries would not fit the registers
            asm volatile("" : "+v"(pos[e][0]), "+v"(pos[e][1]), "+v"(site[e]));
          }
          const int32_t d0 = st[pos[e][0] & 0xffffu], d1 = st[pos[e][0] >> 16];
          const int32_t d2 = st[pos[e][1] & 0xffffu], d3 = st[pos[e][1] >> 16];
          float acc = res_add(0.0f, w[e][0], d0);
          acc = res_add(acc, w[e][1], d1);
          acc = res_add(acc, w[e][2], d2);
          acc = res_add(acc, w[e][3], d3);
          res_decide(st, kss, site[e], bias[e], acc);
          for (uint32_t j = 0; j < nbar[e]; ++j) lds_barrier();
        }
      });
    }
  }
  res_store_bits(a, chain, [&](uint32_t p) { return st[p] == 0; });
}

// Streaming kernel: any slot counts; the entries' data come from the caches for
// every half-sweep, one entry ahead: they do not depend on the state, so the
// loads are in flight across the barriers and the keystream.  With one chain per CU there
// are four waves per SIMD, each of which issues an instruction every four
// clocks at best, so the instructions per entry, scalar ones included, set
// the time: every entry issues the same loads from one address (no branches,
// no clamping: pairs past its last belong to the data that follow), and the
// ring of entries needs no index arithmetic.
template <int PF>
struct ResFrag {
  uint2 sb;
  uint4 v[PF];
};

template <int PF>
__device__ __forceinline__ ResFrag<PF> res_fetch(const ResArgs &a, uint32_t off, uint32_t lane) {
  ResFrag<PF> f;
  const uint8_t *const d = a.data + (lane * 16u + off);
  f.sb = *reinterpret_cast<const uint2 *>(a.data + (lane * 8u + off));
#pragma unroll
  for (int q = 0; q < PF; ++q) f.v[q] = *reinterpret_cast<const uint4 *>(d + RES_SITES + q * RES_PAIRS);
  return f;
}

// every load into f has landed (and the compiler knows it)
template <int PF>
__device__ __forceinline__ void res_landed(ResFrag<PF> &f) {
  asm volatile("" : "+v"(f.sb.x), "+v"(f.sb.y));
#pragma unroll
  for (int q = 0; q < PF; ++q)
    asm volatile("" : "+v"(f.v[q].x), "+v"(f.v[q].y), "+v"(f.v[q].z), "+v"(f.v[q].w));
}

template <int NG>
__device__ __forceinline__ float res_sum(const uint4 *v, const int8_t *st, float acc) {
  int32_t d[2 * NG];
#pragma unroll
  for (int q = 0; q < NG; ++q) {
    d[2 * q] = st[v[q].x];
    d[2 * q + 1] = st[v[q].z];
  }
#pragma unroll
  for (int q = 0; q < NG; ++q) {
    acc = res_add(acc, v[q].y, d[2 * q]);
    acc = res_add(acc, v[q].w, d[2 * q + 1]);
  }
  return acc;
}

template <int PF>
__global__ __launch_bounds__(1024) void resident_stream_kernel(ResArgs a) {
  extern __shared__ __align__(16) uint8_t rlds[];
  int8_t *const st = reinterpret_cast<int8_t *>(rlds);
  uint8_t *const ks = rlds + res_state_bytes(a.n_total);
  const uint32_t lane = threadIdx.x & 63u, n_waves = blockDim.x >> 6;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t chain = blockIdx.x;
  res_load_state(a, chain, [&](uint32_t p, uint32_t up) { st[p] = up ? 0 : -128; });

  // f: the records to sum, e0 their entry, e1 the entry after it
  uint4 e0 = uload(a.ents, uload(a.woff, wave).w);
  uint4 e1 = uload(a.ents, e0.z);
  ResFrag<PF> f = res_fetch<PF>(a, e0.x, lane);
  float acc = 0.0f;  // the sum of the slice's entries so far
  // sums entry f, and decides its sites with their slice's last entry, while
  // the next one, returned, is fetched
  auto step = [&](ResFrag<PF> &f, const uint8_t *kss) {
    res_landed(f);
    const uint32_t meta = e0.y, ng = meta & 15u;
    ResFrag<PF> n = res_fetch<PF>(a, e1.x, lane);
    e0 = e1;
    e1 = uload(a.ents, e1.z);
    if (ng == (uint32_t)PF) {
      acc = res_sum<PF>(f.v, st, acc);
    } else {
      static_for<PF - 1>([&](auto g_c) {
        constexpr int g = decltype(g_c)::value + 1;
        if (ng == (uint32_t)g) acc = res_sum<g>(f.v, st, acc);
      });
    }
    if (meta & 16u) {
      res_decide(st, kss, f.sb.x, bitsf(f.sb.y), acc);
      acc = 0.0f;
      for (uint32_t j = 0; j < meta >> 5; ++j) lds_barrier();
    }
    return n;
  };
  lds_barrier();
  for (uint32_t s0 = 0; s0 < a.n_sweeps; s0 += a.per_phase) {
    const uint32_t ns = min(a.per_phase, a.n_sweeps - s0);
    for (uint32_t part = 0; part < a.n_parts; ++part) {
      res_keystream(a, part, s0, ns, chain, ks);
      lds_barrier();
      const uint4 wo = uload(a.woff, part * n_waves + wave);
      const uint32_t kb_part = uload(a.parts, part).kb;
      for (uint32_t ss = 0; ss < ns; ++ss) {
        const uint8_t *const kss = ks + ss * kb_part * 64u;
        for (uint32_t j = 0; j < wo.z; ++j) lds_barrier();
        uint32_t k = 0;
        for (; k + 2u <= wo.y; k += 2u) {  // (two fragments in turn: no copies)
          ResFrag<PF> n = step(f, kss);
          f = step(n, kss);
        }
        if (k < wo.y) f = step(f, kss);
      }
    }
  }
  res_store_bits(a, chain, [&](uint32_t p) { return st[p] == 0; });
}

// The chains' new spins (64 positions per word) back into the state words
// (64 chains per word): a wave takes 64 chains x 64 positions, lane = chain.
__global__ __launch_bounds__(256) void resident_commit_kernel(const uint64_t *__restrict__ bits,
                                                              uint32_t n_words, uint32_t C,
                                                              uint32_t n_total, uint32_t n_tasks,
                                                              uint64_t *__restrict__ words) {
  const uint32_t task = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (task >= n_tasks) return;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t g = task / n_words, k = task - g * n_words;
  const uint32_t c = g * 64u + lane;
  const uint64_t x = c < C ? bits[(size_t)c * n_words + k] : 0ull;
  const uint32_t xl = (uint32_t)x, xh = (uint32_t)(x >> 32);
  uint32_t lo = 0u, hi = 0u;
  static_for<64>([&](auto j_c) {
    constexpr int j = decltype(j_c)::value;
    const uint64_t m = __builtin_amdgcn_ballot_w64(((j < 32 ? xl : xh) >> (j & 31)) & 1u);
    lo = writelane<j>(lo, (uint32_t)m);
    hi = writelane<j>(hi, (uint32_t)(m >> 32));
  });
  const uint32_t pos = k * 64u + lane;
  if (pos < n_total) words[(size_t)g * n_total + pos] = ((uint64_t)hi << 32) | lo;
}

// The entries' data: one thread per (slice, lane).
struct ResSlice {
  uint32_t first, last;  // byte offsets of the first entry's pairs and of the last entry's
  uint32_t ng, pf;       // slot pairs, pairs per entry
};
__global__ void resident_table_kernel(const ResSlice *__restrict__ slices,
                                      const uint2 *__restrict__ rows,
                                      const uint32_t *__restrict__ row_off,
                                      const uint2 *__restrict__ slots,
                                      const float *__restrict__ bias_w, uint32_t n,
                                      uint8_t *__restrict__ data) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const uint2 sr = rows[t];  // {site record, free position | RES_NONE}
  const ResSlice sl = slices[t >> 6];
  const uint32_t lane = t & 63u;
  const bool live = sr.y != RES_NONE;
  const uint32_t s0 = live ? row_off[sr.y] : 0u;
  const uint32_t deg = live ? row_off[sr.y + 1] - s0 : 0u;
  // the pairs of all entries but the last follow each other; the last entry's
  // follow the site records
  const uint32_t head = sl.ng > sl.pf ? (sl.ng - 1u) / sl.pf * sl.pf : 0u;
  for (uint32_t q = 0; q < sl.ng; ++q) {
    const uint2 u = 2u * q < deg ? slots[s0 + 2u * q] : make_uint2(0u, 0u);
    const uint2 v = 2u * q + 1u < deg ? slots[s0 + 2u * q + 1u] : make_uint2(0u, 0u);
    uint8_t *o = data + (q < head ? sl.first + q * RES_PAIRS : sl.last + (q - head) * RES_PAIRS);
    reinterpret_cast<uint4 *>(o)[lane] = make_uint4(u.x, u.y, v.x, v.y);
  }
  reinterpret_cast<uint2 *>(data + sl.last - RES_SITES)[lane] =
      make_uint2(sr.x, live ? fbits(bias_w[sr.y]) : 0u);
}

// ---------------------------------------------------------------------------
static const void *stream_kernel(uint32_t pf) {
  switch (pf) {
    case 2: return reinterpret_cast<const void *>(&resident_stream_kernel<2>);
    case 3: return reinterpret_cast<const void *>(&resident_stream_kernel<3>);
    case 4: return reinterpret_cast<const void *>(&resident_stream_kernel<4>);
    case 5: return reinterpret_cast<const void *>(&resident_stream_kernel<5>);
    case 6: return reinterpret_cast<const void *>(&resident_stream_kernel<6>);
    case 7: return reinterpret_cast<const void *>(&resident_stream_kernel<7>);
    default: return reinterpret_cast<const void *>(&resident_stream_kernel<8>);
  }
}
static const void *reg_kernel(uint32_t entries) {
  return entries <= 2u   ? reinterpret_cast<const void *>(&resident_reg_kernel<2>)
         : entries <= 4u ? reinterpret_cast<const void *>(&resident_reg_kernel<4>)
                         : reinterpret_cast<const void *>(&resident_reg_kernel<RES_MAX_ENT>);
}

// Builds the resident tables of a program when its chains can run resident:
// the state and one phase's keystream fit LDS.  row_off (host) and d_row_off /
// d_slots / d_bias (device) describe the free positions' slots.  The upload
// reads keep and the launch the arrays until the stream is synchronised.
int resident_tables(thrml_prog *p, const std::vector<uint32_t> &row_off, const uint32_t *d_row_off,
                    const uint2 *d_slots, const float *d_bias, std::vector<uint8_t> &keep) {
  if (p->stage_max != 0 || p->n_total > RES_MAX_NODES) return THRML_OK;
  uint64_t n_max = 0;
  for (uint32_t b = 0; b < p->n_free; ++b) n_max = std::max(n_max, p->blk_off[b + 1] - p->blk_off[b]);
  const uint32_t T = (uint32_t)std::min<uint64_t>(1024u, (n_max + 63u) / 64u * 64u);
  const uint32_t n_waves = T / 64u;
  // pieces and parts: each part takes at most T keystream blocks
  std::vector<ResPiece> pieces;
  std::vector<ResPart> parts;
  ResPart cur{0u, 0u, 0u};
  uint32_t n_slices = 0;
  for (uint32_t b = 0; b < p->n_free; ++b) {
    const uint32_t n_b = (uint32_t)(p->blk_off[b + 1] - p->blk_off[b]);
    for (uint32_t s = 0; s < n_b;) {
      uint32_t kb = (n_b - s + 15u) / 16u;
      if (kb > T - cur.kb) kb = (T - cur.kb) & ~3u;  // whole slices until the block's end
      if (kb == 0u) {
        cur.piece1 = (uint32_t)pieces.size();
        parts.push_back(cur);
        cur = ResPart{(uint32_t)pieces.size(), 0u, 0u};
        continue;
      }
      const uint32_t n = std::min(n_b - s, kb * 16u);
      pieces.push_back(ResPiece{b, s, n, cur.kb, (uint32_t)p->blk_off[b] + s, n_slices});
      n_slices += (n + 63u) / 64u;
      cur.kb += kb;
      s += n;
    }
  }
  cur.piece1 = (uint32_t)pieces.size();
  parts.push_back(cur);
  // sites of each piece by slot count, most first; a padding site writes the
  // spare byte after the state
  std::vector<uint2> rows((size_t)n_slices * 64u, make_uint2((uint32_t)p->n_total, RES_NONE));
  std::vector<ResSlice> slices(n_slices);
  uint32_t maxdeg = 0;
  std::vector<uint32_t> start;
  for (const ResPiece &pc : pieces) {
    const uint32_t *ro = row_off.data() + pc.row0;
    uint32_t md = 0;
    for (uint32_t i = 0; i < pc.n; ++i) md = std::max(md, ro[i + 1] - ro[i]);
    maxdeg = std::max(maxdeg, md);
    // start[d]: sites with more than d slots
    start.assign((size_t)md + 2, 0u);
    for (uint32_t i = 0; i < pc.n; ++i) ++start[ro[i + 1] - ro[i]];
    for (uint32_t d = md + 1, above = 0; d-- > 0;) {
      const uint32_t n = start[d];
      start[d] = above;
      above += n;
    }
    for (uint32_t i = 0; i < pc.n; ++i) {
      const uint32_t d = ro[i + 1] - ro[i], k = start[d]++;
      const uint32_t word = res_word(pc.kb0 + i / 16u, i % 16u) * 4u;
      rows[(size_t)pc.slice0 * 64u + k] = make_uint2((pc.row0 + i) | (word << 16), pc.row0 + i);
      if (k % 64u == 0u) slices[pc.slice0 + k / 64u].ng = (d + 1u) / 2u;
    }
  }
  if (p->kind == K_LATTICE && (parts.size() != 1 || maxdeg > 4u)) return THRML_OK;
  // Pairs per entry: an entry costs about as much as 5 pairs besides its
  // loads (it issues pf of them, used or not)
  uint32_t pf = 2u;
  uint64_t best = ~0ull;
  for (uint32_t c = 2u; c <= RES_MAX_PF; ++c) {
    uint64_t cost = 0;
    for (const ResSlice &sl : slices) cost += (uint64_t)std::max(1u, (sl.ng + c - 1u) / c) * (c + 5u);
    if (cost < best) {
      best = cost;
      pf = c;
    }
  }
  uint64_t at = RES_SITES;  // (an entry's data start 512 bytes before its pairs)
  for (ResSlice &sl : slices) {
    sl.pf = pf;
    const uint32_t head = sl.ng > pf ? (sl.ng - 1u) / pf * pf : 0u;
    sl.first = (uint32_t)at;
    at += (uint64_t)head * RES_PAIRS + RES_SITES;
    sl.last = (uint32_t)at;
    at += (uint64_t)(sl.ng - head) * RES_PAIRS;
  }
  at += (uint64_t)RES_MAX_PF * RES_PAIRS;  // the last entry's unused loads
  // records mostly padding (a few hubs among sparse sites): the per-block kernels
  if (at > 40ull * row_off[p->blk_off[p->n_free]] + 1024ull * n_slices + 65536u || at >= (1ull << 31))
    return THRML_OK;
  // each wave's entries: slices wave, wave + n_waves, ... of every piece, with
  // the barriers (one per piece) that follow each
  std::vector<uint4> ents, woff;
  std::vector<uint32_t> first(n_waves, RES_NONE), prev(n_waves, RES_NONE);
  uint32_t max_ent = 0;
  for (const ResPart &pt : parts)
    for (uint32_t w = 0; w < n_waves; ++w) {
      uint4 wo = make_uint4((uint32_t)ents.size(), 0u, 0u, 0u);
      for (uint32_t q = pt.piece0; q < pt.piece1; ++q) {
        const ResPiece &pc = pieces[q];
        for (uint32_t k = w; k * 64u < pc.n; k += n_waves) {
          const ResSlice &sl = slices[pc.slice0 + k];
          uint32_t g = 0;
          do {
            const uint32_t ng = std::min(sl.ng - g, pf);
            const bool last = g + ng == sl.ng;
            const uint32_t id = (uint32_t)ents.size();
            if (prev[w] == RES_NONE) first[w] = id;
            else ents[prev[w]].z = id;
            prev[w] = id;
            ents.push_back(make_uint4((last ? sl.last : sl.first + g * RES_PAIRS) - RES_SITES,
                                      ent_meta(ng, last, 0u), 0u, 0u));
            g += ng;
            ++wo.y;
          } while (g < sl.ng);
        }
        if (wo.y) ents.back().y += ent_meta(0u, false, 1u);
        else ++wo.z;
      }
      max_ent = std::max(max_ent, wo.y);
      woff.push_back(wo);
    }
  for (uint32_t w = 0; w < n_waves; ++w) {
    if (prev[w] != RES_NONE) ents[prev[w]].z = first[w];
    for (size_t q = 0; q < parts.size(); ++q)  // (a wave without entries fetches entry 0 and never uses it)
      woff[q * n_waves + w].w = first[w] == RES_NONE ? 0u : first[w];
  }
  // the register kernel: its entries, or 0 when the program does not fit it
  const uint32_t ent = parts.size() == 1 && maxdeg <= 4u && max_ent <= RES_MAX_ENT ? max_ent : 0u;
  // (a lattice that does not fit it always goes faster block by block)
  if (p->kind == K_LATTICE && !ent) return THRML_OK;
  // one buffer and one upload: the tables, then the data that the kernel below writes
  size_t off[6], end = 0;
  const struct { const void *p; size_t n; } tab[6] = {
      {pieces.data(), pieces.size() * sizeof(ResPiece)}, {parts.data(), parts.size() * sizeof(ResPart)},
      {ents.data(), ents.size() * sizeof(uint4)},        {woff.data(), woff.size() * sizeof(uint4)},
      {slices.data(), slices.size() * sizeof(ResSlice)}, {rows.data(), rows.size() * sizeof(uint2)}};
  for (int k = 0; k < 6; ++k) {
    off[k] = end;
    end += (tab[k].n + 255u) / 256u * 256u;
  }
  keep.resize(end);
  for (int k = 0; k < 6; ++k) std::memcpy(keep.data() + off[k], tab[k].p, tab[k].n);
  if (int rc = p->r_tab.alloc(end + at, &p->ctx->pool)) return rc;
  uint8_t *const d = p->r_tab.as<uint8_t>();
  THRML_HIP(hipMemcpyAsync(d, keep.data(), end, hipMemcpyHostToDevice, p->ctx->stream));
  const uint32_t n = n_slices * 64u;
  hipLaunchKernelGGL(resident_table_kernel, dim3((n + 255u) / 256u), dim3(256), 0, p->ctx->stream,
                     reinterpret_cast<const ResSlice *>(d + off[4]),
                     reinterpret_cast<const uint2 *>(d + off[5]), d_row_off, d_slots, d_bias, n, d + end);
  THRML_HIP(hipGetLastError());
  THRML_HIP(hipFuncSetAttribute(ent ? reg_kernel(ent) : stream_kernel(pf),
                                hipFuncAttributeMaxDynamicSharedMemorySize, RES_LDS));
  for (int k = 0; k < 4; ++k) p->r_off[k] = off[k];
  p->r_off[4] = end;
  p->res_T = T;
  p->res_pf = pf;
  p->res_parts = (uint32_t)parts.size();
  p->res_kb = parts[0].kb;
  p->res_ent = ent;
  p->res_deg = (double)row_off[p->blk_off[p->n_free]] / (double)p->blk_off[p->n_free];
  p->res_work = ent ? n_slices * (ent <= 4u ? 0.0145 : 0.025) : (double)best * 0.0068;
  p->device_bytes += p->r_tab.bytes;
  return THRML_OK;
}

// LDS of a workgroup: the state, and a keystream block per thread.
static size_t res_lds(const thrml_prog *p) { return ((p->n_total + 16u) & ~15ull) + (size_t)p->res_T * 64u; }

// Whether n_seg segments (runs of sweeps between observations) of n_sweeps
// sweeps in all go faster resident than block by block; fused: the lattice
// kernel would count the observations itself.  Both sides are fits, in us, to
// run times on MI355X (tori of side 10 .. 256, Erdos-Renyi graphs of 200 ..
// 60000 nodes and mean degree 4 .. 12, double grids, 64 .. 2048 free sites among
// 1000 .. 60000 clamped ones; 1 .. 1024 chains).
// Resident, per sweep: 0.35 per block and 0.0068 per (pair + 5) of the entries
// (0.0145 or 0.025 per slice from registers), for every turn of the chains over
// the CUs.  Per segment: 6.5 for its two launches (4 for one chain's single
// one) and 0.38 (0.19) for each step of the workgroup over all positions, on the
// way into and out of LDS; where a launch for the observation comes on top, 3 and
// 0.2 per 1000 words of the state.  Block by block: a launch takes 3.2 on a lattice
// (between 2.4 and 4.1, by the host), 4.0 (7.6 with 16-site runs) and more with
// the degree otherwise, and grows with the sites times the chain groups.
//   us per sweep, + per segment beyond an observation   resident    block by block
//   64^2, C = 1                                         1.6 + 7.8   4.9-8.3
//   64^2, C = 512                                       3.3 + 21    7.6
//   96^2, C = 256                                       4.3 + 18    6.5-9.3
//   128^2, C = 64                                       9.5         5.4
//   E-R 20K deg 6, C = 200                              21 + 15     52
//   E-R 60K deg 6, C = 200                              56 + 35     80
//   E-R 60K deg 6, C = 512                              113 + 66    101
//   grid 2 x 40^2, C = 1                                4.1         8.0
//   64 sites + 1000 clamped, C = 32                     0.43 + 13   5.0
//   64 sites + 60000 clamped, C = 32                    0.43 + 353  4.9
//   2048 sites + 60000 clamped, C = 256                 1.7 + 37    5.7
bool resident_pays(const thrml_prog *p, const thrml_state *st, uint64_t n_sweeps, uint64_t n_seg,
                   bool fused) {
  if (!p->res_T) return false;
  const double C = st->C, G = st->G;
  // workgroups of at most 512 threads share a CU, as many as its LDS holds
  const double per_cu = p->res_T > 512u ? 1.0 : (double)std::min<size_t>(2048u / p->res_T, (size_t)RES_LDS / res_lds(p));
  const double turns = std::ceil(C / (p->ctx->cu_count * per_cu));
  const double rounds = per_cu > 1.0 ? std::max(1.0, C / p->ctx->cu_count) : turns;
  const double res = 0.35 * p->n_free + rounds * p->res_work;
  const double steps = std::ceil((double)p->n_total / p->res_T);
  const double seg = (C > 1.0 ? 6.5 + 0.38 * turns * steps : 4.0 + 0.19 * steps) +
                     (fused ? 3.0 + 0.2e-3 * (double)p->n_total * G : 0.0);
  double blk = 0.0;
  for (uint32_t b = 0; b < p->n_free; ++b) {
    const double n = (double)(p->blk_off[b + 1] - p->blk_off[b]);
    if (p->kind == K_LATTICE) {
      blk += std::max(3.2, 1.0 + n * G * 0.05e-3);
    } else {
      const double deg = p->res_deg;
      const bool run16 = C > 32.0 && std::ceil(n / 16.0) * G >= 4096.0;  // as launch_csr_half
      blk += 0.1 * deg + (run16 ? 7.6 + n * G * 0.11e-3 : 4.0 + n * (C <= 32.0 ? 0.06e-3 : (G - 0.5) * 0.22e-3));
    }
  }
  return res * (double)n_sweeps + seg * (double)n_seg < 0.95 * blk * (double)n_sweeps;
}

int launch_resident(thrml_prog *p, thrml_state *st, const uint32_t *d_keys, uint32_t n_sweeps) {
  ResArgs a{};
  a.words = st->words.as<uint64_t>();
  a.bits = st->bits.as<uint64_t>();
  a.keys = d_keys;
  const uint8_t *tab = p->r_tab.as<uint8_t>();
  a.pieces = reinterpret_cast<const ResPiece *>(tab + p->r_off[0]);
  a.parts = reinterpret_cast<const ResPart *>(tab + p->r_off[1]);
  a.ents = reinterpret_cast<const uint4 *>(tab + p->r_off[2]);
  a.woff = reinterpret_cast<const uint4 *>(tab + p->r_off[3]);
  a.data = tab + p->r_off[4];
  a.n_total = (uint32_t)p->n_total;
  a.n_words = (a.n_total + 63u) / 64u;
  a.n_sweeps = n_sweeps;
  a.n_blocks = p->n_free;
  a.C_pad = st->G * 64u;
  a.n_parts = p->res_parts;
  a.div_kb = make_fastdiv(p->res_kb);
  a.per_phase = p->res_parts == 1u ? p->res_T / p->res_kb : 1u;
  hipStream_t s = p->ctx->stream;
  hipEvent_t t0 = nullptr;
  if (p->ctx->time_begin(0, &t0)) return THRML_EHIP;
  void *args[] = {&a};
  THRML_HIP(hipLaunchKernel(p->res_ent ? reg_kernel(p->res_ent) : stream_kernel(p->res_pf), dim3(st->C),
                            dim3(p->res_T), args, res_lds(p), s));
  if (st->C > 1u) {
    const uint32_t n_tasks = a.n_words * st->G;
    hipLaunchKernelGGL(resident_commit_kernel, dim3((n_tasks + 3u) / 4u), dim3(256), 0, s, a.bits,
                       a.n_words, st->C, a.n_total, n_tasks, st->words.as<uint64_t>());
    THRML_HIP(hipGetLastError());
  }
  return p->ctx->time_end(0, t0, (uint64_t)n_sweeps * p->n_free);
}

}  // namespace thrml

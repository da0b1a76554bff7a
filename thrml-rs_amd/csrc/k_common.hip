// k_common.hip -- key schedule, state import/export, moment accumulation,
// hinton initialisation and the kernel-level exports.
#include <cstring>

#include "dev_util.hpp"
#include "internal.hpp"

namespace thrml {

static inline uint32_t cdiv(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// ---------------------------------------------------------------------------
// Key schedule.  Chain c's key is RngKey::split(root, C)[c]; below it the
// reference's tree of splits (crates/thrml-samplers/src/sampling.rs) gives
// the key of every sweep:
//   run_blocks(key, n_iters)           sweep s: split(n_iters)[s]       (:93)
//   sample_with_observation(key, ...)  (wk, sk) = key.split_two()      (:189)
//     warm-up sweep w:                 split(wk, n_warmup)[w]
//     sample i (of n_samples-1), step t: split(split(sk, n_samples-1)[i],
//                                          steps_per_sample)[t]          (:222,:264)
// and sample_blocks splits a sweep key into one key per block (:37).  The
// stored value is the seed_from_u64 expansion of the block key: the ChaCha8
// key of the per-site uniform stream, stored expanded (key_expand).  Output
// layout keys[s - s0][b][c_pad][KEY_WORDS].
__device__ uint64_t sweep_key(const KeyPlan &kp, uint64_t chain_key, uint64_t s) {
  if (kp.mode == 0) return split_at(chain_key, kp.n_iters, s);
  if (s < kp.n_warmup) return split_at(split_at(chain_key, 2, 0), kp.n_warmup, s);
  s -= kp.n_warmup;
  const uint64_t i = s / kp.steps, t = s - i * kp.steps;
  const uint64_t ks = split_at(split_at(chain_key, 2, 1), kp.n_samples - 1, i);
  return split_at(ks, kp.steps, t);
}

__global__ void key_schedule_kernel(KeyPlan kp, uint64_t s0, uint32_t n_sweeps,
                                    uint32_t *__restrict__ keys) {
  const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t total = (uint64_t)n_sweeps * kp.n_blocks * kp.C_pad;
  if (tid >= total) return;
  const uint32_t c = (uint32_t)(tid % kp.C_pad);
  const uint64_t rest = tid / kp.C_pad;
  const uint32_t b = (uint32_t)(rest % kp.n_blocks);
  const uint64_t s = s0 + rest / kp.n_blocks;
  uint4 *o = reinterpret_cast<uint4 *>(keys + tid * KEY_WORDS);
  uint32_t x[KEY_WORDS];
#pragma unroll
  for (int i = 0; i < KEY_WORDS; ++i) x[i] = 0u;
  if (c < kp.C) {
    const uint64_t k = split_at(sweep_key(kp, split_at(kp.root, kp.C, c), s), kp.n_blocks, b);
    key_expand(seed_from_u64(k).k, x);
  }
#pragma unroll
  for (int q = 0; q < KEY_WORDS / 4; ++q) o[q] = make_uint4(x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]);
}

int launch_key_schedule(thrml_ctx *ctx, const KeyPlan &kp, uint64_t s0, uint32_t n_sweeps,
                        uint32_t *d_keys) {
  if (n_sweeps == 0) return THRML_OK;
  const uint64_t total = (uint64_t)n_sweeps * kp.n_blocks * kp.C_pad;
  hipLaunchKernelGGL(key_schedule_kernel, dim3(cdiv(total, 256)), dim3(256), 0, ctx->stream, kp,
                     s0, n_sweeps, d_keys);
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

// ---------------------------------------------------------------------------
// State import / export: positions p0 .. p0 + n - 1 of every chain, the caller's
// side one row of `stride` values per chain (u8 or f32) starting at column
// col0.  Lane = position (IO_PER consecutive ones for u8), so that a row's
// values and the state words both move in whole cache lines; a lane's 64
// chain bits of a word are its own, and no bits cross lanes.
struct StateIo {
  uint64_t *words;        // first word of position p0, group 0
  uint64_t plane_stride;
  uint32_t C, n, n_chunks;
  uint64_t stride, col0;
};
constexpr uint32_t IO_PER = 4;     // positions per lane, u8 rows
constexpr uint32_t IO_CHAINS = 16; // chains per wave, export
typedef uint32_t u32_a1 __attribute__((aligned(1)));

// The import is checked before (import_check_kernel): *bad is IMPORT_OK or
// nothing is written.  A wave takes one chain group.
template <class V>
__global__ __launch_bounds__(256) void pack_kernel(const V *__restrict__ src, StateIo a, uint32_t n_tasks,
                                                   const uint32_t *__restrict__ bad) {
  constexpr uint32_t PER = sizeof(V) == 1 ? IO_PER : 1u;
  const uint32_t task = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (task >= n_tasks || *bad != IMPORT_OK) return;
  const uint32_t g = task / a.n_chunks, chunk = task - g * a.n_chunks;
  const uint32_t i = (chunk * 64u + (threadIdx.x & 63u)) * PER;
  if (i >= a.n) return;
  const uint32_t live = min(a.C - g * 64u, 64u);
  const V *row = src + (size_t)g * 64u * a.stride + a.col0 + i;
  uint32_t lo[PER] = {}, hi[PER] = {};
  const bool whole = i + PER <= a.n;
#pragma unroll 16
  for (uint32_t c = 0; c < live; ++c, row += a.stride) {
    uint32_t v[PER];
    if constexpr (sizeof(V) == 1) {
      uint32_t x = 0;
      if (whole) x = *reinterpret_cast<const u32_a1 *>(row);
      else
        for (uint32_t k = 0; i + k < a.n; ++k) x |= (uint32_t)row[k] << (8u * k);
#pragma unroll
      for (uint32_t k = 0; k < PER; ++k) v[k] = (x >> (8u * k)) & 1u;
    } else {
      v[0] = *row == 1.0f ? 1u : 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < PER; ++k) {
      if (c < 32u) lo[k] |= v[k] << c;
      else hi[k] |= v[k] << (c - 32u);
    }
  }
  uint64_t *w = a.words + (size_t)g * a.plane_stride + i;
#pragma unroll
  for (uint32_t k = 0; k < PER; ++k)
    if (i + k < a.n) w[k] = ((uint64_t)hi[k] << 32) | lo[k];
}

// A wave takes IO_CHAINS chains of one group.
template <class V>
__global__ __launch_bounds__(256) void unpack_kernel(V *__restrict__ dst, StateIo a, uint32_t n_tasks) {
  constexpr uint32_t PER = sizeof(V) == 1 ? IO_PER : 1u;
  const uint32_t task = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (task >= n_tasks) return;
  const uint32_t q = task / a.n_chunks, chunk = task - q * a.n_chunks;
  const uint32_t c0 = q * IO_CHAINS, g = c0 >> 6;
  const uint32_t i = (chunk * 64u + (threadIdx.x & 63u)) * PER;
  if (i >= a.n || c0 >= a.C) return;
  const uint64_t *w = a.words + (size_t)g * a.plane_stride + i;
  uint32_t b[PER];  // this wave's chains' bits of the lane's positions
#pragma unroll
  for (uint32_t k = 0; k < PER; ++k) b[k] = i + k < a.n ? (uint32_t)(w[k] >> (c0 & 63u)) : 0u;
  V *row = dst + (size_t)c0 * a.stride + a.col0 + i;
  const bool whole = i + PER <= a.n;
#pragma unroll
  for (uint32_t c = 0; c < IO_CHAINS; ++c, row += a.stride) {
    if (c0 + c >= a.C) break;
    if constexpr (sizeof(V) == 1) {
      uint32_t x = 0;
#pragma unroll
      for (uint32_t k = 0; k < PER; ++k) x |= ((b[k] >> c) & 1u) << (8u * k);
      if (whole) *reinterpret_cast<u32_a1 *>(row) = x;
      else
        for (uint32_t k = 0; i + k < a.n; ++k) row[k] = (uint8_t)(x >> (8u * k));
    } else {
      *row = (b[0] >> c) & 1u ? 1.0f : 0.0f;
    }
  }
}

// Export of few positions: a wave takes a chain group, lane = chain, so that all
// lanes have a row (above, two positions leave one lane of 64).  Bound by its
// stores, a row apart per lane, so that it loses from some width on.  us per
// launch, above -> here:
//   u8   2 positions, 1,024 chains 5.6 -> 3.6;  3, 600,000 38 -> 3.8
//        16, 600,000 22 -> 14;  24, 600,000 22 -> 27
//   f32  2, 600,000 15 -> 3.8;  8, 600,000 17 -> 14;  12, 600,000 16 -> 28
constexpr uint32_t IO_NARROW_U8 = 16, IO_NARROW_F32 = 8;
template <class V>
__global__ __launch_bounds__(256) void unpack_narrow_kernel(V *__restrict__ dst, StateIo a, uint32_t G) {
  const uint32_t g = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t c = g * 64u + (threadIdx.x & 63u);
  if (g >= G || c >= a.C) return;
  const uint64_t *w = a.words + (size_t)g * a.plane_stride;
  V *row = dst + (size_t)c * a.stride + a.col0;
  for (uint32_t i = 0; i < a.n; ++i) row[i] = (V)((w[i] >> (c & 63u)) & 1ull);
}

// Import check before any write: *bad becomes the smallest column that holds
// something else than a state value (0..q-1 as u8, or the floats 0.0..q-1.0),
// among columns col0 .. col0 + n - 1 of the rows of `stride` values.
__global__ __launch_bounds__(256) void import_check_kernel(const void *__restrict__ src, int dtype,
                                                           uint32_t C, uint32_t n, uint64_t stride,
                                                           uint64_t col0, uint32_t q, uint32_t n_chunks,
                                                           uint32_t *__restrict__ bad) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t c = (uint32_t)(t / n_chunks), k = (uint32_t)(t - (uint64_t)c * n_chunks);
  if (c >= C) return;
  const uint32_t i0 = k * 16u, i1 = min(i0 + 16u, n);
  const size_t at = (size_t)c * stride + col0;
  if (dtype == THRML_DTYPE_U8) {
    const uint8_t *p = reinterpret_cast<const uint8_t *>(src) + at;
    if (i0 + 16u <= n && q <= 128u) {
      // a byte is 128 or more, or its low seven bits plus 128 - q carry into bit 7
      uint32_t any = 0u;
#pragma unroll
      for (uint32_t j = 0; j < 4u; ++j) {
        const uint32_t x = *reinterpret_cast<const u32_a1 *>(p + i0 + 4u * j);
        any |= (x | ((x & 0x7f7f7f7fu) + (128u - q) * 0x01010101u)) & 0x80808080u;
      }
      if (any == 0u) return;
    }
    for (uint32_t i = i0; i < i1; ++i)
      if (p[i] >= q) {
        atomicMin(bad, (uint32_t)(col0 + i));
        return;
      }
  } else {
    const float *p = reinterpret_cast<const float *>(src) + at;
    for (uint32_t i = i0; i < i1; ++i) {
      const float x = p[i];
      if (!(x >= 0.0f && x < (float)q && x == __builtin_floorf(x))) {
        atomicMin(bad, (uint32_t)(col0 + i));
        return;
      }
    }
  }
}

__global__ void import_reset_kernel(uint32_t *bad) { *bad = IMPORT_OK; }

int launch_import_reset(thrml_ctx *ctx, uint32_t *d_bad) {
  hipLaunchKernelGGL(import_reset_kernel, dim3(1), dim3(1), 0, ctx->stream, d_bad);
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

int launch_import_check(thrml_ctx *ctx, const void *d_src, int dtype, uint32_t C, uint32_t n,
                        uint64_t stride, uint64_t col0, uint32_t q, uint32_t *d_bad) {
  const uint32_t n_chunks = cdiv(n, 16);
  const uint64_t nb = ((uint64_t)C * n_chunks + 255) / 256;
  if (nb > 0x7fffffffull) return fail(THRML_EUNSUPPORTED, "block too large to import");
  hipLaunchKernelGGL(import_check_kernel, dim3((uint32_t)nb), dim3(256), 0, ctx->stream, d_src,
                     dtype, C, n, stride, col0, q, n_chunks, d_bad);
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

static StateIo state_io_args(thrml_state *st, uint64_t p0, uint32_t n, uint64_t stride, uint64_t col0,
                             int dtype) {
  const uint32_t per = 64u * (dtype == THRML_DTYPE_U8 ? IO_PER : 1u);
  return StateIo{st->words.as<uint64_t>() + p0, st->prog->n_total, st->C, n, cdiv(n, per), stride, col0};
}

int launch_pack(thrml_state *st, uint64_t p0, uint32_t n, const void *d_src, int dtype,
                uint64_t stride, uint64_t col0, const uint32_t *d_bad) {
  hipStream_t s = st->prog->ctx->stream;
  const StateIo a = state_io_args(st, p0, n, stride, col0, dtype);
  const uint64_t tasks = (uint64_t)a.n_chunks * st->G;
  if (tasks > 0x7fffffffull) return fail(THRML_EUNSUPPORTED, "block too large to import");
  if (dtype == THRML_DTYPE_U8)
    hipLaunchKernelGGL(pack_kernel<uint8_t>, dim3(cdiv(tasks, 4)), dim3(256), 0, s,
                       static_cast<const uint8_t *>(d_src), a, (uint32_t)tasks, d_bad);
  else
    hipLaunchKernelGGL(pack_kernel<float>, dim3(cdiv(tasks, 4)), dim3(256), 0, s,
                       static_cast<const float *>(d_src), a, (uint32_t)tasks, d_bad);
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

int launch_unpack(thrml_state *st, uint64_t p0, uint32_t n, void *d_dst, int dtype, uint64_t stride,
                  uint64_t col0) {
  hipStream_t s = st->prog->ctx->stream;
  const StateIo a = state_io_args(st, p0, n, stride, col0, dtype);
  const uint64_t tasks = (uint64_t)a.n_chunks * cdiv(st->C, IO_CHAINS);
  if (tasks > 0x7fffffffull) return fail(THRML_EUNSUPPORTED, "block too large to export");
  const dim3 grid(cdiv(tasks, 4)), narrow(cdiv(st->G, 4)), wg(256);
  if (dtype == THRML_DTYPE_U8) {
    uint8_t *dst = static_cast<uint8_t *>(d_dst);
    if (n <= IO_NARROW_U8) hipLaunchKernelGGL(unpack_narrow_kernel<uint8_t>, narrow, wg, 0, s, dst, a, st->G);
    else hipLaunchKernelGGL(unpack_kernel<uint8_t>, grid, wg, 0, s, dst, a, (uint32_t)tasks);
  } else {
    float *dst = static_cast<float *>(d_dst);
    if (n <= IO_NARROW_F32) hipLaunchKernelGGL(unpack_narrow_kernel<float>, narrow, wg, 0, s, dst, a, st->G);
    else hipLaunchKernelGGL(unpack_kernel<float>, grid, wg, 0, s, dst, a, (uint32_t)tasks);
  }
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

// ---------------------------------------------------------------------------
// Moment accumulation (MomentAccumulatorObserver::observe,
// crates/thrml-observers/src/moment.rs:157-237): per observation,
//   ones[k] += #chains with s = 1 at node k,
//   diff[k] += #chains with s_a != s_b for pair k,
// so that sum_c t = 2*ones - C*n_obs and sum_c t_a t_b = C*n_obs - 2*diff.
// Bound by the random reads of a pair's words.  A workgroup takes 256 >> lg
// items (nodes, then pairs), 1 << lg threads per item, thread `slice` of an item
// the chain groups slice, slice + (1 << lg), ..., summed through LDS: with few
// items a thread alone has too few of its loads in flight (5,120 nodes and
// their pairs, 4,096 chains: 19.1 us per observation with one thread per item,
// 5.0 us with 32), and above MOMENTS_FILL threads, 16 waves per compute unit,
// the items fill the chip by themselves.
constexpr uint32_t MOMENTS_MAX_LG = 5;
constexpr uint64_t MOMENTS_FILL = 1u << 18;

// W: uint64_t, or uint32_t where one chain group has at most 32 chains and the
// state keeps a copy of its words' low halves (half the bytes to gather: a
// million nodes and their 6 million pairs 57.9 -> 41.3 us).
template <class W>
__global__ __launch_bounds__(256) void moments_kernel(
    const W *__restrict__ words, uint64_t plane_stride, uint32_t G, uint32_t C,
    const uint32_t *__restrict__ npos, uint64_t n1, const uint32_t *__restrict__ ppos, uint64_t n2,
    uint32_t *__restrict__ ones, uint32_t *__restrict__ diff, uint32_t lg) {
  __shared__ uint32_t part[256];
  const uint32_t per = 256u >> lg;
  const uint32_t slice = threadIdx.x >> (8u - lg);
  const uint64_t i = (uint64_t)blockIdx.x * per + (threadIdx.x & (per - 1u));
  // (threads past the last item take the last and store nothing)
  const uint64_t k = i < n1 + n2 ? i : n1 + n2 - 1u;
  const bool node = k < n1;
  const uint32_t *at = node ? npos + k : ppos + 2u * (k - n1);
  const uint32_t pa = at[0], pb = at[node ? 0 : 1];
  const W two = node ? (W)0 : (W)~(W)0;  // a node's second word counts as 0
  uint32_t *cnt = node ? ones + k : diff + (k - n1);
  const uint32_t old = *cnt;
  uint32_t sum = 0u;
#pragma unroll 4
  for (uint32_t g = slice; g < G; g += 1u << lg) {
    const W *w = words + (size_t)g * plane_stride;
    const uint32_t rem = C - g * 64u;
    const uint64_t valid = rem < 64u ? (1ull << rem) - 1ull : ~0ull;
    sum += (uint32_t)__builtin_popcountll((uint64_t)(w[pa] ^ (w[pb] & two)) & valid);
  }
  if (lg != 0u) {
    part[threadIdx.x] = sum;
    __syncthreads();
    if (slice != 0u) return;
    for (uint32_t t = 1; t < 1u << lg; ++t) sum += part[t * per + threadIdx.x];
  }
  if (i < n1 + n2) *cnt = old + sum;
}

int launch_moments(thrml_state *st, const uint32_t *d_npos, uint64_t n1, const uint32_t *d_ppos,
                   uint64_t n2, uint32_t *d_ones, uint32_t *d_diff) {
  thrml_prog *p = st->prog;
  const uint64_t total = n1 + n2;
  if (total == 0) return THRML_OK;
  hipEvent_t t0 = nullptr;
  if (p->ctx->time_begin(1, &t0)) return THRML_EHIP;
  uint32_t lg = 0;
  while (lg < MOMENTS_MAX_LG && (2u << lg) <= st->G && (total << lg) < MOMENTS_FILL) ++lg;
  const dim3 grid(cdiv(total, 256u >> lg));
  if (st->low_live)
    hipLaunchKernelGGL(moments_kernel<uint32_t>, grid, dim3(256), 0, p->ctx->stream,
                       st->low.as<uint32_t>(), (uint64_t)p->n_total, st->G, st->C, d_npos, n1, d_ppos,
                       n2, d_ones, d_diff, lg);
  else
    hipLaunchKernelGGL(moments_kernel<uint64_t>, grid, dim3(256), 0, p->ctx->stream,
                       st->words.as<uint64_t>(), (uint64_t)p->n_total, st->G, st->C, d_npos, n1,
                       d_ppos, n2, d_ones, d_diff, lg);
  THRML_HIP(hipGetLastError());
  return p->ctx->time_end(1, t0);
}

// One observation of a general moment observer (moment.rs:153-231): thread
// r adds sum over chains of prod f(x) over row r's positions.  Spin words
// (64 chains per word): with f = 2s - 1 the product is -1 where an odd
// number of the row's spins are down, so the row's sum over a word is
// (chains) - 2 popcount(xor of the inverted words); with f = s it is the
// popcount of the words' AND.  Byte states: the product per chain in int64.
// 1 << lg lanes take a row: lane l of it the chain groups (spin words), or the
// runs of 4 consecutive chains (byte states, one load per position), l,
// l + (1 << lg), ...; then a sum over the row's lanes that the first adds to
// the row's total.  Bound by the dependent loads (row, positions, states): as
// many lanes as a row has units of work, so that a wave holds as many rows as
// it can, and two positions at a time.  131,072 rows of one byte-state
// node, 32 chains: 34.2 us with a wave per row, 7.1 us so.
// T: the byte states' element, or uint64_t for spin words.
template <class T>
__global__ __launch_bounds__(256) void observe_kernel(
    const T *__restrict__ state, uint64_t plane_stride,
    uint32_t G, uint32_t C, uint32_t Cp, const uint64_t *__restrict__ row_off,
    const uint32_t *__restrict__ pos, uint64_t n_rows, int transform, int64_t *__restrict__ acc,
    uint32_t lg) {
  const uint64_t row = ((uint64_t)blockIdx.x * 256u + threadIdx.x) >> lg;
  const uint32_t l = threadIdx.x & ((1u << lg) - 1u);
  const uint64_t r = row < n_rows ? row : n_rows - 1u;
  const uint64_t a = row_off[r], b = row_off[r + 1];
  int64_t sum = 0;
  if constexpr (sizeof(T) == 8) {
    for (uint32_t g = l; g < G; g += 1u << lg) {
      const uint32_t rem = C - g * 64u;
      const uint64_t valid = rem < 64u ? (1ull << rem) - 1ull : ~0ull;
      uint64_t m = transform ? 0ull : ~0ull;
      for (uint64_t k = a; k < b; k += 2) {
        // (a last position without a partner is read twice and counts once)
        const bool pair = k + 1 < b;
        const uint32_t p0 = pos[k], p1 = pos[pair ? k + 1 : k];
        const uint64_t w0 = state[(size_t)g * plane_stride + p0];
        const uint64_t w1 = state[(size_t)g * plane_stride + p1];
        if (transform) m ^= ~w0 ^ (pair ? ~w1 : 0ull);
        else m &= w0 & w1;
      }
      const int64_t n = __builtin_popcountll(valid);
      sum += transform ? n - 2 * (int64_t)__builtin_popcountll(m & valid)
                       : (int64_t)__builtin_popcountll(m & valid);
    }
  } else {
    // the observer's creation bounds every row's product (and the run its
    // sum over chains and observations) below 2^63
    struct alignas(4 * sizeof(T)) Four {
      T v[4];
    };
    for (uint32_t c = 4u * l; c < C; c += 4u << lg) {
      uint64_t prod[4] = {1, 1, 1, 1};  // (chains past C may hold anything)
      for (uint64_t k = a; k < b; k += 2) {
        const bool pair = k + 1 < b;
        const uint32_t p0 = pos[k], p1 = pos[pair ? k + 1 : k];
        // (Cp is a multiple of 4)
        const Four x0 = *reinterpret_cast<const Four *>(state + (size_t)p0 * Cp + c);
        const Four x1 = *reinterpret_cast<const Four *>(state + (size_t)p1 * Cp + c);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int32_t f0 = transform ? 2 * (int32_t)x0.v[u] - 1 : (int32_t)x0.v[u];
          const int32_t f1 = !pair ? 1 : transform ? 2 * (int32_t)x1.v[u] - 1 : (int32_t)x1.v[u];
          // (below 2^34: the factors are 16 bits and a sign)
          prod[u] *= (uint64_t)((int64_t)f0 * f1);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) sum += c + (uint32_t)u < C ? (int64_t)prod[u] : 0;
    }
  }
  for (uint32_t off = (1u << lg) >> 1; off > 0u; off >>= 1) sum += __shfl_xor(sum, (int)off);
  if (l == 0u && row < n_rows) acc[r] += sum;
}

template <class T>
static void launch_observe_t(thrml_state *st, thrml_observer *obs, const T *state) {
  // lanes per row: one per chain group or run of 4 chains, up to a wave
  const uint32_t units = sizeof(T) == 8 ? st->G : cdiv(st->C, 4);
  uint32_t lg = 0;
  while (lg < 6u && (1u << lg) < units) ++lg;
  hipLaunchKernelGGL(observe_kernel<T>, dim3(cdiv(obs->n_rows << lg, 256)), dim3(256), 0,
                     st->prog->ctx->stream, state, (uint64_t)st->prog->n_total, st->G, st->C, st->Cp,
                     obs->row_off.as<uint64_t>(), obs->pos.as<uint32_t>(), obs->n_rows,
                     obs->transform ? 1 : 0, obs->acc.as<int64_t>(), lg);
}

int launch_observe(thrml_state *st, thrml_observer *obs) {
  thrml_prog *p = st->prog;
  if (obs->n_rows == 0) return THRML_OK;
  if (!byte_layout(p)) launch_observe_t(st, obs, st->words.as<uint64_t>());
  else if (p->cat_bytes == 2) launch_observe_t(st, obs, st->cat.as<uint16_t>());
  else launch_observe_t(st, obs, st->cat.as<uint8_t>());
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

// Folds u32 observation counters into u64 totals and clears them.
__global__ void fold_counts_kernel(uint32_t *__restrict__ cnt, uint64_t *__restrict__ acc,
                                   uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  acc[i] += cnt[i];
  cnt[i] = 0u;
}

// Final sums in the caller's order: sum over chains and observations of t_i
// (2*ones - C*n_obs) and of t_a*t_b (C*n_obs - 2*diff), t = 2s - 1.
__global__ void finalize_moments_kernel(const uint32_t *__restrict__ cnt1,
                                        const uint64_t *__restrict__ acc1,
                                        const uint32_t *__restrict__ slot1, uint64_t n1,
                                        const uint32_t *__restrict__ cnt2,
                                        const uint64_t *__restrict__ acc2,
                                        const uint32_t *__restrict__ slot2, uint64_t n2,
                                        int64_t cn, int64_t *__restrict__ out1,
                                        int64_t *__restrict__ out2) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n1) {
    const uint32_t s = slot1 ? slot1[i] : (uint32_t)i;
    out1[i] = 2 * (int64_t)(acc1[s] + cnt1[s]) - cn;
  } else if (i < n1 + n2) {
    const uint64_t k = i - n1;
    const uint32_t s = slot2 ? slot2[k] : (uint32_t)k;
    out2[k] = cn - 2 * (int64_t)(acc2[s] + cnt2[s]);
  }
}

int launch_fold_counts(thrml_ctx *ctx, uint32_t *cnt, uint64_t *acc, uint64_t n) {
  if (n == 0) return THRML_OK;
  hipLaunchKernelGGL(fold_counts_kernel, dim3(cdiv(n, 256)), dim3(256), 0, ctx->stream, cnt, acc, n);
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

int launch_finalize_moments(thrml_ctx *ctx, const uint32_t *cnt1, const uint64_t *acc1,
                            const uint32_t *slot1, uint64_t n1, const uint32_t *cnt2,
                            const uint64_t *acc2, const uint32_t *slot2, uint64_t n2, int64_t cn,
                            int64_t *out1, int64_t *out2) {
  if (n1 + n2 == 0) return THRML_OK;
  hipLaunchKernelGGL(finalize_moments_kernel, dim3(cdiv(n1 + n2, 256)), dim3(256), 0, ctx->stream,
                     cnt1, acc1, slot1, n1, cnt2, acc2, slot2, n2, cn, out1, out2);
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

// ---------------------------------------------------------------------------
// hinton_init (crates/thrml-models/src/ising.rs:602-673) of free block b:
// entry (c, i) of the [C, n_b] uniform tensor is keystream word c*n_b + i of
// the block key; s = (word <= threshold(sigmoid(b_i * beta))).
// A wave takes 16 sites of a chain group.  Bound by instructions: the two
// blocks that hold a chain's 16 words, whose alignment differs by lane, are
// picked from through LDS (a select over 32 registers per word took most of
// the time: blocks of 100,000 sites on average, 32 chains 28.9 -> 15 us, of
// 800 sites, one chain 15.2 -> 5.4 us).
__global__ void hinton_kernel(const uint32_t *__restrict__ key8, const float *__restrict__ prob,
                              uint32_t C, uint32_t n_b, uint64_t *__restrict__ words,
                              uint64_t group_stride, uint64_t blk_off, uint32_t n_seg,
                              uint32_t n_tasks) {
  const uint32_t task = blockIdx.x * 4u + (threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63u;
  if (task >= n_tasks) return;
  const uint32_t g = task / n_seg, seg = task % n_seg;
  const uint32_t c = g * 64u + lane;
  uint64_t *__restrict__ out = words + (size_t)g * group_stride + blk_off;
  Key8 key;
#pragma unroll
  for (int i = 0; i < 8; ++i) key.k[i] = key8[i];
  const uint32_t i0 = seg * 16u;
  const uint64_t w0 = (uint64_t)c * n_b + i0;
  // the 16 words start anywhere in their first block: both blocks go through
  // LDS, lane-major (lane 0's words are at ks[0], ks[64], ...)
  __shared__ uint32_t ks_all[4 * 32 * 64];
  uint32_t *ks = ks_all + (threadIdx.x >> 6) * (32u * 64u) + lane;
  const uint32_t sh = (uint32_t)(w0 & 15u);
  {
    uint32_t a[16];
    chacha_block<8>(key.k, w0 >> 4, a);
#pragma unroll
    for (uint32_t t = 0; t < 16u; ++t) ks[t * 64u] = a[t];
    chacha_block<8>(key.k, (w0 >> 4) + 1, a);
#pragma unroll
    for (uint32_t t = 0; t < 16u; ++t) ks[(t + 16u) * 64u] = a[t];
  }
  // lane k keeps site i0 + k's word and probability
  const float pr = prob[min(i0 + (lane & 15u), n_b - 1u)];
  const uint32_t thr = word_threshold(pr);
  uint64_t mine = 0;
#pragma unroll
  for (uint32_t k = 0; k < 16u; ++k) {
    const uint32_t th = (uint32_t)__builtin_amdgcn_readlane((int)thr, (int)k);
    const uint64_t m = __builtin_amdgcn_ballot_w64(c < C && ks[(sh + k) * 64u] <= th);
    mine = lane == k ? m : mine;
  }
  if (lane < 16u && i0 + lane < n_b) out[i0 + lane] = mine;
}

int launch_hinton(thrml_prog *p, thrml_state *st, uint32_t b, const uint32_t *d_key8,
                  const float *d_prob) {
  const uint32_t n_b = (uint32_t)(p->blk_off[b + 1] - p->blk_off[b]);
  const uint32_t n_seg = cdiv(n_b, 16);
  const uint32_t n_tasks = n_seg * st->G;
  hipLaunchKernelGGL(hinton_kernel, dim3(cdiv(n_tasks, 4)), dim3(256), 0, p->ctx->stream, d_key8,
                     d_prob, st->C, n_b, st->words.as<uint64_t>(),
                     (uint64_t)p->planes * p->n_total, (uint64_t)p->blk_off[b], n_seg, n_tasks);
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

// ---------------------------------------------------------------------------
// FusedKernelBackend counterparts (crates/thrml-kernels/src/lib.rs:55-106).
__global__ void sigmoid_bernoulli_kernel(const float *__restrict__ g, const float *__restrict__ u,
                                         float *__restrict__ o, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  // the inputs are arbitrary floats: the full-range sigmoid, so that a
  // pre-activation below -40 gives probability 0 (u = 0 then samples 0)
  const float prob = sigmoid_full(2.0f * g[i]);
  o[i] = (u[i] < prob) ? 1.0f : 0.0f;  // strict, as sigmoid_bernoulli/kernel.rs:53
}

// gumbel = 0 - log(0 - log(u)) and perturbed = logit + gumbel, as written in
// gumbel_argmax/kernel.rs:61-75, with the full-range log: u = 0 scores -inf
// (never taken after index 0), u = 1 scores +inf, a NaN score never wins.
__device__ __forceinline__ float gumbel_score(float logit, float u) {
  return logit + (0.0f - log_full(0.0f - log_full(u)));
}

__global__ void gumbel_argmax_kernel(const float *__restrict__ l, const float *__restrict__ u,
                                     int32_t *__restrict__ o, uint64_t n, uint32_t q) {
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const float *lr = l + r * q;
  const float *ur = u + r * q;
  float best = gumbel_score(lr[0], ur[0]);
  int32_t arg = 0;
  for (uint32_t k = 1; k < q; ++k) {
    const float v = gumbel_score(lr[k], ur[k]);
    if (v > best) {  // first maximum, gumbel_argmax/kernel.rs:81-83
      best = v;
      arg = (int32_t)k;
    }
  }
  o[r] = arg;
}

int launch_sigmoid_bernoulli(thrml_ctx *ctx, const float *g, const float *u, float *o, uint64_t n) {
  if (n == 0) return THRML_OK;
  hipLaunchKernelGGL(sigmoid_bernoulli_kernel, dim3(cdiv(n, 256)), dim3(256), 0, ctx->stream, g, u,
                     o, n);
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

int launch_gumbel_argmax(thrml_ctx *ctx, const float *l, const float *u, int32_t *o, uint64_t n,
                         uint32_t q) {
  if (n == 0) return THRML_OK;
  hipLaunchKernelGGL(gumbel_argmax_kernel, dim3(cdiv(n, 256)), dim3(256), 0, ctx->stream, l, u, o,
                     n, q);
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

// batch_gather_fused (batch_gather/kernel.rs, launched by batch_gather/forward.rs):
// out[b] = weights[b * batch_stride + sum_i u32(indices[b][i]) * strides[i]],
// the index arithmetic in u32 as the reference's (wrapping).  A linear index
// at or past n_weights reads 0.0 (one of the values a bounds-checked read of
// the reference's buffer may give) instead of leaving the array.
__global__ void batch_gather_kernel(const float *__restrict__ w, uint64_t n_w,
                                    const int32_t *__restrict__ idx, uint64_t batch, uint32_t n_idx,
                                    BatchGatherStrides st, float *__restrict__ out) {
  const uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  uint32_t lin = (uint32_t)b * st.batch_stride;
  const int32_t *ib = idx + b * n_idx;
  for (uint32_t i = 0; i < n_idx; ++i) lin += (uint32_t)ib[i] * st.s[i];
  out[b] = lin < n_w ? w[lin] : 0.0f;
}

int launch_batch_gather(thrml_ctx *ctx, const float *w, uint64_t n_w, const int32_t *idx,
                        uint64_t batch, uint32_t n_idx, const BatchGatherStrides &st, float *out) {
  if (batch == 0) return THRML_OK;
  hipLaunchKernelGGL(batch_gather_kernel, dim3(cdiv(batch, 256)), dim3(256), 0, ctx->stream, w,
                     n_w, idx, batch, n_idx, st, out);
  THRML_HIP(hipGetLastError());
  return THRML_OK;
}

// ---------------------------------------------------------------------------
// Self-check of the hardware-math fast paths (no counterpart in the
// reference): thread i takes uniform numerator 2i+1 for the Gumbel bound and
// every 2^23-th float of [0, 40] (both signs) for the spin decision's two
// relative errors, against double-precision references.
// bits of the smallest float >= v (v >= 0), so that no bound is understated
__device__ __forceinline__ uint32_t f32_bits_up(double v) {
  const float f = (float)v;
  return __builtin_bit_cast(uint32_t, f) + ((double)f < v ? 1u : 0u);
}

__global__ void fast_math_check_kernel(uint32_t *__restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (1u << 23)) return;
  const uint32_t w = (2u * i + 1u) << 8;
  const float eg = fabsf(gumbel_fast(w) - gumbel_b(w));
  double ee = 0.0, es = 0.0;
  for (uint32_t b = i; b <= 0x42200000u; b += (1u << 23)) {  // bits of 40.0f
    const float gp = __builtin_bit_cast(float, b);
#pragma unroll
    for (int sgn = 0; sgn < 2; ++sgn) {
      const float g = sgn ? -gp : gp;
      const double en = exp(-2.0 * (double)g);
      ee = fmax(ee, fabs((double)spin_exp_neg(g) - en) / en);
      const double sig = 1.0 / (1.0 + en);
      es = fmax(es, fabs((double)sigmoid_b(2.0f * g) - sig) / sig);
    }
  }
  // non-negative floats order as their bits
  atomicMax(out + 0, __builtin_bit_cast(uint32_t, eg));
  atomicMax(out + 1, f32_bits_up(ee));
  atomicMax(out + 2, f32_bits_up(es));
}

int launch_fast_math_check(thrml_ctx *ctx, float out[3]) {
  uint32_t *d = nullptr;
  THRML_HIP(hipMalloc(&d, 12));
  uint32_t h[3] = {0u, 0u, 0u};
  hipError_t e = hipMemcpyAsync(d, h, 12, hipMemcpyHostToDevice, ctx->stream);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(fast_math_check_kernel, dim3((1u << 23) / 256), dim3(256), 0, ctx->stream, d);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(h, d, 12, hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  (void)hipFree(d);
  if (e != hipSuccess) return hip_fail(e, "fast math check");
  std::memcpy(out, h, 12);
  return THRML_OK;
}

}  // namespace thrml

// Candidate assignments without a forbidden entry, drawn on the device (gfx950),
// and the C ABI of the sampler.
//
// The ILP forbids every decision variable whose cost is not finite
// (add_inf_cost_constraint, autoparallel/optimize_sharding.py:803-812).  An
// assignment made of independent uniform draws per node nearly always selects
// one, so it scores an objective no feasible plan has.  This sampler walks the
// nodes in graph order and gives node v, uniformly, one of the strategies whose
// entries against the choices already made for its producers are all finite;
// a node that has none takes the plain draw and is counted.  Consistency of the
// flow rows holds by construction, as for the plain draws: an edge's inp_idx is
// its producer's choice.
//
// Two steps.  apc_pack_allowed_columns turns the flags of a build into bit
// columns: for an argument row (edge) and a choice j of its producer, one bit per
// strategy of the consumer, set where the entry is finite.  The strategies a node
// may take are then the AND of one column per argument row, a few 64-bit words,
// instead of a walk over the flag bytes of every strategy; their number is a
// population count, and the draw is the r-th set bit with r one hash of (seed,
// assignment, node) scaled to the count: a function of counters alone, which a
// host can repeat.  (When a lane walked the flag bytes and hashed once per allowed
// strategy, a reservoir walk, 2^20 assignments of the 5.5 M-entry Llama-3-8B graph
// took 136 ms on MI355X.)
#include <algorithm>
#include <exception>
#include <queue>
#include <vector>

#include "apc_device.h"

namespace {

constexpr int kSampleArgs = 6;   // argument rows of a node whose columns a lane keeps in registers
constexpr int kSampleWords = 8;  // words of a node's strategies a lane keeps in registers (512 strategies)
typedef uint64_t u64x2_t __attribute__((ext_vector_type(2)));

// Which of the count allowed strategies of a node is taken, counted in out_idx order:
// uniform in [0, count), from a hash of its own (not the plain draw's).
__host__ __device__ __forceinline__ uint32_t rank_draw(uint32_t h0, int32_t gid, uint32_t count) {
  const uint32_t h = finalise32(h0 ^ node_key(gid) ^ kRankSalt);
  return (uint32_t)(((uint64_t)h * (uint64_t)count) >> 32);
}

// position of the r-th set bit of m (r < popcount(m)): the half, then five halvings of 32 bits
__device__ __forceinline__ int select_bit(uint64_t m, uint32_t r) {
  const uint32_t low = (uint32_t)m, n_low = (uint32_t)__popc(low);
  const bool upper = r >= n_low;
  uint32_t x = upper ? (uint32_t)(m >> 32) : low;
  r -= upper ? n_low : 0u;
  int base = upper ? 32 : 0;
#pragma unroll
  for (int s = 16; s >= 1; s >>= 1) {
    const uint32_t c = (uint32_t)__popc(x & ((1u << s) - 1u));
    const bool above = r >= c;
    r -= above ? c : 0u;
    x = above ? x >> s : x;  // bits past the half that was chosen are never counted
    base += above ? s : 0;
  }
  return base;
}

// the strategies of word w of a node with S strategies
__device__ __forceinline__ uint64_t word_mask(int S, int w) {
  const int left = S - 64 * w;
  return left >= 64 ? ~0ull : (left <= 0 ? 0ull : ((1ull << left) - 1ull));
}

// One wavefront per (argument row e, 64 strategies of the consumer).  lane = choice j of the
// producer, so a load reads 64 consecutive flag bytes of one row of the block; a walk over the
// 64 strategies o fills, one bit a step, the word every lane keeps of its own column.
__global__ void __launch_bounds__(kBlock)
pack_allowed_columns_kernel(apc_problem p, const uint8_t* __restrict__ flags,
                            const int64_t* __restrict__ col_off, int max_words,
                            uint64_t* __restrict__ colbits) {
  const int64_t unit = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  const int e = __builtin_amdgcn_readfirstlane((int)(unit / max_words));
  const int w = __builtin_amdgcn_readfirstlane((int)(unit % max_words));
  if (e >= p.n_edge) return;
  const apc_edge* ed = p.edges + e;  // wave-uniform: scalar loads
  const int sdst = ed->sdst, ssrc = ed->ssrc;
  const int W = (sdst + 63) >> 6;
  if (w >= W) return;
  const int Wc = (W + 1) & ~1;  // words from one column to the next: whole pairs
  const int lane = threadIdx.x & 63;
  const int rows = min(64, sdst - 64 * w);
  const uint8_t* __restrict__ tile = flags + ed->off + (int64_t)(64 * w) * ssrc;
  uint64_t* __restrict__ out = colbits + col_off[e] + w;
  for (int j0 = 0; j0 < ssrc; j0 += 64) {
    const int j = j0 + lane;
    const bool mine = j < ssrc;
    const uint8_t* __restrict__ col = tile + (mine ? j : 0);
    uint64_t m = 0;
#pragma unroll 8
    for (int k = 0; k < rows; ++k)
      m |= (uint64_t)((col[(int64_t)k * ssrc] & APC_ENTRY_NONFINITE) == 0) << k;
    if (mine) out[(int64_t)j * Wc] = m;
  }
}

// One lane per assignment.  The lanes of a wave read, per argument row and word, the column
// their producer's choice names: 8-byte gathers inside one block of columns.
// kAhead: for launches of few wavefronts (see below).
template <bool kAhead>
__global__ void __launch_bounds__(kBlock)
sample_feasible_kernel(apc_problem p, const uint64_t* __restrict__ colbits,
                       const int64_t* __restrict__ col_off, uint64_t seed, int64_t first,
                       int64_t n_assign, const int32_t* __restrict__ node_gid, int first_node,
                       const uint64_t* __restrict__ row_filter, const int64_t* __restrict__ filter_off,
                       uint16_t* __restrict__ assign, int32_t* __restrict__ n_fallback) {
  const int64_t a = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (a >= n_assign) return;
  const uint32_t h0 = assignment_hash(seed, first + a);
  int fallbacks = 0;
  // What the walk needs to know about a node is the same for every lane.  With few
  // assignments a launch is a handful of wavefronts and lasts as long as its chain of
  // dependent loads; kAhead requests this part one node ahead, which takes two links out of
  // the chain (16 384 assignments of a 5 000-node window: 11.0 -> 9.8 ms).  A launch that
  // fills the chip hides the chain by itself and only pays for the registers (2^20
  // assignments of the same window: 62 -> 72 ms), so it runs without.
  struct Head {
    int S, gid, e0, e1;
    int64_t keep;  // first word of the node's filter, or -1
    int src[kSampleArgs];
    int64_t off[kSampleArgs];
  };
  auto load_head = [&](int v) -> Head {
    Head h;
    h.S = p.node_nstrat[v];
    h.gid = node_gid ? node_gid[v] : v;
    h.e0 = p.node_edge_off[v];
    h.e1 = p.node_edge_off[v + 1];
    h.keep = filter_off ? filter_off[v] : -1;
    if (kAhead) {
#pragma unroll
      for (int i = 0; i < kSampleArgs; ++i) {
        h.src[i] = -1;
        h.off[i] = 0;
        if (h.e0 + i < h.e1) {
          h.src[i] = p.edges[h.e0 + i].src_node;
          h.off[i] = col_off[h.e0 + i];
        }
      }
    }
    return h;
  };
  Head next = {};
  if (kAhead && first_node < p.n_node) next = load_head(first_node);
  for (int v = first_node; v < p.n_node; ++v) {
    const Head head = kAhead ? next : load_head(v);
    if (kAhead && v + 1 < p.n_node) next = load_head(v + 1);
    const int S = head.S, gid = head.gid, e0 = head.e0, e1 = head.e1;
    const int W = (S + 63) >> 6;
    const int Wc = (W + 1) & ~1;  // words from one column to the next: whole pairs, 16-byte aligned
    // the column of every argument row: that of the producer's choice
    const u64x2_t* col[kSampleArgs];
#pragma unroll
    for (int i = 0; i < kSampleArgs; ++i) {
      col[i] = reinterpret_cast<const u64x2_t*>(colbits);
      if (e0 + i < e1) {
        const int u = kAhead ? head.src[i] : p.edges[e0 + i].src_node;
        const int64_t j = u >= 0 ? (int64_t)assign[(size_t)u * n_assign + a] : 0;
        col[i] = reinterpret_cast<const u64x2_t*>(colbits + (kAhead ? head.off[i] : col_off[e0 + i]) + j * Wc);
      }
    }
    // words 2 q and 2 q + 1 of the node's allowed strategies: a lane reads its columns 16 bytes at
    // a time (the lanes of a wave read different columns, and such a load costs the same for 8
    // bytes as for 16)
    auto allowed_pair = [&](int q) -> u64x2_t {
      u64x2_t m = {word_mask(S, 2 * q), word_mask(S, 2 * q + 1)};
      if (head.keep >= 0) {  // the strategies the node may take at all
        m.x &= row_filter[head.keep + 2 * q];
        if (2 * q + 1 < W) m.y &= row_filter[head.keep + 2 * q + 1];
      }
#pragma unroll
      for (int i = 0; i < kSampleArgs; ++i)
        if (e0 + i < e1) m &= col[i][q];
      for (int e = e0 + kSampleArgs; e < e1; ++e) {  // a node with more argument rows than the registers hold
        const int u = p.edges[e].src_node;
        const int64_t j = u >= 0 ? (int64_t)assign[(size_t)u * n_assign + a] : 0;
        m &= reinterpret_cast<const u64x2_t*>(colbits + col_off[e] + j * Wc)[q];
      }
      return m;
    };
    uint32_t count = 0;
    int pick = 0;
    if (W == 1) {  // up to 64 strategies (most nodes of a traced model): one word, read by itself
      uint64_t m = word_mask(S, 0);
      if (head.keep >= 0) m &= row_filter[head.keep];
#pragma unroll
      for (int i = 0; i < kSampleArgs; ++i)
        if (e0 + i < e1) m &= reinterpret_cast<const uint64_t*>(col[i])[0];
      for (int e = e0 + kSampleArgs; e < e1; ++e) {
        const int u = p.edges[e].src_node;
        const int64_t j = u >= 0 ? (int64_t)assign[(size_t)u * n_assign + a] : 0;
        m &= colbits[col_off[e] + j * Wc];
      }
      count = (uint32_t)__popcll(m);
      if (count > 0) pick = select_bit(m, rank_draw(h0, gid, count));
    } else if (W <= kSampleWords) {  // wave-uniform: the words stay in registers
      uint64_t m[kSampleWords];
#pragma unroll
      for (int q = 0; q < kSampleWords / 2; ++q) {
        const u64x2_t mm = 2 * q < W ? allowed_pair(q) : u64x2_t{0ull, 0ull};
        m[2 * q] = mm.x;
        m[2 * q + 1] = mm.y;
        count += (uint32_t)__popcll(mm.x) + (uint32_t)__popcll(mm.y);
      }
      if (count > 0) {
        uint32_t r = rank_draw(h0, gid, count);
        bool found = false;
#pragma unroll
        for (int w = 0; w < kSampleWords; ++w) {
          const uint32_t c = (uint32_t)__popcll(m[w]);
          if (!found && r < c) {
            pick = 64 * w + select_bit(m[w], r);
            found = true;
          }
          if (!found) r -= c;
        }
      }
    } else {  // more than 512 strategies: the words are formed twice
      for (int q = 0; 2 * q < W; ++q) {
        const u64x2_t mm = allowed_pair(q);
        count += (uint32_t)__popcll(mm.x) + (uint32_t)__popcll(mm.y);
      }
      if (count > 0) {
        uint32_t r = rank_draw(h0, gid, count);
        for (int q = 0; 2 * q < W; ++q) {
          const u64x2_t mm = allowed_pair(q);
          const uint32_t cx = (uint32_t)__popcll(mm.x), cy = (uint32_t)__popcll(mm.y);
          if (r < cx) {
            pick = 128 * q + select_bit(mm.x, r);
            break;
          }
          r -= cx;
          if (r < cy) {
            pick = 128 * q + 64 + select_bit(mm.y, r);
            break;
          }
          r -= cy;
        }
      }
    }
    if (count == 0) {
      pick = (int)plain_draw(h0, gid, S);
      ++fallbacks;
    }
    assign[(size_t)v * n_assign + a] = (uint16_t)pick;
  }
  n_fallback[a] = fallbacks;
}

// ---------------------------------------------------------------------------
// The same draws by several wavefronts per 64 assignments, for batches whose lane-per-assignment
// walk is too few wavefronts to hide its chain of loads.  A node waits only for its own
// producers, so a workgroup takes the nodes in steps (apc_sample_steps): up to n_waves nodes
// whose producers all lie in earlier steps, one wavefront each, a barrier behind them.  The
// choices of the last kRing places travel through LDS; older ones are read back from the
// matrix, requested a step ahead.  Every kRing / 4 places the workgroup waits for its stores
// too, so a choice that has left the ring is in the matrix by the time it is read.
// Bound by the latency of a step (a column from L2, the draw's instructions, the barrier: about
// 1 us) while the workgroups are few, by instructions from 131 072 assignments of a decoder on.
// Against one lane per assignment, Llama-3-8B graph: 65 536 assignments 9.5 -> 3.8 ms, 131 072
// 10.0 -> 5.1, 524 288 21.2 -> 17.5; planner DAG window of 1 600 nodes, 16 384 assignments:
// 5.0 -> 0.55 ms.
// ---------------------------------------------------------------------------
constexpr int kRing = 128;
static_assert(sizeof(apc_sample_rec) == 64, "a record is one scalar load");
typedef uint32_t u32x16_t __attribute__((ext_vector_type(16)));

constexpr int kRingZero = kRing;  // a row of zeros: the choice of a missing producer
constexpr uint32_t kFromMatrix = 255;

// kNamed: argument rows whose choices are requested a step ahead (from the ring and from the
// matrix, one of the two is used: no branch, so nothing waits for one row before the next is
// requested); kIds: node ids or filters are given.
template <int kWaves, int kNamed, bool kIds>
__global__ void __launch_bounds__(64 * kWaves)
sample_steps_kernel(apc_problem p, const apc_sample_rec* __restrict__ recs, int n_step,
                    const uint64_t* __restrict__ colbits, const int64_t* __restrict__ col_off, uint64_t seed,
                    int64_t first, int64_t n_assign, const int32_t* __restrict__ node_gid,
                    const uint64_t* __restrict__ row_filter, const int64_t* __restrict__ filter_off,
                    uint16_t* __restrict__ assign, int32_t* __restrict__ n_fallback) {
  __shared__ uint16_t s_ring[kRing + 1][64];
  __shared__ int s_fallback[64];
  constexpr int kSync = kRing / 4 / kWaves;  // steps from one wait for the stores to the next
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t a_raw = (int64_t)blockIdx.x * 64 + lane;
  const bool mine = a_raw < n_assign;
  const int64_t a = mine ? a_raw : n_assign - 1;  // lanes past the end repeat the last one and store nothing
  const uint32_t h0 = assignment_hash(seed, first + a);
  if (threadIdx.x < 64) {
    s_fallback[threadIdx.x] = 0;
    s_ring[kRingZero][threadIdx.x] = 0;
  }
  int fallbacks = 0;
  auto load_rec = [&](int t) -> apc_sample_rec {
    union { u32x16_t raw; apc_sample_rec rec; } u;
    u.raw = *reinterpret_cast<const u32x16_t*>(recs + (int64_t)(t < n_step ? t : n_step - 1) * kWaves + wave);
    return u.rec;
  };
  const u64x2_t* const columns = reinterpret_cast<const u64x2_t*>(colbits);
  const uint16_t* const my_assign = assign + a;
  auto matrix_choice = [&](uint32_t src) -> uint32_t { return my_assign[(size_t)src * n_assign]; };
  auto ring_choice = [&](uint32_t from) -> uint32_t {
    const uint32_t slot = from >> 24;
    return s_ring[slot == kFromMatrix ? (uint32_t)kRingZero : slot][lane];
  };
  // A step is a chain: ring -> columns -> draw -> ring.  What else it needs is requested
  // behind its columns' addresses: a step ahead the choices from the matrix, two steps ahead
  // the record (not earlier in a step: a wait for the ring is one for every scalar load, too).
  apc_sample_rec rec = load_rec(0), next = load_rec(1);
  uint32_t far[kNamed], far_next[kNamed];
#pragma unroll
  for (int i = 0; i < kNamed; ++i) far[i] = matrix_choice(rec.arg[i].from & 0xFFFFFFu);
  __syncthreads();
  for (int t = 0; t < n_step; ++t) {
    const int S = rec.nstrat, n_arg = rec.n_arg;
    const int W = (S + 63) >> 6;
    const int Wq = (W + 1) >> 1;  // pairs of words from one column to the next
    const u64x2_t* col[kSampleArgs];  // the column of every argument row: that of the producer's choice
#pragma unroll
    for (int i = 0; i < kSampleArgs; ++i) col[i] = columns;
    uint32_t near[kNamed];
#pragma unroll
    for (int i = 0; i < kNamed; ++i) near[i] = ring_choice(rec.arg[i].from);
#pragma unroll
    for (int i = 0; i < kNamed; ++i) {
      const uint32_t j = (rec.arg[i].from >> 24) == kFromMatrix ? far[i] : near[i];
      col[i] = columns + rec.arg[i].col + j * (uint32_t)Wq;
    }
#pragma unroll
    for (int i = 0; i < kNamed; ++i) far_next[i] = matrix_choice(next.arg[i].from & 0xFFFFFFu);
    __builtin_amdgcn_sched_barrier(0);
    const apc_sample_rec after = load_rec(t + 2);
    if (rec.node >= 0) {  // else no node for this wavefront in this step
      const int v = rec.node;
      const int gid = kIds && node_gid ? node_gid[v] : v;
      const int64_t keep = kIds && filter_off ? filter_off[v] : -1;  // first word of the node's filter, or -1
      if (n_arg > kNamed) {
#pragma unroll
        for (int i = kNamed; i < kSampleArgs; ++i) {
          if (i >= n_arg) break;
          const uint32_t from = rec.arg[i].from;
          const uint32_t j = (from >> 24) == kFromMatrix ? matrix_choice(from & 0xFFFFFFu) : ring_choice(from);
          col[i] = columns + rec.arg[i].col + j * (uint32_t)Wq;
        }
      }
      // argument rows past those of a record: their producers are in the matrix (apc_sample_steps)
      auto more_column = [&](int e) -> const u64x2_t* {
        const int src = p.edges[e].src_node;
        return columns + (col_off[e] >> 1) + (src >= 0 ? matrix_choice((uint32_t)src) * (uint32_t)Wq : 0u);
      };
      auto allowed_pair = [&](int q) -> u64x2_t {  // words 2 q and 2 q + 1 of the node's allowed strategies
        u64x2_t m = {word_mask(S, 2 * q), word_mask(S, 2 * q + 1)};
        if (keep >= 0) {
          m.x &= row_filter[keep + 2 * q];
          if (2 * q + 1 < W) m.y &= row_filter[keep + 2 * q + 1];
        }
#pragma unroll
        for (int i = 0; i < kSampleArgs; ++i)
          if (i < n_arg) m &= col[i][q];
        for (int i = kSampleArgs; i < n_arg; ++i) m &= more_column(p.node_edge_off[v] + i)[q];
        return m;
      };
      uint32_t count = 0;
      int pick = 0;
      if (W == 1 && n_arg <= 2) {  // most nodes of a traced model
        const uint64_t w0 = *reinterpret_cast<const uint64_t*>(col[0]);
        const uint64_t w1 = *reinterpret_cast<const uint64_t*>(col[n_arg > 1 ? 1 : 0]);
        uint64_t m = word_mask(S, 0);
        if (kIds && keep >= 0) m &= row_filter[keep];
        if (n_arg > 0) m &= w0 & w1;
        count = (uint32_t)__popcll(m);
        if (count > 0) pick = select_bit(m, rank_draw(h0, gid, count));
      } else if (W == 1) {
        uint64_t m = word_mask(S, 0);
        if (kIds && keep >= 0) m &= row_filter[keep];
#pragma unroll
        for (int i = 0; i < kSampleArgs; ++i)
          if (i < n_arg) m &= reinterpret_cast<const uint64_t*>(col[i])[0];
        for (int i = kSampleArgs; i < n_arg; ++i)
          m &= reinterpret_cast<const uint64_t*>(more_column(p.node_edge_off[v] + i))[0];
        count = (uint32_t)__popcll(m);
        if (count > 0) pick = select_bit(m, rank_draw(h0, gid, count));
      } else if (W <= kSampleWords) {
        uint64_t m[kSampleWords];
#pragma unroll
        for (int q = 0; q < kSampleWords / 2; ++q) {
          const u64x2_t mm = 2 * q < W ? allowed_pair(q) : u64x2_t{0ull, 0ull};
          m[2 * q] = mm.x;
          m[2 * q + 1] = mm.y;
          count += (uint32_t)__popcll(mm.x) + (uint32_t)__popcll(mm.y);
        }
        if (count > 0) {
          uint32_t r = rank_draw(h0, gid, count);
          uint64_t word = m[0];
          bool found = false;
#pragma unroll
          for (int w = 0; w < kSampleWords; ++w) {
            const uint32_t c = (uint32_t)__popcll(m[w]);
            if (!found && r < c) {
              pick = 64 * w;
              word = m[w];
              found = true;
            }
            if (!found) r -= c;
          }
          pick += select_bit(word, r);
        }
      } else {  // more than 512 strategies: the words are formed twice
        for (int q = 0; 2 * q < W; ++q) {
          const u64x2_t mm = allowed_pair(q);
          count += (uint32_t)__popcll(mm.x) + (uint32_t)__popcll(mm.y);
        }
        if (count > 0) {
          uint32_t r = rank_draw(h0, gid, count);
          for (int q = 0; 2 * q < W; ++q) {
            const u64x2_t mm = allowed_pair(q);
            const uint32_t cx = (uint32_t)__popcll(mm.x), cy = (uint32_t)__popcll(mm.y);
            if (r < cx) {
              pick = 128 * q + select_bit(mm.x, r);
              break;
            }
            r -= cx;
            if (r < cy) {
              pick = 128 * q + 64 + select_bit(mm.y, r);
              break;
            }
            r -= cy;
          }
        }
      }
      if (count == 0) {
        pick = (int)plain_draw(h0, gid, S);
        ++fallbacks;
      }
      s_ring[(t * kWaves + wave) & (kRing - 1)][lane] = (uint16_t)pick;
      if (mine) assign[(size_t)v * n_assign + a] = (uint16_t)pick;
    }
    rec = next;
    next = after;
#pragma unroll
    for (int i = 0; i < kNamed; ++i) far[i] = far_next[i];
    if ((t + 1) % kSync == 0)
      __syncthreads();  // the stores too
    else
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the ring only
  }
  if (fallbacks) atomicAdd(&s_fallback[lane], fallbacks);
  __syncthreads();
  if (wave == 0 && mine) n_fallback[a] = s_fallback[lane];
}

}  // namespace

extern "C" {

// Host side of sample_steps_kernel: which node every wavefront draws in every step.  Nodes
// with the longest chain of consumers behind them go first.
int apc_sample_steps(int32_t n_node, int32_t n_edge, const int32_t* node_edge_off, const int32_t* edge_src,
                     const int32_t* node_nstrat, const int64_t* col_off, int32_t first_node, int32_t n_waves_asked,
                     apc_sample_rec* recs, int32_t max_step, int32_t* n_step, int32_t* n_waves_out) {
  if (n_node < 0 || n_edge < 0 || first_node < 0 || first_node > n_node || !n_step || !n_waves_out ||
      (n_node > first_node && (!node_edge_off || !node_nstrat || !recs)) || (n_edge > 0 && (!edge_src || !col_off)))
    return fail(APC_ERR_INVALID, "apc_sample_steps: null argument or first_node out of range%s");
  if (n_node > 0xFFFFFF) return fail(APC_ERR_INVALID, "apc_sample_steps: more than 2^24 - 1 nodes%s");
  if (n_waves_asked != 0 && n_waves_asked != 2 && n_waves_asked != 16)
    return fail(APC_ERR_INVALID, "apc_sample_steps: n_waves must be 0 (choose), 2 or 16%s");
  for (int v = first_node; v < n_node; ++v) {
    if (node_edge_off[v] < 0 || node_edge_off[v] > node_edge_off[v + 1] || node_edge_off[v + 1] > n_edge)
      return fail(APC_ERR_INVALID, "apc_sample_steps: node_edge_off is no list of offsets%s");
    for (int e = node_edge_off[v]; e < node_edge_off[v + 1]; ++e)
      if (edge_src[e] >= v) return fail(APC_ERR_INVALID, "apc_sample_steps: a producer behind its consumer%s");
  }
  *n_step = 0;
  try {
    const int n = n_node - first_node;
    std::vector<int32_t> height(n, 0), waits(n, 0), off(n + 1, 0), place(n, -1);
    for (int v = n_node - 1; v >= first_node; --v)
      for (int e = node_edge_off[v]; e < node_edge_off[v + 1]; ++e)
        if (edge_src[e] >= first_node) {
          const int u = edge_src[e] - first_node;
          height[u] = std::max(height[u], height[v - first_node] + 1);
          ++off[u + 1];
          ++waits[v - first_node];
        }
    // Two wavefronts for a graph that is a few chains (a decoder has two nodes ready at a time:
    // four save a tenth of the time of a small batch and cost 40% at 131 072), sixteen where
    // there is work for most of them (16 384 assignments of a 1 600-node window of the planner
    // DAG: 0.55 ms with sixteen, 2.15 with two).
    const int depth = n > 0 ? 1 + *std::max_element(height.begin(), height.end()) : 1;
    const int n_waves = n_waves_asked ? n_waves_asked : n >= 6 * depth ? 16 : 2;
    *n_waves_out = n_waves;
    for (int u = 0; u < n; ++u) off[u + 1] += off[u];
    std::vector<int32_t> consumer(off[n]), at(off.begin(), off.end() - 1);
    for (int v = first_node; v < n_node; ++v)
      for (int e = node_edge_off[v]; e < node_edge_off[v + 1]; ++e)
        if (edge_src[e] >= first_node) consumer[at[edge_src[e] - first_node]++] = v - first_node;
    auto later = [&](int32_t x, int32_t y) { return height[x] != height[y] ? height[x] < height[y] : x > y; };
    std::priority_queue<int32_t, std::vector<int32_t>, decltype(later)> ready(later);
    // a node whose record cannot name all its producers reads the others from the matrix: it
    // waits until they have left the ring
    std::vector<std::vector<int32_t>> held;  // [step]: nodes that become ready then
    std::vector<int32_t> released;
    const int ring_steps = kRing / n_waves;
    for (int v = 0; v < n; ++v)
      if (waits[v] == 0) ready.push(v);
    int left = n, t = 0;
    std::vector<int32_t> taken;
    for (; left > 0; ++t) {
      if (t >= max_step) return fail(APC_ERR_UNSUPPORTED, "apc_sample_steps: more steps than max_step%s");
      if (t < (int)held.size())
        for (int v : held[t]) ready.push(v);
      taken.clear();
      while (!ready.empty() && (int)taken.size() < n_waves) {
        taken.push_back(ready.top());
        ready.pop();
      }
      for (int w = 0; w < n_waves; ++w) {
        apc_sample_rec r;
        memset(&r, 0, sizeof(r));
        r.node = -1;
        for (auto& arg : r.arg) arg.from = (uint32_t)kRingZero << 24;
        if (w < (int)taken.size()) {
          const int v = taken[w] + first_node;
          place[taken[w]] = t * n_waves + w;
          r.node = v;
          r.nstrat = node_nstrat[v];
          const int e0 = node_edge_off[v];
          r.n_arg = node_edge_off[v + 1] - e0;
          for (int i = 0; i < r.n_arg && i < kSampleArgs; ++i) {
            const int src = edge_src[e0 + i];
            r.arg[i].from = src < 0 ? (uint32_t)kRingZero << 24 : (kFromMatrix << 24) | (uint32_t)src;
            // in the ring unless a place of this step or an earlier one has taken its slot
            if (src >= first_node && (t + 1) * n_waves - place[src - first_node] <= kRing)
              r.arg[i].from = (uint32_t)(place[src - first_node] & (kRing - 1)) << 24 | (uint32_t)src;
            const int64_t col = col_off[e0 + i];
            if (col < 0 || (col & 1) || (col >> 1) > 0x7FFFFFFF)
              return fail(APC_ERR_INVALID, "apc_sample_steps: col_off must be even and below 2^32%s");
            r.arg[i].col = (uint32_t)(col >> 1);
          }
        }
        recs[(int64_t)t * n_waves + w] = r;
      }
      left -= (int)taken.size();
      for (int u : taken)
        for (int q = off[u]; q < off[u + 1]; ++q) {
          const int v = consumer[q];
          if (--waits[v] > 0) continue;
          if (node_edge_off[first_node + v + 1] - node_edge_off[first_node + v] <= kSampleArgs) {
            released.push_back(v);
          } else {
            if ((int)held.size() <= t + ring_steps) held.resize(t + ring_steps + 1);
            held[t + ring_steps].push_back(v);
          }
        }
      for (int v : released) ready.push(v);
      released.clear();
    }
    *n_step = t;
  } catch (const std::exception&) {
    return fail(APC_ERR_INVALID, "apc_sample_steps: out of host memory%s");
  }
  return 0;
}

int apc_sample_feasible_steps(const apc_problem* p, const apc_sample_rec* recs, int32_t n_step, int32_t n_waves,
                              const uint64_t* colbits, const int64_t* col_off, uint64_t seed, int64_t first,
                              int64_t n_assign, const int32_t* node_gid, const uint64_t* row_filter,
                              const int64_t* filter_off, uint16_t* assign, int32_t* n_fallback, void* stream) {
  if (int rc = validate_problem(p)) return rc;
  if (n_assign <= 0) return 0;
  if (!assign || !n_fallback || !recs || n_step <= 0 || (p->n_entry > 0 && (!colbits || !col_off)))
    return fail(APC_ERR_INVALID, "apc_sample_feasible_steps: null argument or no steps%s");
  if ((row_filter == nullptr) != (filter_off == nullptr))
    return fail(APC_ERR_INVALID, "apc_sample_feasible_steps: row_filter and filter_off come together%s");
  const int64_t blocks = (n_assign + 63) / 64;
  if (blocks > 0x7FFFFFFF) return fail(APC_ERR_INVALID, "apc_sample_feasible_steps: too many assignments for one launch%s");
#define APC_SAMPLE_STEPS(W, NAMED, IDS)                                                                             \
  hipLaunchKernelGGL((sample_steps_kernel<W, NAMED, IDS>), dim3((unsigned)blocks), dim3(64 * W), 0,                  \
                     (hipStream_t)stream, *p, recs, n_step, colbits, col_off, seed, first, n_assign, node_gid,      \
                     row_filter, filter_off, assign, n_fallback)
  const bool ids = node_gid || row_filter;
  switch (n_waves) {
    case 2: if (ids) APC_SAMPLE_STEPS(2, 2, true); else APC_SAMPLE_STEPS(2, 2, false); break;
    case 16: if (ids) APC_SAMPLE_STEPS(16, 4, true); else APC_SAMPLE_STEPS(16, 4, false); break;
    default: return fail(APC_ERR_INVALID, "apc_sample_feasible_steps: n_waves must be 2 or 16%s");
  }
#undef APC_SAMPLE_STEPS
  return check_launch("sample_steps_kernel");
}

int apc_pack_allowed_columns(const apc_problem* p, const uint8_t* flags, const int64_t* col_off,
                             int32_t max_words, uint64_t* colbits, void* stream) {
  if (int rc = validate_problem(p)) return rc;
  if (p->n_edge == 0 || p->n_entry == 0) return 0;
  if (!flags || !col_off || !colbits || max_words <= 0)
    return fail(APC_ERR_INVALID, "apc_pack_allowed_columns: null argument or max_words <= 0%s");
  const int64_t units = (int64_t)p->n_edge * max_words;
  const int64_t grid = (units + (kBlock / 64) - 1) / (kBlock / 64);
  if (grid > 0x7FFFFFFF)
    return fail(APC_ERR_INVALID, "apc_pack_allowed_columns: too many argument rows for one launch%s");
  hipLaunchKernelGGL(pack_allowed_columns_kernel, dim3((unsigned)grid), dim3(kBlock), 0, (hipStream_t)stream, *p,
                     flags, col_off, (int)max_words, colbits);
  return check_launch("pack_allowed_columns_kernel");
}

int apc_sample_feasible(const apc_problem* p, const uint64_t* colbits, const int64_t* col_off, uint64_t seed,
                        int64_t first, int64_t n_assign, const int32_t* node_gid, int32_t first_node,
                        const uint64_t* row_filter, const int64_t* filter_off, uint16_t* assign,
                        int32_t* n_fallback, void* stream) {
  if (int rc = validate_problem(p)) return rc;
  if (n_assign <= 0) return 0;
  if (!assign || !n_fallback || (p->n_entry > 0 && (!colbits || !col_off)))
    return fail(APC_ERR_INVALID, "apc_sample_feasible: null argument%s");
  if (first_node < 0 || first_node > p->n_node)
    return fail(APC_ERR_INVALID, "apc_sample_feasible: first_node out of range%s");
  if ((row_filter == nullptr) != (filter_off == nullptr))
    return fail(APC_ERR_INVALID, "apc_sample_feasible: row_filter and filter_off come together%s");
  const dim3 grid((unsigned)((n_assign + kBlock - 1) / kBlock));
  // Fewer wavefronts than SIMDs: batches that apc_sample_feasible_steps does not take (a layout that
  // cannot be had or would be longer than the walk).
  if (n_assign < 65536)
    hipLaunchKernelGGL(sample_feasible_kernel<true>, grid, dim3(kBlock), 0, (hipStream_t)stream, *p, colbits, col_off,
                       seed, first, n_assign, node_gid, (int)first_node, row_filter, filter_off, assign, n_fallback);
  else
    hipLaunchKernelGGL(sample_feasible_kernel<false>, grid, dim3(kBlock), 0, (hipStream_t)stream, *p, colbits, col_off,
                       seed, first, n_assign, node_gid, (int)first_node, row_filter, filter_off, assign, n_fallback);
  return check_launch("sample_feasible_kernel");
}

uint32_t apc_sample_rank(uint64_t seed, int64_t a, int32_t node, uint32_t count) {
  return count ? rank_draw(assignment_hash(seed, a), node, count) : 0u;
}

}  // extern "C"

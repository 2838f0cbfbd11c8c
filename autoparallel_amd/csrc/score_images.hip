// Batch scoring of graphs with small blocks from tile images (gfx950), and its C ABI.
//
// With a lane per assignment and one workgroup per CU, batches of up to 2^18 are a few wavefronts per SIMD, and a walk
// over tiles (score_tiles.hip) is bound by everything that a step does besides its sums: scalar loads of its record and
// the wait for them at every LDS read, branches on what kind of step it is, the look-ups before a copy can be asked
// for.  So a launch in front of it lays every tile out in one piece, in the form in which it then lies in LDS: its
// matrices, the terms of its nodes, a few words per edge, per node and per row of choices, and what a workgroup has to
// know to ask for the next tile.  A copy is then consecutive memory, 4 KB per instruction group; explicit choices come
// the same way, rows of 16 bits straight into LDS, a tile further ahead where three buffers fit (they come from memory,
// and a tile lasts about as long as that takes); the words of an edge are in the lanes' registers (lane i: edge i) and
// come from there with v_readlane; and eight edges are walked side by side, with one branch per four, taken where one of them
// is not of the common kind.
// Measured, MI355X, Llama-3-8B graph (8 533 edges): 131 072 explicit assignments 5.7 -> 2.6 ms, 262 144 6.7 -> 3.8,
// 131 072 random ones 4.8 -> 2.9; the images (43 MB) take 20 us of that.  What bounds it: at 262 144 about as much
// the LDS (20 cycles of reads per edge and wavefront and the copies, half of the time) as instructions (0.5 busy; 41
// vector and 30 scalar ones per edge); at 131 072 and below the latency of a wavefront's own chain, 2.4 ms however few.
// Not better: a word per field instead of packed words (fewer scalar instructions, 4.1 against 3.8 ms at 262 144),
// twelve edges side by side, or the reads left to the compiler's order (it waits for each pair).
// Sums run in node order, then argument order, as in score_kernel: the same bits.
#include <algorithm>

#include "apc_device.h"
#include "score_tiles.h"

namespace {

using namespace apc_tiles;

constexpr int kHeadBytes = 2048;  // of an image: edges, nodes, rows, Head
constexpr int kNodesAt = 1024, kRowsAt = 1536, kHeadAt = 1792;
constexpr int kImageBytes = APC_SCORE_IMAGE_BYTES;
constexpr int kUnroll = 4;
typedef const __attribute__((address_space(3))) uint16_t* lds_u16_ptr_t;
typedef const __attribute__((address_space(3))) double* lds_f64_ptr_t;
constexpr int kRowSlots = kRows + 1;  // the last one: zeros, the choice of a missing producer
static_assert(kHeadBytes + kTileDoubles * 8 <= kImageBytes && kImageBytes % 1024 == 0, "an image");

// Edge i of a tile: what a walk needs of it, in few words (a v_readlane each; taking them apart costs the vector
// unit nothing).  Edges and nodes are filled up to a multiple of kUnroll with ones that add -0.0, which changes no
// sum: 0.0 times -1.
struct EdgeWords {
  uint32_t matrix;   // in LDS, doubles (bits 0-15), and a row of it, bytes
  uint32_t choices;  // rows of the node's (bits 0-15) and the producer's choices, bytes
  uint32_t terms;    // the node's per-argument terms, doubles (bits 0-15), kEdge*
  int32_t mult;
};
constexpr uint32_t kEdgeOdd = 1u << 16;  // not what nearly all are: with a producer, transitions that count, multiplier 1
constexpr uint32_t kEdgeSource = 1u << 17, kEdgeTransition = 1u << 18;
struct NodeWords {
  uint32_t at;  // row of its choice, bytes (bits 0-15), per-argument terms, doubles
  int32_t nargs;
};
// Row i: what its draw starts from, strategies
struct RowWords { uint32_t w[2]; };
// What a workgroup has to know before it can ask for the tiles behind this one
struct Head {
  int32_t n_edge, n_node, n_row;
  int32_t next_chunks;   // of the next tile's image, 1 KB each
  int32_t any_edge;
  int32_t reserved;
  double zero;
  int32_t row[2][kRows];  // nodes whose choices the next tile and the one behind it read
};
static_assert(sizeof(EdgeWords) * kTileSteps <= kNodesAt && sizeof(NodeWords) * kTileSteps <= kRowsAt - kNodesAt &&
              sizeof(RowWords) * kRows <= kHeadAt - kRowsAt && sizeof(Head) + kHeadAt <= kHeadBytes, "an image's head");

__device__ __forceinline__ int image_doubles(const apc_score_tile& t, const apc_score_unit* __restrict__ units) {
  const apc_score_unit last = units[t.unit1 - 1];  // the units of a tile fill its buffer in order
  return (last.lds + last.n + 1) & ~1;
}

// One workgroup per tile: what the walk reads of it, in one piece.
__global__ void __launch_bounds__(kBlock)
score_images_kernel(apc_problem p, const double* __restrict__ per_arg, const double* __restrict__ table,
                    const apc_score_step* __restrict__ steps, const apc_score_tile* __restrict__ tiles, int n_tile,
                    const apc_score_unit* __restrict__ units, const int32_t* __restrict__ node_gid, int row_bytes,
                    char* __restrict__ images) {
  const int t = blockIdx.x, tid = threadIdx.x;
  const apc_score_tile tile = tiles[t];
  char* const image = images + (size_t)t * kImageBytes;
  double* const body = reinterpret_cast<double*>(image + kHeadBytes);
  for (int u = tile.unit0 + (tid >> 6); u < tile.unit1; u += kBlock / 64) {
    const apc_score_unit unit = units[u];
    const double* __restrict__ from = unit.kind == 0 ? table : unit.kind == 1 ? per_arg : p.default_vals;
    for (int i = tid & 63; i < unit.n; i += 64) body[unit.lds + i] = from[unit.src + i];
  }
  if (tid >= 64) return;
  const int n_step = tile.step1 - tile.step0;
  const apc_score_step r = steps[tile.step0 + (tid < n_step ? tid : 0)];
  const bool is_edge = tid < n_step && (r.flags & APC_STEP_EDGE), is_node = tid < n_step && (r.flags & APC_STEP_FIRST);
  const uint64_t edges = __ballot(is_edge), nodes = __ballot(is_node);
  const uint64_t below = (1ull << tid) - 1ull;
  const uint32_t buffer = (uint32_t)(t & 1) * (kImageBytes / 8);  // in doubles, as what follows
  const uint32_t body_at = buffer + kHeadBytes / 8, terms = body_at + (uint32_t)r.pa;
  const uint32_t zero = buffer + (kHeadAt + (uint32_t)offsetof(Head, zero)) / 8, zero_row = kRows * (uint32_t)row_bytes;
  const int n_edge = (__popcll(edges) + kUnroll - 1) / kUnroll * kUnroll;
  const int n_node = (__popcll(nodes) + kUnroll - 1) / kUnroll * kUnroll;
  EdgeWords* const to_edge = reinterpret_cast<EdgeWords*>(image);
  NodeWords* const to_node = reinterpret_cast<NodeWords*>(image + kNodesAt);
  if (tid >= __popcll(edges) && tid < n_edge) to_edge[tid] = EdgeWords{zero, zero_row | zero_row << 16, zero | kEdgeOdd, -1};
  if (tid >= __popcll(nodes) && tid < n_node) to_node[tid] = NodeWords{zero_row | zero << 16, -1};
  if (is_edge) {
    EdgeWords w;
    w.matrix = (body_at + (uint32_t)r.mat) | (uint32_t)r.ssrc << 19;
    w.choices = (uint32_t)r.row_node * row_bytes | (r.row_src < 0 ? zero_row : (uint32_t)r.row_src * row_bytes) << 16;
    w.terms = terms | (r.src_node >= 0 ? kEdgeSource : 0u) | (r.flags & APC_STEP_TRANSITION ? kEdgeTransition : 0u);
    w.mult = p.node_multiplier[r.node];
    if ((w.terms >> 17) != (kEdgeSource | kEdgeTransition) >> 17 || w.mult != 1) w.terms |= kEdgeOdd;
    to_edge[__popcll(edges & below)] = w;
  }
  if (is_node) to_node[__popcll(nodes & below)] = NodeWords{(uint32_t)r.row_node * row_bytes | terms << 16, r.nargs};
  if (tid < kRows) {
    const int v = tile.row[tid];
    RowWords w;
    w.w[0] = fold16(node_key(node_gid ? node_gid[v] : v));
    w.w[1] = (uint32_t)p.node_nstrat[v];
    reinterpret_cast<RowWords*>(image + kRowsAt)[tid] = w;
  }
  Head* const head = reinterpret_cast<Head*>(image + kHeadAt);
  const int t1 = min(t + 1, n_tile - 1), t2 = min(t + 2, n_tile - 1);
  if (tid < kRows) {
    head->row[0][tid] = tiles[t1].row[tid];
    head->row[1][tid] = tiles[t2].row[tid];
  }
  if (t == 0) {  // and how to begin, behind the images
    Head* const first = reinterpret_cast<Head*>(images + (size_t)n_tile * kImageBytes);
    if (tid < kRows) first->row[0][tid] = tile.row[tid];
    if (tid == 0) first->next_chunks = (kHeadBytes + image_doubles(tile, units) * 8 + 1023) / 1024;
  }
  if (tid == 0) {
    head->n_edge = n_edge;
    head->n_node = n_node;
    head->zero = 0.0;
    head->n_row = tile.n_row;
    head->next_chunks = (kHeadBytes + image_doubles(tiles[t1], units) * 8 + 1023) / 1024;
    head->any_edge = tiles[0].any_edge;
  }
}

// How explicit choices get into LDS: 16 or 4 bytes a lane by loads that write LDS, as the rows' alignment allows,
// or (2) through registers.
enum { kDrawn = 0, kRows16 = 16, kRows4 = 4, kRows2 = 2 };

template <int kGroups> struct Groups { static constexpr int value = kGroups; };

// kAhead: tiles by which the rows of choices are requested ahead (their buffers: kAhead + 1)
template <int kFrom, int kAhead>
__global__ void __launch_bounds__(1024)
score_images_walk_kernel(const char* __restrict__ images, int n_tile, const uint16_t* __restrict__ assign, int64_t stride,
                         int64_t row_len, uint64_t seed, int64_t first, int64_t n_assign, int clamp_inf,
                         const double* __restrict__ init, double* __restrict__ out) {
  extern __shared__ __align__(16) char s_mem[];  // two images, then the rows of choices [kAhead + 1][kRowSlots][lanes]
  const int n_lane = blockDim.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), n_wave = n_lane >> 6;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)s_mem;
  const uint32_t row_bytes = (uint32_t)n_lane * 2u, rows_bytes = row_bytes * kRowSlots;
  const int64_t a0 = (int64_t)blockIdx.x * n_lane;
  const int64_t a_raw = a0 + tid;
  const int64_t a = a_raw < n_assign ? a_raw : n_assign - 1;  // lanes past the end repeat the last one and store nothing
  uint16_t* const my_rows = reinterpret_cast<uint16_t*>(s_mem + 2 * kImageBytes) + tid;
  double t_compute = 0.0, t_comm = 0.0, obj = 0.0;
  uint32_t n_trans = 0, n_forbidden = 0;
  if (init) {
    const double* r = init + a * 6;
    t_compute = r[1]; t_comm = r[2]; obj = r[4];
  }
  // the loads of init end here: the compiler would wait for them where the sums are first added to, in the
  // loop, and with that for every copy under way
  asm volatile("" : "+v"(t_compute), "+v"(t_comm), "+v"(obj));
  const uint32_t h0 = fold16(assignment_hash(seed, first + a));
  for (int b = 0; b <= kAhead; ++b) my_rows[(b * kRowSlots + kRows) * n_lane] = 0;
  auto issue_image = [&](int t, int chunks) {  // into buffer t & 1; nothing waits here
    const char* const from = images + (size_t)t * kImageBytes + lane * 16;
    const uint32_t to = lds0 + (uint32_t)(t & 1) * kImageBytes;
    const int share = (chunks + n_wave - 1) / n_wave;
    int c = wave * share;
    const int end = min(c + share, chunks);
    for (; c + 4 <= end; c += 4) load16x4_lds(from + c * 1024, to + (uint32_t)c * 1024u);
    for (; c < end; ++c) load16_lds(from + c * 1024, to + (uint32_t)c * 1024u);
  };
  // The rows of choices of a tile into their buffer: always kRows of them (a tile's list repeats a node in unused
  // places), so that every wavefront knows how many loads it has under way.
  auto issue_rows = [&](int b, int32_t my_node) {  // my_node: lane i holds the i-th node
    const uint32_t to = lds0 + 2 * kImageBytes + (uint32_t)b * rows_bytes;
    if (kFrom == kRows16) {
      const int segments = (n_lane + 511) >> 9;
      for (int i = wave; i < kRows * segments; i += n_wave) {
        const int r = segments == 1 ? i : i >> 1, seg = segments == 1 ? 0 : i & 1;
        const int v = __builtin_amdgcn_readlane(my_node, r);
        const int at = seg * 512 + lane * 8;
        const int64_t from = min(a0 + at, row_len - 8);  // lanes past the end read the last ones again
        if (at < n_lane) load16_lds(assign + (size_t)v * stride + from, to + (uint32_t)r * row_bytes + (uint32_t)seg * 1024u);
      }
    } else if (kFrom == kRows4) {
      const int segments = n_lane >> 7;
      for (int i = wave; i < kRows * segments; i += n_wave) {
        const int r = i & (kRows - 1), seg = i >> 4;
        const int v = __builtin_amdgcn_readlane(my_node, r);
        const int64_t from = min(a0 + seg * 128 + lane * 2, row_len - 2);
        load4_lds(assign + (size_t)v * stride + from, to + (uint32_t)r * row_bytes + (uint32_t)seg * 256u);
      }
    }
  };
  uint16_t held[kFrom == kRows2 ? kRows : 1];
  auto request_rows = [&](int32_t my_node) {
    if (kFrom != kRows2) return;
#pragma unroll
    for (int r = 0; r < kRows; ++r) held[r] = assign[(size_t)__builtin_amdgcn_readlane(my_node, r) * stride + a];
  };
  auto keep_rows = [&](int b) {
    if (kFrom != kRows2) return;
#pragma unroll
    for (int r = 0; r < kRows; ++r) my_rows[(b * kRowSlots + r) * n_lane] = held[r];
  };
  // loads of rows a wavefront has under way when the image in front of them has to be there
  const int n_rows16 = (kRows * ((n_lane + 511) >> 9) - wave + n_wave - 1) / n_wave;
  {
    const Head* const h = reinterpret_cast<const Head*>(images + kHeadAt);
    // the first tile's own rows and size: found through a head in front of the images
    const Head* const h0 = reinterpret_cast<const Head*>(images + (size_t)n_tile * kImageBytes);
    issue_image(0, h0->next_chunks);
    issue_rows(0, h0->row[0][lane & (kRows - 1)]);
    request_rows(h0->row[0][lane & (kRows - 1)]);
    keep_rows(0);
    if (kAhead == 2) issue_rows(1, h->row[0][lane & (kRows - 1)]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  int b = 0;  // buffer of this tile's rows
  for (int t = 0; t < n_tile; ++t) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // everyone's copies have arrived
    const char* const img = s_mem + (t & 1) * kImageBytes;
    const Head* const head = reinterpret_cast<const Head*>(img + kHeadAt);
    const int next_b = b == kAhead ? 0 : b + 1;
    if (t + 1 < n_tile) issue_image(t + 1, __builtin_amdgcn_readfirstlane(head->next_chunks));
    if (kAhead == 1 && t + 1 < n_tile) {
      issue_rows(next_b, head->row[0][lane & (kRows - 1)]);
      request_rows(head->row[0][lane & (kRows - 1)]);
    }
    if (kAhead == 2 && t + 2 < n_tile) issue_rows(next_b == kAhead ? 0 : next_b + 1, head->row[1][lane & (kRows - 1)]);
    const int n_edge = __builtin_amdgcn_readfirstlane(head->n_edge), n_node = __builtin_amdgcn_readfirstlane(head->n_node);
    union { u32x4_t raw; EdgeWords w; } e;
    e.raw = reinterpret_cast<const u32x4_t*>(img)[lane];
    const NodeWords node = reinterpret_cast<const NodeWords*>(img + kNodesAt)[lane];
    auto word = [&](uint32_t mine, int s) -> uint32_t { return (uint32_t)__builtin_amdgcn_readlane((int)mine, s); };
    uint16_t* const rows = my_rows + b * kRowSlots * n_lane;
    if (kFrom == kDrawn) {
      const int n_row = __builtin_amdgcn_readfirstlane(head->n_row);
      const u32x2_t row = reinterpret_cast<const u32x2_t*>(img + kRowsAt)[lane & (kRows - 1)];
      for (int r0 = 0; r0 < n_row; r0 += kUnroll) {  // past n_row: nodes drawn again, never read
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)  // plain_draw by the node's key
          rows[(r0 + u) * n_lane] = (uint16_t)folded_draw(h0, word(row[0], r0 + u), word(row[1], r0 + u));
      }
    }
    const uint32_t at_rows = (uint32_t)(uintptr_t)(lds_ptr_t)rows;
    auto choice = [&](uint32_t at) -> uint32_t { return *(lds_u16_ptr_t)(uintptr_t)(at_rows + at); };
    auto load = [&](uint32_t at) -> double { return *(lds_f64_ptr_t)(uintptr_t)at; };
    const uint64_t m_odd = __ballot(e.w.terms & kEdgeOdd);  // beyond the edges: anything, not read
    uint32_t counts = 0;  // transitions and, from bit 16, forbidden entries of this tile
    auto edges = [&](int s0, auto groups) {
      constexpr int kN = decltype(groups)::value * kUnroll;
      // in three parts, so that the compiler asks for everything of a part before it waits for any of it
      uint32_t o[kN], j[kN], matrix[kN], terms[kN];
#pragma unroll
      for (int u = 0; u < kN; ++u) {
        const uint32_t choices = word(e.w.choices, s0 + u);
        o[u] = choice(choices & 0xFFFFu);
        j[u] = choice(choices >> 16);
        matrix[u] = word(e.w.matrix, s0 + u);
        terms[u] = word(e.w.terms, s0 + u) & 0xFFFFu;
      }
      __builtin_amdgcn_sched_barrier(0);
      double raw[kN], c[kN];
#pragma unroll
      for (int u = 0; u < kN; ++u) {
        uint32_t at = (j[u] + (matrix[u] & 0xFFFFu)) << 3;
        asm("" : "+v"(at));  // one multiply-add from here
        raw[u] = load(__umul24(o[u], matrix[u] >> 16) + at);
        c[u] = load((o[u] + terms[u]) << 3);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < kN; g += kUnroll) {
        // what the build makes of a matrix element, added up
        bool adds[kUnroll];
#pragma unroll
        for (int u = g; u < g + kUnroll; ++u) {
          const uint32_t hi = (uint32_t)((uint64_t)__double_as_longlong(raw[u]) >> 32);
          c[u] = (fabs(raw[u]) + c[u]) +
                 __longlong_as_double((long long)((uint64_t)((uint32_t)((int32_t)hi >> 31) & 0x3FF00000u) << 32));
          const bool finite = __builtin_amdgcn_class(c[u], kFinite);
          c[u] = finite || !clamp_inf ? c[u] : 10000.0;
          counts += (hi >> 31) + (finite ? 0u : 0x10000u);
          adds[u - g] = __builtin_amdgcn_class(raw[u], kFinite);
        }
        if (m_odd >> (s0 + g) & ((1ull << kUnroll) - 1)) {
#pragma unroll
          for (int u = g; u < g + kUnroll; ++u) {
            const uint32_t flags = word(e.w.terms, s0 + u);
            c[u] *= (double)(int)word((uint32_t)e.w.mult, s0 + u);
            if (!(flags & kEdgeSource)) adds[u - g] = false;
            if (!(flags & kEdgeTransition)) counts -= (uint32_t)((uint64_t)__double_as_longlong(raw[u]) >> 63);
          }
        }
#pragma unroll
        for (int u = g; u < g + kUnroll; ++u) {
          const double more = t_comm + fabs(raw[u]);
          t_comm = adds[u - g] ? more : t_comm;
          obj += c[u];
        }
      }
    };
    auto nodes = [&](int s0, auto groups) {
      constexpr int kN = decltype(groups)::value * kUnroll;
      uint32_t o[kN], terms[kN];
#pragma unroll
      for (int u = 0; u < kN; ++u) {
        const uint32_t at = word(node.at, s0 + u);
        o[u] = choice(at & 0xFFFFu);
        terms[u] = at >> 16;
      }
      __builtin_amdgcn_sched_barrier(0);
      double pa[kN];
#pragma unroll
      for (int u = 0; u < kN; ++u) pa[u] = load((o[u] + terms[u]) << 3);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < kN; ++u) t_compute += pa[u] * (double)(int)word((uint32_t)node.nargs, s0 + u);
    };
    int s = 0;
    for (; s + 2 * kUnroll <= n_edge; s += 2 * kUnroll) edges(s, Groups<2>());
    if (s < n_edge) edges(s, Groups<1>());
    for (s = 0; s + 2 * kUnroll <= n_node; s += 2 * kUnroll) nodes(s, Groups<2>());
    if (s < n_node) nodes(s, Groups<1>());
    n_trans += counts & 0xFFFFu;
    n_forbidden += counts >> 16;
    b = next_b;
    if (kAhead == 1) keep_rows(b);
    // this wavefront's copies of the next tile have arrived (loads complete in order: the rows of the tile
    // behind it may still be under way)
    if (kAhead == 2 && t + 2 < n_tile) {
      const int n = kFrom == kRows4 ? 8 : n_rows16;
      if (n >= 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      else if (n >= 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else if (n >= 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
  }
  if (a_raw >= n_assign) return;
  const Head* const h = reinterpret_cast<const Head*>(images + kHeadAt);
  const double trans = add_ones(init ? init[a * 6 + 3] : 0.0, n_trans);
  double forbidden = init ? init[a * 6 + 5] : 0.0;
  if (h->any_edge) forbidden += 0.0;  // a walk adds 0.0 or 1.0 per edge: a carried -0.0 loses its sign
  forbidden = add_ones(forbidden, n_forbidden);
  double* r = out + a * 6;
  r[0] = (t_compute + t_comm) + trans;
  r[1] = t_compute;
  r[2] = t_comm;
  r[3] = trans;
  r[4] = obj;
  r[5] = forbidden;
}

template <int kFrom, int kAhead>
int launch_walk(const char* images, int n_tile, const uint16_t* assign, int64_t stride, int64_t row_len, uint64_t seed,
                int64_t first, int64_t n_assign, int clamp_inf, const double* init, double* out, int n_lane,
                hipStream_t stream) {
  const int lds = 2 * kImageBytes + (kAhead + 1) * kRowSlots * n_lane * 2;
  const void* const kernel = reinterpret_cast<const void*>(score_images_walk_kernel<kFrom, kAhead>);
  if (int rc = check_lds_from_0(kernel, "score_images_walk_kernel")) return rc;
  hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return fail(APC_ERR_LAUNCH, "hipFuncSetAttribute(score_images_walk_kernel): %s", hipGetErrorString(e));
  hipLaunchKernelGGL((score_images_walk_kernel<kFrom, kAhead>), dim3((unsigned)((n_assign + n_lane - 1) / n_lane)),
                     dim3(n_lane), lds, stream, images, n_tile, assign, stride, row_len, seed, first, n_assign, clamp_inf,
                     init, out);
  return check_launch("score_images_walk_kernel");
}

}  // namespace

extern "C" {

int apc_score_images(const apc_problem* p, const double* per_arg, const double* table, const apc_score_step* steps,
                     int32_t n_step, const apc_score_tile* tiles, int32_t n_tile, const apc_score_unit* units,
                     void* scratch, const uint16_t* assign, uint64_t seed, int64_t first, int64_t n_assign,
                     const int32_t* node_gid, int32_t clamp_inf, const double* init, double* out, void* stream) {
  if (int rc = validate_problem(p)) return rc;
  if (n_assign <= 0) return 0;
  if (!per_arg || !steps || !tiles || !units || !scratch || !out || !p->node_multiplier || n_step <= 0 || n_tile <= 0 ||
      (p->table_size > 0 && !table))
    return fail(APC_ERR_INVALID, "apc_score_images: null argument or an empty layout%s");
  // One workgroup per CU, of as many lanes as the batch has for it; batches beyond 1 024 lanes in equal parts.
  const int64_t parts = (n_assign + 256 * 1024 - 1) / (256 * 1024);
  const int64_t part = ((n_assign + parts - 1) / parts + 1023) / 1024 * 1024;
  const int n_lane = (int)std::max<int64_t>(128, ((std::min(part, n_assign) + 255) / 256 + 127) / 128 * 128);
  char* const images = static_cast<char*>(scratch);
  hipLaunchKernelGGL(score_images_kernel, dim3((unsigned)n_tile), dim3(kBlock), 0, (hipStream_t)stream, *p, per_arg, table,
                     steps, tiles, n_tile, units, node_gid, n_lane * 2, images);
  if (int rc = check_launch("score_images_kernel")) return rc;
  for (int64_t a0 = 0; a0 < n_assign; a0 += part) {
    const int64_t n = std::min(part, n_assign - a0);
    const double* in = init ? init + a0 * 6 : nullptr;
    const uint16_t* rows = assign ? assign + a0 : nullptr;
    const uintptr_t at = (uintptr_t)rows;
#define APC_WALK(FROM, AHEAD)                                                                                       \
  launch_walk<FROM, AHEAD>(images, n_tile, rows, n_assign, n_assign - a0, seed, first + a0, n, (int)clamp_inf, in,  \
                           out + a0 * 6, n_lane, (hipStream_t)stream)
    int rc;
    const bool deep = n_lane <= 640;  // three buffers of rows fit
    if (!assign) rc = APC_WALK(kDrawn, 0);
    else if (at % 16 == 0 && n_assign % 8 == 0) rc = deep ? APC_WALK(kRows16, 2) : APC_WALK(kRows16, 1);
    else if (at % 4 == 0 && n_assign % 2 == 0) rc = deep ? APC_WALK(kRows4, 2) : APC_WALK(kRows4, 1);
    else rc = APC_WALK(kRows2, 1);
#undef APC_WALK
    if (rc) return rc;
  }
  return 0;
}

}  // extern "C"

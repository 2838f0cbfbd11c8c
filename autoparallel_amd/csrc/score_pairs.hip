// Scoring of the largest random batches on graphs with small blocks, from images of finished entries (gfx950), and its
// C ABI.
//
// From 2^18 assignments on the walks over matrices (score_tiles.hip, score_images.hip) are bound by instructions: an
// entry is formed from its matrix element, its node's term and a flag, tested, clamped and counted on every draw.  So the launch in front of the walk forms them: an image holds, per edge and (choice, producer's
// choice), the cost as it is added to the objective, multiplied and clamped, and the communication as it is added, 0
// where it is not.  Communication is never negative: its sign says whether a transition counts.  Costs are not either, but
// for negative multipliers or terms: their sign says whether the entry is forbidden, and the image of a tile with a
// negative one (or a NaN) says so and holds costs as they are, those that are forbidden or not finite as NaNs that name them
// (kBoxed).  A draw then is one 16-byte read, two additions and two counts.  Lanes take up to four assignments, whose
// choices of a row lie in one word; those a tile reads and no slot holds yet are drawn when it begins.
// Measured, MI355X, Llama-3-8B graph (8 533 edges, 2 032 tiles): 2^20 assignments 10.4 -> 7.3 ms, 524 288 6.2 -> 4.9,
// 262 144 4.7 -> 3.7; the images (112 MB) take 40 us of that.  What bounds it: vector instructions, 22.6 a draw (77% of
// the cycles), 8 of them the hashes of the rows (2.3 ms); the LDS reads, 16 cycles with their conflicts, are 60%.  Rows kept
// in their slots from tile to tile and addresses by v_perm and v_dot2 instead of two bit fields and two multiply-adds: 9.95
// -> 7.3.  Not better: one edge at a time or four (7.45), twice the lanes with half the assignments (the same).
// Sums run in node order, then argument order, as in score_kernel: the same bits, as they start from 0.0 (a carried
// -0.0 would not survive the zeros added here).
#include <algorithm>
#include <exception>
#include <unordered_map>
#include <vector>

#include "apc_device.h"
#include "score_tiles.h"

namespace {

using namespace apc_tiles;

constexpr int kPairRows = APC_PAIR_TILE_ROWS;
constexpr int kSlots = kPairRows + 1;  // the last one: zeros, the choice of a missing producer
constexpr int kHeadBytes = 2048;       // of an image: edges, nodes, rows, Head
constexpr int kNodesAt = 1024, kRowsAt = 1536, kHeadAt = 1792;
constexpr int kImageBytes = APC_PAIR_IMAGE_BYTES;
constexpr uint32_t kBoxed = 0x7FFC0000u, kBoxForbidden = 4;  // high word of a NaN: this, kBox*
enum { kBoxClamped = 0, kBoxInf = 1, kBoxMinusInf = 2, kBoxNan = 3 };  // kBoxClamped: 10000.0 times the low word, kBoxNan: that is its high word
constexpr int kUnits = (kImageBytes - kHeadBytes) / 16;  // pairs, two terms each
static_assert(kUnits == APC_PAIR_TILE_UNITS && 2 * kImageBytes + kSlots * 4096 <= 160 * 1024 && kImageBytes % 1024 == 0, "an image");

struct EdgeWords { uint32_t at, row, choices; };  // its pairs in LDS, bytes; bytes of a row of them (bits 0-15) and
                                                  // of one; rows of the node's (bits 0-15) and the producer's choices, bytes
struct NodeWords { uint32_t terms, choice; };     // terms in LDS, row of its choice, bytes
struct RowWords { uint32_t key, nstrat; };        // what its draw starts from; strategies (bits 0-15), its row, bytes
struct Head { int32_t n_edge, n_node, n_row, next_chunks, boxed; };
static_assert(sizeof(EdgeWords) * kTileSteps <= kNodesAt && sizeof(NodeWords) * kTileSteps <= kRowsAt - kNodesAt &&
              sizeof(RowWords) * kPairRows <= kHeadAt - kRowsAt && sizeof(Head) + kHeadAt <= kHeadBytes, "an image's head");
typedef const __attribute__((address_space(3))) double* lds_f64_ptr_t;
typedef const __attribute__((address_space(3))) double2_t* lds_f64x2_ptr_t;
typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));

__global__ void __launch_bounds__(kBlock)
pair_images_kernel(apc_problem p, const double* __restrict__ per_arg, const double* __restrict__ table,
                   const apc_pair_step* __restrict__ steps, const apc_pair_tile* __restrict__ tiles, int n_tile,
                   const int32_t* __restrict__ node_gid, int clamp_inf, int row_bytes, char* __restrict__ images) {
  __shared__ int s_negative;
  const int t = blockIdx.x, tid = threadIdx.x;
  if (tid == 0) s_negative = 0;
  __syncthreads();
  const apc_pair_tile tile = tiles[t];
  char* const image = images + (size_t)t * kImageBytes;
  const int n_step = tile.step1 - tile.step0;
  bool boxed = false;
  for (;;) {
    for (int i = 0; i < n_step; ++i) {
      const apc_pair_step s = steps[tile.step0 + i];  // the same for every lane
      const int S = p.node_nstrat[s.node];
      if (s.terms >= 0) {
        const int nargs = p.node_nargs[s.node] > 1 ? p.node_nargs[s.node] : 1;
        double* const to = reinterpret_cast<double*>(image + kHeadBytes + s.terms * 16);
        for (int o = tid; o < S; o += kBlock) to[o] = per_arg[p.node_comp_off[s.node] + o] * (double)nargs;
      }
      if (s.edge < 0) continue;
      const apc_edge ed = p.edges[s.edge];
      const bool has_src = ed.src_node >= 0;
      const int n_col = has_src ? ed.ssrc : 1;
      const double mult = (double)p.node_multiplier[s.node];
      const bool counts = has_src && (ed.flags & APC_EDGE_SCORE_TRANSITION);
      double2_t* const to = reinterpret_cast<double2_t*>(image + kHeadBytes + s.pairs * 16);
      for (int x = tid; x < S * n_col; x += kBlock) {
        const int o = x / n_col, j = x - o * n_col;
        const double raw = ed.table_off >= 0 ? table[ed.table_off + (int64_t)o * ed.ssrc + j]
                                             : p.default_vals[ed.default_off + (int64_t)o * ed.ssrc + j];
        // as item_store forms an entry from its matrix element
        const bool trans = (uint64_t)__double_as_longlong(raw) >> 63;
        const double cm = fabs(raw);
        double c = (cm + per_arg[p.node_comp_off[s.node] + o]) + (trans ? 1.0 : 0.0);
        const bool finite = isfinite(c);
        if (clamp_inf && !finite) c = 10000.0;
        c *= mult;
        const double comm = has_src && isfinite(cm) ? cm : 0.0;
        if (!(c >= 0.0)) s_negative = 1;  // any lane
        double kept = finite ? fabs(c) : -fabs(c);
        if (boxed) {
          kept = c;
          if (!finite || !isfinite(c)) {
            const uint32_t kind = !finite && clamp_inf ? kBoxClamped : isnan(c) ? kBoxNan : c > 0.0 ? kBoxInf : kBoxMinusInf;
            const uint32_t hi = kBoxed | kind | (finite ? 0u : kBoxForbidden);
            const uint32_t lo = kind == kBoxNan ? (uint32_t)((uint64_t)__double_as_longlong(c) >> 32) : (uint32_t)p.node_multiplier[s.node];
            kept = __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
          }
        }
        to[x] = double2_t{kept, counts && trans ? -comm : comm};
      }
    }
    __syncthreads();
    if (boxed || !s_negative) break;  // the same for every lane
    boxed = true;                     // once more
  }
  if (tid >= 64) return;
  const uint32_t buffer = (uint32_t)(t & 1) * kImageBytes, zero_row = (uint32_t)kPairRows * row_bytes;
  const bool live = tid < n_step;
  const apc_pair_step s = steps[tile.step0 + (live ? tid : 0)];
  const bool is_edge = live && s.edge >= 0, is_node = live && s.terms >= 0;
  const uint64_t edges = __ballot(is_edge), nodes = __ballot(is_node), below = (1ull << tid) - 1ull;
  const int n_edge = __popcll(edges), n_node = __popcll(nodes);
  EdgeWords* const to_edge = reinterpret_cast<EdgeWords*>(image);
  NodeWords* const to_node = reinterpret_cast<NodeWords*>(image + kNodesAt);
  if (is_edge) {
    const apc_edge ed = p.edges[s.edge];
    to_edge[__popcll(edges & below)] =
        EdgeWords{buffer + kHeadBytes + (uint32_t)s.pairs * 16u, (uint32_t)(ed.src_node >= 0 ? ed.ssrc : 1) * 16u | 16u << 16,
                  (uint32_t)s.row_node * row_bytes | (s.row_src < 0 ? zero_row : (uint32_t)s.row_src * row_bytes) << 16};
  }
  if (is_node)
    to_node[__popcll(nodes & below)] = NodeWords{buffer + kHeadBytes + (uint32_t)s.terms * 16u, (uint32_t)s.row_node * row_bytes};
  if (tid < kPairRows) {
    const int v = tile.row[tid];
    reinterpret_cast<RowWords*>(image + kRowsAt)[tid] =
        RowWords{fold16(node_key(node_gid ? node_gid[v] : v)), (uint32_t)p.node_nstrat[v] | tile.slot[tid] * (uint32_t)row_bytes << 16};
  }
  if (tid == 0) {
    Head* const head = reinterpret_cast<Head*>(image + kHeadAt);
    const int t1 = min(t + 1, n_tile - 1);
    *head = Head{n_edge, n_node, tile.n_row, (kHeadBytes + tiles[t1].n_unit * 16 + 1023) / 1024, boxed};
    if (t == 0)  // how to begin, behind the images
      reinterpret_cast<Head*>(images + (size_t)n_tile * kImageBytes)->next_chunks = (kHeadBytes + tile.n_unit * 16 + 1023) / 1024;
  }
}

template <int kPer> struct Packed { typedef uint32_t type; };  // kPer choices of a lane, a byte each
template <> struct Packed<1> { typedef uint8_t type; };
template <> struct Packed<2> { typedef uint16_t type; };

template <int kN> struct Count { static constexpr int value = kN; };

template <int kPer>
__global__ void __launch_bounds__(1024)
score_pairs_kernel(const char* __restrict__ images, int n_tile, uint64_t seed, int64_t first, int64_t n_assign,
                   double* __restrict__ out) {
  extern __shared__ __align__(16) char s_mem[];  // two images, then kSlots rows of packed choices
  constexpr int kEdges = kPer == 1 ? 4 : 2;      // side by side
  typedef typename Packed<kPer>::type packed_t;
  typedef const __attribute__((address_space(3))) packed_t* row_ptr_t;
  typedef __attribute__((address_space(3))) packed_t* row_out_t;
  const int n_lane = blockDim.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), n_wave = n_lane >> 6;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)s_mem;
  const uint32_t row_bytes = (uint32_t)n_lane * kPer, my_rows = lds0 + 2 * kImageBytes + (uint32_t)tid * kPer;
  const int64_t lanes = (int64_t)gridDim.x * n_lane;
  const int64_t t_raw = (int64_t)blockIdx.x * n_lane + tid;
  const int64_t t_first = t_raw < n_assign ? t_raw : 0;
  // assignment k of this lane; a lane past the end repeats another one and stores nothing
  auto asg = [&](int k) -> int64_t {
    const int64_t ak = t_raw + k * lanes;
    return ak < n_assign ? ak : t_first;
  };
  double t_compute[kPer], t_comm[kPer], obj[kPer];
  uint32_t n_trans[kPer], n_forbidden[kPer], h0[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    t_compute[k] = t_comm[k] = obj[k] = 0.0;
    n_trans[k] = n_forbidden[k] = 0;
    h0[k] = fold16(assignment_hash(seed, first + asg(k)));
  }
  *(row_out_t)(uintptr_t)(my_rows + kPairRows * row_bytes) = 0;
  auto issue = [&](int t, int chunks) {  // into buffer t & 1; nothing waits here
    const char* const from = images + (size_t)t * kImageBytes + lane * 16;
    const uint32_t to = lds0 + (uint32_t)(t & 1) * kImageBytes;
    int c = wave * 4;
    for (; c + 4 <= chunks; c += 4 * n_wave) load16x4_lds(from + c * 1024, to + (uint32_t)c * 1024u);
    for (const int end = min(c + 4, chunks); c < end; ++c) load16_lds(from + c * 1024, to + (uint32_t)c * 1024u);
  };
  issue(0, reinterpret_cast<const Head*>(images + (size_t)n_tile * kImageBytes)->next_chunks);
  for (int t = 0; t < n_tile; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                // this wavefront's copies have arrived,
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // and everyone's
    const char* const img = s_mem + (t & 1) * kImageBytes;
    const Head* const head = reinterpret_cast<const Head*>(img + kHeadAt);
    if (t + 1 < n_tile) issue(t + 1, __builtin_amdgcn_readfirstlane(head->next_chunks));
    const int n_edge = __builtin_amdgcn_readfirstlane(head->n_edge), n_node = __builtin_amdgcn_readfirstlane(head->n_node);
    const int n_row = __builtin_amdgcn_readfirstlane(head->n_row), boxed = __builtin_amdgcn_readfirstlane(head->boxed);
    const EdgeWords edge = reinterpret_cast<const EdgeWords*>(img)[lane];
    const NodeWords node = reinterpret_cast<const NodeWords*>(img + kNodesAt)[lane];
    const RowWords row = reinterpret_cast<const RowWords*>(img + kRowsAt)[lane < kPairRows ? lane : 0];
    auto word = [&](uint32_t mine, int s) -> uint32_t { return (uint32_t)__builtin_amdgcn_readlane((int)mine, s); };
    for (int r = 0; r < n_row; ++r) {
      const uint32_t key = word(row.key, r), w = word(row.nstrat, r), nstrat = w & 0xFFFFu;
      uint32_t packed = 0;
#pragma unroll
      for (int k = 0; k < kPer; ++k) packed |= folded_draw(h0[k], key, nstrat) << (8 * k);  // plain_draw by the node's key
      *(row_out_t)(uintptr_t)(my_rows + (w >> 16)) = (packed_t)packed;
    }
    auto choices = [&](uint32_t at) -> uint32_t { return *(row_ptr_t)(uintptr_t)(my_rows + at); };
    auto byte = [&](uint32_t packed, int k) -> uint32_t { return kPer == 1 ? packed : (packed >> (8 * k)) & 0xFFu; };
    auto edges = [&](int s, auto unroll, auto is_boxed) {
      constexpr int kUnroll = decltype(unroll)::value;
      uint32_t o[kUnroll], j[kUnroll], from[kUnroll][kPer];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const uint32_t w = word(edge.choices, s + u);
        o[u] = choices(w & 0xFFFFu);
        j[u] = choices(w >> 16);
      }
      __builtin_amdgcn_sched_barrier(0);
      // the two choices side by side, then by a row's bytes and a pair's
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
#pragma unroll
        for (int k = 0; k < kPer; ++k)
          from[u][k] = __builtin_amdgcn_perm(j[u], o[u], 0x0C040C00u + (uint32_t)k * 0x00010001u);
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const uint32_t at = word(edge.at, s + u), row_len = word(edge.row, s + u);
#pragma unroll
        for (int k = 0; k < kPer; ++k)
          from[u][k] = __builtin_amdgcn_udot2(__builtin_bit_cast(u16x2_t, from[u][k]), __builtin_bit_cast(u16x2_t, row_len), at, false);
      }
      __builtin_amdgcn_sched_barrier(0);
      double2_t e[kUnroll][kPer];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) e[u][k] = *(lds_f64x2_ptr_t)(uintptr_t)from[u][k];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          double c = e[u][k].x;
          const uint64_t bits = (uint64_t)__double_as_longlong(c);
          if (decltype(is_boxed)::value) {
            const int kind = (int)(bits >> 32) & 3;
            const double named = kind == kBoxClamped ? 10000.0 * (double)(int32_t)(uint32_t)bits
                                 : kind == kBoxInf ? INFINITY : kind == kBoxMinusInf ? -INFINITY : __longlong_as_double((long long)(bits << 32));
            const bool box = isnan(c);
            c = box ? named : c;
            n_forbidden[k] += box ? (uint32_t)(bits >> 34) & 1u : 0u;
          } else {
            c = fabs(c);
            n_forbidden[k] += (uint32_t)(bits >> 63);
          }
          obj[k] += c;
          t_comm[k] += fabs(e[u][k].y);
          n_trans[k] += (uint32_t)((uint64_t)__double_as_longlong(e[u][k].y) >> 63);
        }
      }
    };
    int s = 0;
    if (boxed) {
      for (; s < n_edge; ++s) edges(s, Count<1>(), Count<1>());
    } else {
      for (; s + kEdges <= n_edge; s += kEdges) edges(s, Count<kEdges>(), Count<0>());
      if (kEdges > 2)
        for (; s + 2 <= n_edge; s += 2) edges(s, Count<2>(), Count<0>());
      if (s < n_edge) edges(s, Count<1>(), Count<0>());
    }
    auto nodes = [&](int s, auto unroll) {
      constexpr int kN = decltype(unroll)::value;
      uint32_t o[kN];
      double term[kN][kPer];
#pragma unroll
      for (int u = 0; u < kN; ++u) o[u] = choices(word(node.choice, s + u));
#pragma unroll
      for (int u = 0; u < kN; ++u) {
        const uint32_t at = word(node.terms, s + u);
#pragma unroll
        for (int k = 0; k < kPer; ++k) term[u][k] = *(lds_f64_ptr_t)(uintptr_t)(at + (byte(o[u], k) << 3));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < kN; ++u) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) t_compute[k] += term[u][k];
      }
    };
    for (s = 0; s + 2 <= n_node; s += 2) nodes(s, Count<2>());
    if (s < n_node) nodes(s, Count<1>());
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    if (t_raw + k * lanes >= n_assign) continue;
    const double t_trans = (double)n_trans[k];  // ones added up: exact
    double* r = out + asg(k) * 6;
    r[0] = (t_compute[k] + t_comm[k]) + t_trans;
    r[1] = t_compute[k];
    r[2] = t_comm[k];
    r[3] = t_trans;
    r[4] = obj[k];
    r[5] = (double)n_forbidden[k];
  }
}

}  // namespace

extern "C" {

int apc_pair_tiles(const apc_edge* edges, int32_t n_edge, int32_t n_node, const int32_t* node_edge_off,
                   const int32_t* node_nstrat, int32_t first_node, apc_pair_step* steps, int64_t max_step,
                   apc_pair_tile* tiles, int64_t max_tile, int32_t* n_step, int32_t* n_tile) {
  if (n_node < 0 || n_edge < 0 || first_node < 0 || first_node > n_node || !n_step || !n_tile || !steps || !tiles ||
      (n_node > first_node && (!node_edge_off || !node_nstrat)) || (n_edge > 0 && !edges))
    return fail(APC_ERR_INVALID, "apc_pair_tiles: null argument or first_node out of range%s");
  *n_step = *n_tile = 0;
  try {
    int64_t s = 0, t = -1;
    std::unordered_map<int32_t, int> row_of;
    auto row = [&](int32_t v) {  // nodes for now
      if (row_of.emplace(v, tiles[t].n_row).second) tiles[t].row[tiles[t].n_row++] = v;
    };
    for (int v = first_node; v < n_node; ++v) {
      const int e0 = node_edge_off[v], e1 = node_edge_off[v + 1];
      if (e0 < 0 || e0 > e1 || e1 > n_edge) return fail(APC_ERR_INVALID, "apc_pair_tiles: node_edge_off is no list of offsets%s");
      if (node_nstrat[v] < 1 || node_nstrat[v] > 256) return 0;  // a choice does not fit its byte
      for (int e = e0; e < (e1 > e0 ? e1 : e0 + 1); ++e) {
        const apc_edge* const ed = e < e1 ? edges + e : nullptr;
        int64_t pairs = 0;
        if (ed) {
          if ((ed->flags & APC_EDGE_COMPRESSED) || ed->sdst != node_nstrat[v] || ed->ssrc < 1 || ed->src_node >= v) return 0;
          if (ed->src_node >= 0 && ed->ssrc > 256) return 0;
          if (ed->table_off < 0 && ed->default_off < 0) return 0;
          pairs = (int64_t)ed->sdst * (ed->src_node >= 0 ? ed->ssrc : 1);
        }
        const int terms = e == e0 ? (node_nstrat[v] + 1) / 2 : 0;
        if (pairs + terms > kUnits) return 0;
        const int src = ed ? ed->src_node : -1;
        const int rows = !row_of.count(v) + (src >= 0 && !row_of.count(src));
        if (t < 0 || tiles[t].n_unit + pairs + terms > kUnits || tiles[t].n_row + rows > kPairRows || s - tiles[t].step0 >= kTileSteps) {
          if (t >= 0) tiles[t].step1 = (int32_t)s;
          if (++t >= max_tile) return fail(APC_ERR_INVALID, "apc_pair_tiles: max_tile is too small%s");
          memset(&tiles[t], 0, sizeof(tiles[t]));
          tiles[t].step0 = (int32_t)s;
          row_of.clear();
        }
        if (s >= max_step) return fail(APC_ERR_INVALID, "apc_pair_tiles: max_step is too small%s");
        apc_pair_step& r = steps[s++];
        memset(&r, 0, sizeof(r));
        r.node = v;
        r.edge = ed ? e : -1;
        r.pairs = tiles[t].n_unit;
        tiles[t].n_unit += (int32_t)pairs;
        r.terms = -1;
        if (e == e0) {
          r.terms = tiles[t].n_unit;
          tiles[t].n_unit += terms;
        }
        row(v);
        if (src >= 0) row(src);
        r.row_src = src;
      }
    }
    if (t < 0) return 0;
    tiles[t].step1 = (int32_t)s;
    // A row stays in its slot until one is needed for another node: that of the node read again last.  A draw costs about as
    // much as an edge: 0.91 instead of 1.37 of them per edge of the Llama-3-8B graph.
    std::vector<int32_t> next((size_t)(t + 1) * kPairRows), seen(n_node, (int32_t)t + 1);
    for (int64_t i = t; i >= 0; --i) {
      for (int r = 0; r < tiles[i].n_row; ++r) {
        next[i * kPairRows + r] = seen[tiles[i].row[r]];
        seen[tiles[i].row[r]] = (int32_t)i;
      }
    }
    std::fill(seen.begin(), seen.end(), -1);  // now the slot of a node
    int32_t held[kPairRows], until[kPairRows];
    for (int q = 0; q < kPairRows; ++q) {
      held[q] = -1;
      until[q] = (int32_t)t + 1;
    }
    for (int64_t i = 0; i <= t; ++i) {
      apc_pair_tile& tile = tiles[i];
      bool used[kPairRows] = {};
      for (int r = 0; r < tile.n_row; ++r) {
        const int q = seen[tile.row[r]];
        if (q < 0) continue;
        used[q] = true;
        until[q] = next[i * kPairRows + r];
      }
      int n_draw = 0;
      for (int r = 0; r < tile.n_row; ++r) {
        const int32_t v = tile.row[r];
        if (seen[v] >= 0) continue;
        int q = -1;
        for (int c = 0; c < kPairRows; ++c)
          if (!used[c] && (q < 0 || until[c] > until[q])) q = c;
        if (held[q] >= 0) seen[held[q]] = -1;
        seen[v] = q;
        held[q] = v;
        used[q] = true;
        until[q] = next[i * kPairRows + r];
        tile.slot[n_draw] = (uint8_t)q;
        tile.row[n_draw++] = v;
      }
      tile.n_row = n_draw;
      for (int r = n_draw; r < kPairRows; ++r) tile.row[r] = steps[tile.step0].node;  // a node that there is
      for (int32_t x = tile.step0; x < tile.step1; ++x) {
        steps[x].row_node = seen[steps[x].node];
        steps[x].row_src = steps[x].row_src < 0 ? -1 : seen[steps[x].row_src];
      }
    }
    *n_step = (int32_t)s;
    *n_tile = (int32_t)(t + 1);
  } catch (const std::exception&) {
    return fail(APC_ERR_INVALID, "apc_pair_tiles: out of host memory%s");
  }
  return 0;
}

int apc_score_pairs(const apc_problem* p, const double* per_arg, const double* table, const apc_pair_step* steps,
                    int32_t n_step, const apc_pair_tile* tiles, int32_t n_tile, void* scratch, uint64_t seed,
                    int64_t first, int64_t n_assign, const int32_t* node_gid, int32_t clamp_inf, double* out,
                    void* stream) {
  if (int rc = validate_problem(p)) return rc;
  if (n_assign <= 0) return 0;
  if (!per_arg || !steps || !tiles || !scratch || !out || !p->node_multiplier || n_step <= 0 || n_tile <= 0 ||
      (p->table_size > 0 && !table))
    return fail(APC_ERR_INVALID, "apc_score_pairs: null argument or an empty layout%s");
  // One workgroup per CU, of as many lanes as the batch has for it; from 1 024 on, two or four assignments per lane;
  // batches beyond in equal parts.
  const int64_t kMost = (int64_t)256 * 1024 * 4;
  const int64_t parts = (n_assign + kMost - 1) / kMost;
  const int64_t part = (n_assign + parts - 1) / parts;
  const int64_t share = (part + 255) / 256;
  const int per = share <= 1024 ? 1 : share <= 2048 ? 2 : 4;
  const int n_lane = (int)std::max<int64_t>(128, ((share + per - 1) / per + 63) / 64 * 64);
  char* const images = static_cast<char*>(scratch);
  hipLaunchKernelGGL(pair_images_kernel, dim3((unsigned)n_tile), dim3(kBlock), 0, (hipStream_t)stream, *p, per_arg, table,
                     steps, tiles, n_tile, node_gid, (int)clamp_inf, n_lane * per, images);
  if (int rc = check_launch("pair_images_kernel")) return rc;
  void (*const kernel)(const char*, int, uint64_t, int64_t, int64_t, double*) =
      per == 1 ? score_pairs_kernel<1> : per == 2 ? score_pairs_kernel<2> : score_pairs_kernel<4>;
  const int lds = 2 * kImageBytes + kSlots * n_lane * per;
  if (int rc = check_lds_from_0(reinterpret_cast<const void*>(kernel), "score_pairs_kernel")) return rc;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return fail(APC_ERR_LAUNCH, "hipFuncSetAttribute(score_pairs_kernel): %s", hipGetErrorString(e));
  for (int64_t a0 = 0; a0 < n_assign; a0 += part) {
    const int64_t n = std::min(part, n_assign - a0);
    const int64_t per_block = (int64_t)n_lane * per;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((n + per_block - 1) / per_block)), dim3(n_lane), lds, (hipStream_t)stream, images,
                       n_tile, seed, first + a0, n, out + a0 * 6);
    if (int rc = check_launch("score_pairs_kernel")) return rc;
  }
  return 0;
}

}  // extern "C"

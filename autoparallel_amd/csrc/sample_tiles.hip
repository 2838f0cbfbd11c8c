// Feasible draws (sample.hip says which) for graphs of at most 64 strategies a node, by tiles of nodes through LDS
// (gfx950), and the C ABI.
//
// A lane per assignment and one workgroup per CU walk the nodes in order.  A node's draw is a chain, choices of its
// producers -> their columns -> the draw; from memory a link of it is 1 us, and the walk in steps (sample_steps_kernel)
// can only share it among the nodes that are ready, two in a decoder.  Here every link is an LDS read: a tile of up to 32
// nodes and argument rows has its columns, packed, and a few words per node and row there, copied in one piece while
// the tile before is walked; choices of the last 64 nodes stay in LDS, and those of older producers are requested
// from the matrix a tile ahead.  What is left of a node's chain is its draw: the choice of the node in front is taken
// from a register, and everything else that a node reads is read while that one is drawn.
// Measured, MI355X, in steps and by tiles: Llama-3-8B graph, 131 072 assignments 5.07 -> 2.42 ms, 100 2.97 -> 2.02, 524 288
// (a lane each) 21.2 -> 7.2; 12-layer GPT-2 graph, 131 072 1.56 -> 0.86.  What bounds it: below 65 536 that chain (0.33 us
// a node with a wavefront a SIMD: 65 dependent instructions and an LDS read), at 2^18 instructions (0.59 us for four
// wavefronts, 90 vector ones a node).
// Not better: the choice of the node in front through LDS, too (2.95 ms for 131 072), the position of the set bit by
// compares (2.18 for 100), always among 64 bits (4.39 against 3.65 for 262 144).
#include <algorithm>
#include <exception>
#include <unordered_map>
#include <vector>

#include "apc_device.h"
#include "score_tiles.h"

namespace {

using namespace apc_tiles;

constexpr int kNodes = APC_SAMPLE_TILE_NODES;  // and argument rows, of a tile
constexpr int kFar = APC_SAMPLE_TILE_FAR;
constexpr int kRing = 2 * kNodes;
constexpr int kSlots = kRing + 2 * kFar + 1;  // rows of choices in LDS, a byte per lane: the ring, older producers' of
                                              // this tile and of the next one, zeros
constexpr int kMaxStrategies = 64;
constexpr int kImageBytes = APC_SAMPLE_IMAGE_BYTES;
constexpr int kAllAt = 2560, kColumnsAt = 3072;  // kAllAt: columns that allow everything, one for every choice

// An argument row: its columns (their place in LDS), its producer's choices (bytes of a row per lane)
struct ArgWords { uint32_t columns, choices; };
// Node i of a tile.  One argument row whose producer is the node in front is apart: its choice is in a register, and
// all else is read while that one is drawn.  Two more rows are named, further ones are in the list of rows; the second
// name goes to the node's own word of allowed strategies (as a column of a choice 0) where that is not implied:
// without a second row, or with a filter.
struct NodeWords {
  uint32_t key_rank, before;  // what its draw starts from; columns of the row of the node in front
  ArgWords arg[2];
  uint32_t key_plain, nstrat;
  uint64_t allowed;           // its strategies, those its filter leaves
  uint32_t n_more, more0;
  uint32_t reserved[4];
};
struct Head {
  int32_t n_node, next_chunks, n_far, node0, seq0;  // n_far: of the next tile
  int32_t far[kFar];
};
constexpr int kArgsAt = 2048, kHeadAt = 2304;
static_assert(sizeof(NodeWords) * kNodes == kArgsAt && sizeof(ArgWords) * kNodes == kHeadAt - kArgsAt &&
              sizeof(Head) + kHeadAt <= kAllAt && kMaxStrategies * 8 == kColumnsAt - kAllAt && kColumnsAt + kNodes * kMaxStrategies * 8 <= kImageBytes &&
              kImageBytes % 1024 == 0 && sizeof(apc_sample_tile) == 160, "an image");
typedef const __attribute__((address_space(3))) uint8_t* lds_u8_ptr_t;
typedef __attribute__((address_space(3))) uint8_t* lds_u8_out_t;
typedef const __attribute__((address_space(3))) uint64_t* lds_u64_ptr_t;

__device__ __forceinline__ int columns_of(const apc_problem& p, int e) {
  return p.edges[e].src_node >= 0 ? p.edges[e].ssrc : 1;
}

__global__ void __launch_bounds__(kBlock)
sample_images_kernel(apc_problem p, const uint64_t* __restrict__ colbits, const int64_t* __restrict__ col_off,
                     const apc_sample_tile* __restrict__ tiles, int n_tile, const uint8_t* __restrict__ arg_row,
                     const int32_t* __restrict__ node_gid, const uint64_t* __restrict__ row_filter,
                     const int64_t* __restrict__ filter_off, int row_bytes, char* __restrict__ images) {
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const apc_sample_tile tile = tiles[t];
  char* const image = images + (size_t)t * kImageBytes;
  auto bytes_of = [&](int tt) -> int {  // every wavefront by itself
    const int e = tiles[tt].edge0 + lane;
    int n = lane < tiles[tt].n_edge ? columns_of(p, e) : 0;
    for (int d = 32; d >= 1; d >>= 1) n += __shfl_xor(n, d);
    return kColumnsAt + n * 8;
  };
  // columns one behind the other; where an argument row's begin: a sum over the rows before
  int n = lane < tile.n_edge ? columns_of(p, tile.edge0 + lane) : 0, begin = n;
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(begin, d);
    if (lane >= d) begin += up;
  }
  begin -= n;
  uint64_t* const columns = reinterpret_cast<uint64_t*>(image + kColumnsAt);
  for (int i = tid >> 6; i < tile.n_edge; i += kBlock / 64) {
    const int count = __shfl(n, i), to = __shfl(begin, i);
    const uint64_t* __restrict__ from = colbits + col_off[tile.edge0 + i];
    if (lane < count) columns[to + lane] = from[2 * lane];  // a column is two words there, the second one unused
  }
  if (tid >= 64) return;
  const uint32_t buffer = (uint32_t)(t & 1) * kImageBytes, zero_row = (uint32_t)(kSlots - 1) * row_bytes;
  uint32_t my_choices = zero_row, my_columns = buffer + kColumnsAt + (uint32_t)begin * 8u;
  int my_src = -1;
  if (lane < tile.n_edge) {
    const int row = arg_row[tile.edge0 + lane];
    my_src = p.edges[tile.edge0 + lane].src_node;
    if (row != APC_SAMPLE_ROW_NONE) my_choices = (uint32_t)(row < kRing ? row : row + (t & 1 ? kFar : 0)) * row_bytes;
  }
  const bool is_node = lane < tile.n_node;
  const int v = tile.node0 + (is_node ? lane : 0);
  const int e0 = p.node_edge_off[v] - tile.edge0, n_arg = is_node ? p.node_edge_off[v + 1] - p.node_edge_off[v] : 0;
  int most = n_arg;
  for (int d = 32; d >= 1; d >>= 1) most = max(most, __shfl_xor(most, d));
  const uint32_t all_at = buffer + kAllAt;
  reinterpret_cast<uint64_t*>(image + kAllAt)[lane] = ~0ull;
  const bool filtered = is_node && filter_off && filter_off[v] >= 0;
  NodeWords w = {};
  w.before = all_at;
  w.arg[0] = ArgWords{all_at, zero_row};
  w.arg[1] = ArgWords{buffer + (uint32_t)(lane * sizeof(NodeWords) + offsetof(NodeWords, allowed)), zero_row};
  // two passes: how many rows are in the list, then where
  int more0 = 0;
  for (int pass = 0; pass < 2; ++pass) {
    int named = 0, more = 0;
    bool before = false;
    for (int q = 0; q < most; ++q) {
      const ArgWords arg = {(uint32_t)__shfl((int)my_columns, (e0 + q) & 63), (uint32_t)__shfl((int)my_choices, (e0 + q) & 63)};
      const int src = __shfl(my_src, (e0 + q) & 63);
      if (q >= n_arg) continue;
      const bool in_front = src == v - 1 && tile.seq0 + lane > 0;
      if (in_front && !before) {
        before = true;
        w.before = arg.columns;
      } else if (!in_front && named < (filtered ? 1 : 2)) {
        w.arg[named++] = arg;
      } else {
        if (pass == 1) reinterpret_cast<ArgWords*>(image + kArgsAt)[more0 + more] = arg;
        ++more;
      }
    }
    if (pass == 0) {
      more0 = more;
      for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(more0, d);
        if (lane >= d) more0 += up;
      }
      more0 -= more;
      w.n_more = (uint32_t)more;
      w.more0 = (uint32_t)more0;
    }
  }
  if (is_node) {
    const int S = p.node_nstrat[v];
    w.allowed = S >= 64 ? ~0ull : (1ull << S) - 1ull;
    if (filtered) w.allowed &= row_filter[filter_off[v]];
    const uint32_t key = node_key(node_gid ? node_gid[v] : v);
    w.nstrat = (uint32_t)S;
    w.key_rank = fold16(key ^ kRankSalt);
    w.key_plain = fold16(key);
    reinterpret_cast<NodeWords*>(image)[lane] = w;
  }
  Head* const head = reinterpret_cast<Head*>(image + kHeadAt);
  const int t1 = min(t + 1, n_tile - 1);
  const int next_chunks = (bytes_of(t1) + 1023) >> 10;
  if (lane < kFar) head->far[lane] = tiles[t1].far[lane];
  if (lane == 0) {
    head->n_node = tile.n_node;
    head->node0 = tile.node0;
    head->seq0 = tile.seq0;
    head->next_chunks = next_chunks;
    head->n_far = tiles[t1].n_far;
  }
  if (t == 0) {  // and how to begin, behind the images
    Head* const first = reinterpret_cast<Head*>(images + (size_t)n_tile * kImageBytes);
    const int chunks = (bytes_of(0) + 1023) >> 10;
    if (lane < kFar) first->far[lane] = tile.far[lane];
    if (lane == 0) {
      first->next_chunks = chunks;
      first->n_far = tile.n_far;
    }
  }
}

// Position of the r-th set bit of m (r < popcount(m)); kWide: beyond the low 32, too.  By masks instead of compares:
// what a compare writes can be used two instructions later only, and this is the longest link of a node's chain.
template <bool kWide>
__device__ __forceinline__ uint32_t nth_bit(uint64_t m, uint32_t r) {
  uint32_t x = (uint32_t)m, base = 0;
  auto take = [](uint32_t mask, uint32_t a, uint32_t b) -> uint32_t { return (mask & a) | (~mask & b); };
  if (kWide) {
    const uint32_t d = r - (uint32_t)__popc(x), low = (uint32_t)((int32_t)d >> 31);
    x = take(low, x, (uint32_t)(m >> 32));
    r = take(low, r, d);
    base = 32u & ~low;
  }
  uint32_t at = 0;
#pragma unroll
  for (int s = 16; s >= 1; s >>= 1) {
    const uint32_t d = r - (uint32_t)__popc(__builtin_amdgcn_ubfe(x, at, s)), low = (uint32_t)((int32_t)d >> 31);
    r = take(low, r, d);
    at = take(low, at, at + s);
  }
  return base + at;
}

template <bool kWide>
__global__ void __launch_bounds__(1024)
sample_tiles_kernel(const char* __restrict__ images, int n_tile, uint64_t seed, int64_t first, int64_t n_assign,
                    int64_t stride, uint16_t* __restrict__ assign, int32_t* __restrict__ n_fallback) {
  extern __shared__ __align__(16) char s_mem[];  // two images, then kSlots rows of choices
  const int n_lane = blockDim.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), n_wave = n_lane >> 6;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)s_mem;
  const int64_t a_raw = (int64_t)blockIdx.x * n_lane + tid;
  const bool mine = a_raw < n_assign;
  const uint32_t a = (uint32_t)(mine ? a_raw : n_assign - 1);  // lanes past the end repeat the last one
  const uint32_t my_rows = lds0 + 2 * kImageBytes + (uint32_t)tid;
  const uint32_t h0 = fold16(assignment_hash(seed, first + a));
  const uint32_t a2 = a * 2u;
  uint16_t* const my_assign = assign + a;
  uint32_t pick = 0;  // of the node in front
  int fallbacks = 0;
  *(lds_u8_out_t)(uintptr_t)(my_rows + (uint32_t)(kSlots - 1) * n_lane) = 0;
  auto issue_image = [&](int t, int chunks) {  // into buffer t & 1; nothing waits here
    const char* const from = images + (size_t)t * kImageBytes + lane * 16;
    const uint32_t to = lds0 + (uint32_t)(t & 1) * kImageBytes;
    for (int c = wave; c < chunks; c += n_wave) load16_lds(from + c * 1024, to + (uint32_t)c * 1024u);
  };
  // older producers' choices: in the matrix since before the tile in front of the one that reads them began (this
  // lane's own stores, so in order)
  uint32_t held[kFar];
  auto request = [&](int32_t my_node, int n) {  // my_node: lane i holds the i-th; eight at a time (the list ends in zeros)
#pragma unroll
    for (int i0 = 0; i0 < kFar; i0 += 8)
      if (i0 < n) {
#pragma unroll
        for (int i = i0; i < i0 + 8; ++i) held[i] = my_assign[(int64_t)__builtin_amdgcn_readlane(my_node, i) * stride];
      }
  };
  auto keep = [&](int t, int n) {
#pragma unroll
    for (int i0 = 0; i0 < kFar; i0 += 8)
      if (i0 < n) {
#pragma unroll
        for (int i = i0; i < i0 + 8; ++i)
          *(lds_u8_out_t)(uintptr_t)(my_rows + (uint32_t)(kRing + (t & 1) * kFar + i) * n_lane) = (uint8_t)held[i];
      }
  };
  {
    const Head* const h = reinterpret_cast<const Head*>(images + (size_t)n_tile * kImageBytes);
    issue_image(0, h->next_chunks);
    const int32_t node = h->far[lane < kFar ? lane : 0];
    request(node, h->n_far);
    keep(0, h->n_far);
  }
  for (int t = 0; t < n_tile; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                // this wavefront's copies have arrived,
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // and everyone's
    const char* const img = s_mem + (t & 1) * kImageBytes;
    const Head* const head = reinterpret_cast<const Head*>(img + kHeadAt);
    const int n_node = __builtin_amdgcn_readfirstlane(head->n_node);
    const int n_far = t + 1 < n_tile ? __builtin_amdgcn_readfirstlane(head->n_far) : 0;
    if (t + 1 < n_tile) issue_image(t + 1, __builtin_amdgcn_readfirstlane(head->next_chunks));
    request(head->far[lane < kFar ? lane : 0], n_far);
    union { u32x4_t raw[4]; NodeWords w; } node;
#pragma unroll
    for (int q = 0; q < 4; ++q) node.raw[q] = reinterpret_cast<const u32x4_t*>(img)[4 * (lane & (kNodes - 1)) + q];
    const ArgWords more = reinterpret_cast<const ArgWords*>(img + kArgsAt)[lane & (kNodes - 1)];
    uint16_t* row = assign + (int64_t)__builtin_amdgcn_readfirstlane(head->node0) * stride;
    auto word = [&](uint32_t w, int s) -> uint32_t { return (uint32_t)__builtin_amdgcn_readlane((int)w, s); };
    auto choice = [&](uint32_t choices) -> uint32_t { return *(lds_u8_ptr_t)(uintptr_t)(my_rows + choices); };
    auto column = [&](uint32_t columns, uint32_t j) -> uint64_t { return *(lds_u64_ptr_t)(uintptr_t)(columns + (j << 3)); };
    const uint64_t m_more = __ballot(lane < n_node && node.w.n_more > 0), m_wide = __ballot(lane < n_node && node.w.nstrat > 32);
    int seq = __builtin_amdgcn_readfirstlane(head->seq0);
    uint64_t rest = column(word(node.w.arg[0].columns, 0), choice(word(node.w.arg[0].choices, 0))) &
                    column(word(node.w.arg[1].columns, 0), choice(word(node.w.arg[1].choices, 0)));
    for (int i = 0; i < n_node; ++i, ++seq) {
      // of the next node (or this one again): producers' choices, all but the one that is drawn here
      const int i1 = i + 1 < n_node ? i + 1 : i;
      const uint32_t j0 = choice(word(node.w.arg[0].choices, i1)), j1 = choice(word(node.w.arg[1].choices, i1));
      const uint64_t c_before = column(word(node.w.before, i), pick);
      const uint32_t h = finalise32_folded(h0 ^ word(node.w.key_rank, i));  // rank_draw by the node's key
      uint64_t m = rest & c_before;
      if (m_more >> i & 1) {
        const uint32_t n_more = word(node.w.n_more, i);
        for (uint32_t q = 0; q < n_more; ++q) {
          const int at = (int)(word(node.w.more0, i) + q);
          m &= column(word(more.columns, at), choice(word(more.choices, at)));
        }
      }
      const uint64_t c0 = column(word(node.w.arg[0].columns, i1), j0), c1 = column(word(node.w.arg[1].columns, i1), j1);
      const uint32_t count = (uint32_t)__popcll(m);
      const uint32_t r = __umulhi(h, count);
      pick = kWide && (m_wide >> i & 1) ? nth_bit<true>(m, r) : nth_bit<false>(m, r);
      if (__ballot(count == 0)) {
        const uint32_t g = finalise32_folded(h0 ^ word(node.w.key_plain, i));  // plain_draw
        pick = count == 0 ? __umulhi(g, word(node.w.nstrat, i)) : pick;
        fallbacks += count == 0;
      }
      *(lds_u8_out_t)(uintptr_t)(my_rows + (uint32_t)((seq & (kRing - 1)) * n_lane)) = (uint8_t)pick;
      *reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(row) + a2) = (uint16_t)pick;  // lanes past the end: what the last one stores
      row += stride;
      rest = c0 & c1;
    }
    keep(t + 1, n_far);
  }
  if (mine) n_fallback[a] = fallbacks;
}

}  // namespace

extern "C" {

int apc_sample_tiles(int32_t n_node, int32_t n_edge, const int32_t* node_edge_off, const int32_t* edge_src,
                     const int32_t* edge_ssrc, const int32_t* node_nstrat, int32_t first_node, apc_sample_tile* tiles,
                     int32_t max_tile, uint8_t* arg_row, int32_t* n_tile) {
  if (n_node < 0 || n_edge < 0 || first_node < 0 || first_node > n_node || !n_tile ||
      (n_node > first_node && (!node_edge_off || !node_nstrat || !tiles)) ||
      (n_edge > 0 && (!edge_src || !edge_ssrc || !arg_row)))
    return fail(APC_ERR_INVALID, "apc_sample_tiles: null argument or first_node out of range%s");
  *n_tile = 0;
  try {
    int t = -1;
    std::unordered_map<int32_t, int> far;
    std::vector<int32_t> fresh, level((size_t)(n_node - first_node));  // nodes of the longest chain that ends in it
    int32_t depth = 0;
    for (int v = first_node; v < n_node; ++v) {
      const int e0 = node_edge_off[v], e1 = node_edge_off[v + 1];
      if (e0 < 0 || e0 > e1 || e1 > n_edge) return fail(APC_ERR_INVALID, "apc_sample_tiles: node_edge_off is no list of offsets%s");
      if (node_nstrat[v] < 1 || node_nstrat[v] > kMaxStrategies || e1 - e0 > kNodes) return 0;
      const int seq = v - first_node;
      fresh.clear();
      for (int e = e0; e < e1; ++e) {
        const int u = edge_src[e];
        if (u >= v || (u >= 0 && (edge_ssrc[e] < 1 || edge_ssrc[e] > kMaxStrategies))) return 0;
        if (u >= first_node) level[seq] = std::max(level[seq], level[u - first_node]);
        if (u >= 0 && (u < first_node || seq - (u - first_node) >= kRing) && !far.count(u) &&
            std::find(fresh.begin(), fresh.end(), u) == fresh.end())
          fresh.push_back(u);
      }
      if (t < 0 || tiles[t].n_node == kNodes || tiles[t].n_edge + (e1 - e0) > kNodes ||
          (int)(far.size() + fresh.size()) > kFar) {
        if (++t >= max_tile) return fail(APC_ERR_INVALID, "apc_sample_tiles: max_tile is too small%s");
        memset(&tiles[t], 0, sizeof(tiles[t]));
        tiles[t].node0 = v;
        tiles[t].edge0 = e0;
        tiles[t].seq0 = seq;
        far.clear();
      }
      apc_sample_tile& tile = tiles[t];
      for (int e = e0; e < e1; ++e) {
        const int u = edge_src[e];
        if (u < 0) {
          arg_row[e] = APC_SAMPLE_ROW_NONE;
        } else if (u >= first_node && seq - (u - first_node) < kRing) {
          arg_row[e] = (uint8_t)((u - first_node) & (kRing - 1));
        } else {
          auto found = far.find(u);
          if (found == far.end()) {
            if (tile.n_far == kFar) return 0;  // one node's own producers
            found = far.emplace(u, tile.n_far).first;
            tile.far[tile.n_far++] = u;
          }
          arg_row[e] = (uint8_t)(kRing + found->second);
        }
      }
      ++tile.n_node;
      tile.n_edge += e1 - e0;
      depth = std::max(depth, ++level[seq]);
    }
    if (t >= 0) tiles[0].depth = depth;
    *n_tile = t + 1;
  } catch (const std::exception&) {
    return fail(APC_ERR_INVALID, "apc_sample_tiles: out of host memory%s");
  }
  return 0;
}

int apc_sample_feasible_tiles(const apc_problem* p, const apc_sample_tile* tiles, int32_t n_tile, const uint8_t* arg_row,
                              const uint64_t* colbits, const int64_t* col_off, void* scratch, uint64_t seed, int64_t first,
                              int64_t n_assign, const int32_t* node_gid, const uint64_t* row_filter,
                              const int64_t* filter_off, int32_t wide, uint16_t* assign, int32_t* n_fallback, void* stream) {
  if (int rc = validate_problem(p)) return rc;
  if (n_assign <= 0) return 0;
  if (!assign || !n_fallback || !tiles || !arg_row || !scratch || n_tile <= 0 || (p->n_entry > 0 && (!colbits || !col_off)))
    return fail(APC_ERR_INVALID, "apc_sample_feasible_tiles: null argument or no tiles%s");
  if ((row_filter == nullptr) != (filter_off == nullptr))
    return fail(APC_ERR_INVALID, "apc_sample_feasible_tiles: row_filter and filter_off come together%s");
  // One workgroup per CU, of as many lanes as the batch has for it; batches beyond 1 024 lanes in equal parts.
  const int64_t parts = (n_assign + 256 * 1024 - 1) / (256 * 1024);
  const int64_t part = ((n_assign + parts - 1) / parts + 63) / 64 * 64;
  const int n_lane = (int)(((part + 255) / 256 + 63) / 64 * 64);
  char* const images = static_cast<char*>(scratch);
  hipLaunchKernelGGL(sample_images_kernel, dim3((unsigned)n_tile), dim3(kBlock), 0, (hipStream_t)stream, *p, colbits,
                     col_off, tiles, n_tile, arg_row, node_gid, row_filter, filter_off, n_lane, images);
  if (int rc = check_launch("sample_images_kernel")) return rc;
  const int lds = 2 * kImageBytes + kSlots * n_lane;
  void (*const kernel)(const char*, int, uint64_t, int64_t, int64_t, int64_t, uint16_t*, int32_t*) =
      wide ? sample_tiles_kernel<true> : sample_tiles_kernel<false>;
  if (int rc = check_lds_from_0(reinterpret_cast<const void*>(kernel), "sample_tiles_kernel")) return rc;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return fail(APC_ERR_LAUNCH, "hipFuncSetAttribute(sample_tiles_kernel): %s", hipGetErrorString(e));
  for (int64_t a0 = 0; a0 < n_assign; a0 += part) {
    const int64_t n = std::min(part, n_assign - a0);
    hipLaunchKernelGGL(kernel, dim3((unsigned)((n + n_lane - 1) / n_lane)), dim3(n_lane), lds,
                       (hipStream_t)stream, images, n_tile, seed, first + a0, n, n_assign, assign + a0, n_fallback + a0);
    if (int rc = check_launch("sample_tiles_kernel")) return rc;
  }
  return 0;
}

}  // extern "C"

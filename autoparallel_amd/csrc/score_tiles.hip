// Batch scoring of graphs with small blocks, from the block table through LDS (gfx950), and its
// C ABI.
//
// A draw of an entry is a gather inside a matrix of a few hundred to a few thousand doubles.
// From memory, cached or not, a CU serves about one lane of such a gather per cycle: the walk
// over 16-byte records takes 15.6 ms for 2^20 assignments of the Llama-3-8B graph (8 533 edges),
// of which that rate alone is 14.6.  So a workgroup, one per CU, takes the edges in tiles: runs of
// consecutive steps whose matrices and per-argument terms fit one of two LDS buffers, each
// distinct matrix once; the loads of the next tile (they write LDS directly) are issued before
// the lanes draw from this one, with one barrier per tile.  The layout of the tiles is made on
// the host, once per graph (apc_score_tiles).
// From 2^18 assignments on what is left is instructions, the hash of a random choice first of all
// (its four 32-bit multiplications run at a quarter of the rate): a choice is drawn once per node
// and kept for the next kRows - 1 nodes, packed to a byte per assignment, where three quarters of
// the edges find their producer's; explicit choices are read a tile ahead into the same place.
// Below, it is the chain of LDS reads of a step and the few wavefronts a CU has to hide it.
// Measured, from records and by tiles: 2^20 random assignments of that graph 15.4 -> 10.4 ms, of the 16-layer
// mixture-of-experts graph 8.4 -> 5.7 (random ones that carry no sums are faster from images of
// finished entries, score_pairs.hip, 7.3 ms for the first figure; explicit ones, and few random ones, from tile images,
// score_images.hip; they are walked here where there is no room for the images).  Not better: step records in LDS instead of scalar loads
// (11.8 for the first figure; eight readfirstlane a step).
// Sums run in node order, then argument order, as in score_kernel: the same bits.
#include <algorithm>
#include <exception>
#include <unordered_map>
#include <vector>

#include "apc_device.h"
#include "score_tiles.h"

namespace {

using namespace apc_tiles;

constexpr int kNoRow = 255;
constexpr int kMaxLanes = 1024;
constexpr int kUnitDoubles = 128;   // what one wavefront copies with one 16-byte load per lane
constexpr int kUnitSingles = 32;    // and with one 4-byte load per lane, where 16 bytes may not be aligned

typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));

// A step as the walk reads it, one scalar load:
//   [0] matrix (bits 0-12) and per-argument terms (13-25) in the tile's buffer, APC_STEP_* (26-28)
//   [1] producer's strategies (0-8), the node's (9-17)   [2] rows: the node's (0-7), the producer's (8-15)
//   [3] divisor of the node's terms   [4] multiplier   [5] whether it has a producer
struct StepWords { uint32_t lo[4], hi[4]; };
typedef uint32_t u32x8_t __attribute__((ext_vector_type(8)));
// The same unpacked, for random choices: there the walk is bound by instructions, unpacking
// included (2^20 assignments of the Llama-3-8B graph 10.5 ms against 11.1 with packed records);
// with explicit ones, which keep three records at a time, the scalar registers do not suffice.
struct StepFields {
  int32_t mat, pa, flags, ssrc, nstrat, row_node, row_src, has_src, nargs, mult;
  uint32_t key_node, key_src;
  int32_t reserved[4];
};
typedef uint32_t u32x16_t __attribute__((ext_vector_type(16)));
static_assert(sizeof(StepWords) == 32 && sizeof(StepFields) == 64 && sizeof(apc_score_step) == 64 && sizeof(apc_score_unit) == 16 &&
              sizeof(apc_score_tile) == 128, "layout");
static_assert(kTileDoubles <= 8192 && kRows < kNoRow, "a step's fields");

// The steps of a call, with the multipliers (they can be replaced between calls) and the ids
// the draws hash.
template <bool kRandom>
__global__ void __launch_bounds__(kBlock)
score_steps_kernel(apc_problem p, const apc_score_step* __restrict__ steps, int n_step,
                   const int32_t* __restrict__ node_gid, void* __restrict__ out) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= n_step) return;
  const apc_score_step r = steps[s];
  const uint32_t mult = (uint32_t)p.node_multiplier[r.node];
  if (kRandom) {
    StepFields f = {};
    f.mat = r.mat; f.pa = r.pa; f.flags = r.flags; f.ssrc = r.ssrc; f.nstrat = r.nstrat;
    f.row_node = r.row_node; f.row_src = r.row_src; f.has_src = r.src_node >= 0; f.nargs = r.nargs;
    f.mult = (int32_t)mult;
    f.key_node = node_key(node_gid ? node_gid[r.node] : r.node);
    if (r.src_node >= 0) f.key_src = node_key(node_gid ? node_gid[r.src_node] : r.src_node);
    static_cast<StepFields*>(out)[s] = f;
  } else {
    StepWords w = {};
    w.lo[0] = (uint32_t)r.mat | (uint32_t)r.pa << 13 | (uint32_t)r.flags << 26;
    w.lo[1] = (uint32_t)r.ssrc | (uint32_t)r.nstrat << 9;
    w.lo[2] = (uint32_t)r.row_node | (uint32_t)(r.row_src < 0 ? kNoRow : r.row_src) << 8;
    w.lo[3] = (uint32_t)r.nargs;
    w.hi[0] = mult;
    w.hi[1] = r.src_node >= 0;
    static_cast<StepWords*>(out)[s] = w;
  }
}

template <bool kRandom, int kPer>
__global__ void __launch_bounds__(kMaxLanes)
score_tiles_kernel(apc_problem p, const double* __restrict__ per_arg, const double* __restrict__ table,
                   const void* __restrict__ steps, const apc_score_tile* __restrict__ tiles, int n_tile,
                   const apc_score_unit* __restrict__ units, const uint16_t* __restrict__ assign, int64_t stride,
                   uint64_t seed, int64_t first, int64_t n_assign, int clamp_inf, const double* __restrict__ init,
                   double* __restrict__ out) {
  extern __shared__ __align__(16) double s_buf[];  // [2][kTileDoubles], then [kRows][lanes] packed choices
  uint32_t* const s_rows = reinterpret_cast<uint32_t*>(s_buf + 2 * kTileDoubles);
  const int n_lane = blockDim.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), n_wave = n_lane >> 6;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)s_buf;
  const int64_t lanes = (int64_t)gridDim.x * n_lane;
  const int64_t t_raw = (int64_t)blockIdx.x * n_lane + tid;
  const int64_t t_first = t_raw < n_assign ? t_raw : 0;
  // assignment k of this lane; a lane past the end repeats another one and stores nothing
  auto asg = [&](int k) -> int64_t {
    const int64_t ak = t_raw + k * lanes;
    return ak < n_assign ? ak : t_first;
  };
  double t_compute[kPer], t_comm[kPer], obj[kPer], pa[kPer];
  uint32_t n_trans[kPer], n_forbidden[kPer], h0[kPer], o[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    t_compute[k] = 0.0; t_comm[k] = 0.0; obj[k] = 0.0; pa[k] = 0.0; n_trans[k] = 0; n_forbidden[k] = 0; o[k] = 0;
    if (init) {
      const double* r = init + asg(k) * 6;
      t_compute[k] = r[1]; t_comm[k] = r[2]; obj[k] = r[4];
    }
    h0[k] = assignment_hash(seed, first + asg(k));
  }
  // the loads of init end here: the compiler would wait for them where the sums are first added to, in the
  // loop, and with that for every copy under way
#pragma unroll
  for (int k = 0; k < kPer; ++k) asm volatile("" : "+v"(t_compute[k]), "+v"(t_comm[k]), "+v"(obj[k]));
  auto draw = [&](int k, uint32_t key, uint32_t nstrat) -> uint32_t {  // plain_draw by the node's key
    return __umulhi(finalise32(h0[k] ^ key), nstrat);
  };
  // The copies of a tile are shared out by wavefronts; a lane holds the record of one of its
  // wavefront's copies, read a tile before the copies are issued.
  const uint64_t at_table = (uint64_t)(uintptr_t)table, to_per_arg = (uint64_t)(uintptr_t)per_arg - at_table,
                 to_default = (uint64_t)(uintptr_t)p.default_vals - at_table;
  struct Head { int step0, step1, unit0, unit1; };
  auto load_head = [&](int t) -> Head {
    union { i32x4_t raw; Head h; } u;
    u.raw = *reinterpret_cast<const i32x4_t*>(tiles + (t < n_tile ? t : n_tile - 1));
    return u.h;
  };
  auto load_unit = [&](const Head& h, int i) -> i32x4_t {  // the i-th of this wavefront's copies
    const int u = h.unit0 + wave + i * n_wave;
    return reinterpret_cast<const i32x4_t*>(units)[u < h.unit1 ? u : h.unit0];
  };
  auto issue = [&](const Head& h, int t, i32x4_t mine) {  // into tile t's buffer; nothing waits here
    const uint32_t base = lds0 + (uint32_t)(t & 1) * (kTileDoubles * 8);
    const int n = (h.unit1 - h.unit0 - wave + n_wave - 1) / n_wave;  // copies of this wavefront
    for (int i = 0; i < n; ++i) {
      if (i > 0 && (i & 63) == 0) mine = load_unit(h, i + lane);
      const uint32_t s_lo = (uint32_t)__builtin_amdgcn_readlane(mine[0], i & 63);
      const uint32_t s_hi = (uint32_t)__builtin_amdgcn_readlane(mine[1], i & 63);
      const uint32_t to = (uint32_t)__builtin_amdgcn_readlane(mine[2], i & 63);  // lds, n
      const int kind = __builtin_amdgcn_readlane(mine[3], i & 63);
      const int64_t src = (int64_t)((uint64_t)s_hi << 32 | s_lo);
      const uint32_t lds = base + (to & 0xFFFFu) * 8u;
      const int n_double = (int)(to >> 16);
      // the array by its distance from the table: a choice between what this lambda captured goes
      // through scratch memory, and the wait for that is one for the copies before
      const uint64_t from = at_table + (to_per_arg & (kind == 1 ? ~0ull : 0ull)) + (to_default & (kind == 2 ? ~0ull : 0ull)) +
                            (uint64_t)src * 8u;
      if (kind == 0) {
        if (2 * lane < n_double) load16_lds(reinterpret_cast<const double2_t*>(from) + lane, lds);
      } else {
        if (lane < 2 * n_double) load4_lds(reinterpret_cast<const uint32_t*>(from) + lane, lds);
      }
    }
  };
  // explicit choices of a tile (its list repeats a node in unused places): requested before the
  // tile in front of it is walked, put into the rows (a lane's own, so no barrier) behind it
  constexpr int kHeld = kRandom ? 1 : kRows;
  uint16_t ahead[kHeld][kPer];
  auto request = [&](int t) {
    if (kRandom) return;
#pragma unroll
    for (int r = 0; r < kHeld; ++r) {
      const uint16_t* const row = assign + (size_t)tiles[t].row[r] * stride;
#pragma unroll
      for (int k = 0; k < kPer; ++k) ahead[r][k] = row[asg(k)];
    }
  };
  auto keep_rows = [&]() {
    if (kRandom) return;
#pragma unroll
    for (int r = 0; r < kHeld; ++r) {
      uint32_t packed = 0;
#pragma unroll
      for (int k = 0; k < kPer; ++k) packed |= (uint32_t)(uint8_t)ahead[r][k] << (8 * k);
      s_rows[r * n_lane + tid] = packed;
    }
  };
  Head head = load_head(0), head1 = load_head(1);
  issue(head, 0, load_unit(head, lane));
  i32x4_t unit1 = load_unit(head1, lane);
  request(0);
  keep_rows();
  for (int t = 0; t < n_tile; ++t) {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // this wave's copies of tile t have arrived (vmcnt 0),
    __syncthreads();                     // and everyone's; and the tile before is done with its buffer
    if (t + 1 < n_tile) {
      issue(head1, t + 1, unit1);
      request(t + 1);
    }
    const Head head2 = load_head(t + 2);
    const double* const buf = s_buf + (t & 1) * kTileDoubles;
    // what the build makes of a matrix element, added up
    auto add_entries = [&](const double (&raw)[kPer], bool has_src, bool count_trans, int mult) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const uint64_t bits = (uint64_t)__double_as_longlong(raw[k]);
        const uint32_t trans = (uint32_t)(bits >> 63);
        const double one = __longlong_as_double((long long)((uint64_t)((0u - trans) & 0x3FF00000u) << 32));
        const double cm = fabs(raw[k]);
        double c = (cm + pa[k]) + one;
        const bool finite = isfinite(c);
        if (clamp_inf && !finite) c = 10000.0;
        obj[k] += mult == 1 ? c : c * (double)mult;
        n_forbidden[k] += finite ? 0u : 1u;
        if (has_src && isfinite(cm)) t_comm[k] += cm;
        n_trans[k] += count_trans ? trans : 0u;
      }
    };
    if (kRandom) {
      auto load_step = [&](int s) -> StepFields {
        union { u32x16_t raw; StepFields f; } u;
        u.raw = *reinterpret_cast<const u32x16_t*>(static_cast<const StepFields*>(steps) + s);
        return u.f;
      };
      StepFields next = load_step(head.step0);
      for (int s = head.step0; s < head.step1; ++s) {
        const StepFields st = next;
        next = load_step(s + 1 < head.step1 ? s + 1 : s);
        if (st.flags & APC_STEP_FIRST) {
          uint32_t packed = 0;
#pragma unroll
          for (int k = 0; k < kPer; ++k) {
            o[k] = draw(k, st.key_node, (uint32_t)st.nstrat);
            packed |= o[k] << (8 * k);
          }
          s_rows[st.row_node * n_lane + tid] = packed;
#pragma unroll
          for (int k = 0; k < kPer; ++k) pa[k] = buf[st.pa + o[k]];
          const double fargs = (double)st.nargs;
#pragma unroll
          for (int k = 0; k < kPer; ++k) t_compute[k] += pa[k] * fargs;
        }
        if (st.flags & APC_STEP_EDGE) {
          uint32_t j[kPer];
          if (st.row_src >= 0) {
            const uint32_t packed = s_rows[st.row_src * n_lane + tid];
#pragma unroll
            for (int k = 0; k < kPer; ++k) j[k] = (packed >> (8 * k)) & 0xFFu;
          } else if (st.has_src) {
#pragma unroll
            for (int k = 0; k < kPer; ++k) j[k] = draw(k, st.key_src, (uint32_t)st.ssrc);
          } else {
#pragma unroll
            for (int k = 0; k < kPer; ++k) j[k] = 0;
          }
          double raw[kPer];
#pragma unroll
          for (int k = 0; k < kPer; ++k) raw[k] = buf[st.mat + __umul24(o[k], (uint32_t)st.ssrc) + j[k]];
          add_entries(raw, st.has_src != 0, (st.flags & APC_STEP_TRANSITION) != 0, st.mult);
        }
      }
    } else {
      // A step's record is requested two steps ahead of its use and its producer's choices one
      // step ahead, behind everything else a step asks of LDS.
      const int s0 = head.step0, n_step = head.step1 - head.step0;
      auto load_words = [&](int s) -> StepWords {
        union { u32x8_t raw; StepWords w; } u;
        u.raw = *reinterpret_cast<const u32x8_t*>(static_cast<const StepWords*>(steps) + s0 + (s < n_step ? s : n_step - 1));
        return u.w;
      };
      auto row_choices = [&](uint32_t row) -> uint32_t { return s_rows[(row == kNoRow ? 0u : row) * n_lane + tid]; };
      StepWords st = load_words(0), next = load_words(1);
      uint32_t kept = row_choices((st.lo[2] >> 8) & 0xFFu);
      for (int s = 0; s < n_step; ++s) {
        const StepWords after = load_words(s + 2);
        const uint32_t flags = st.lo[0] >> 26, mat = st.lo[0] & 0x1FFFu, at_pa = (st.lo[0] >> 13) & 0x1FFFu;
        const uint32_t ssrc = st.lo[1] & 0x1FFu;
        if (flags & APC_STEP_FIRST) {
          const uint32_t packed = row_choices(st.lo[2] & 0xFFu);
#pragma unroll
          for (int k = 0; k < kPer; ++k) o[k] = (packed >> (8 * k)) & 0xFFu;
#pragma unroll
          for (int k = 0; k < kPer; ++k) pa[k] = buf[at_pa + o[k]];
        }
        const uint32_t packed = st.hi[1] ? kept : 0u;
        kept = row_choices((next.lo[2] >> 8) & 0xFFu);
        if (flags & APC_STEP_EDGE) {
          double raw[kPer];
#pragma unroll
          for (int k = 0; k < kPer; ++k) raw[k] = buf[mat + __umul24(o[k], ssrc) + ((packed >> (8 * k)) & 0xFFu)];
          add_entries(raw, st.hi[1] != 0, (flags & APC_STEP_TRANSITION) != 0, (int)st.hi[0]);
        }
        if (flags & APC_STEP_FIRST) {
          const double fargs = (double)(int)st.lo[3];
#pragma unroll
          for (int k = 0; k < kPer; ++k) t_compute[k] += pa[k] * fargs;
        }
        st = next;
        next = after;
      }
    }
    head = head1;
    head1 = head2;
    if (t + 2 < n_tile) unit1 = load_unit(head1, lane);
    if (t + 1 < n_tile) keep_rows();
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    if (t_raw + k * lanes >= n_assign) continue;
    const double t_trans = add_ones(init ? init[asg(k) * 6 + 3] : 0.0, n_trans[k]);
    double forbidden = init ? init[asg(k) * 6 + 5] : 0.0;
    if (tiles[0].any_edge) forbidden += 0.0;  // a walk adds 0.0 or 1.0 per edge: a carried -0.0 loses its sign
    forbidden = add_ones(forbidden, n_forbidden[k]);
    double* r = out + asg(k) * 6;
    r[0] = (t_compute[k] + t_comm[k]) + t_trans;
    r[1] = t_compute[k];
    r[2] = t_comm[k];
    r[3] = t_trans;
    r[4] = obj[k];
    r[5] = forbidden;
  }
}

template <bool kRandom, int kPer>
int launch_tiles(const apc_problem& p, const double* per_arg, const double* table, const void* steps,
                 const apc_score_tile* tiles, int n_tile, const apc_score_unit* units, const uint16_t* assign,
                 int64_t stride, uint64_t seed, int64_t first, int64_t n_assign, int clamp_inf, const double* init,
                 double* out, int n_lane, hipStream_t stream) {
  const int lds = 2 * kTileDoubles * 8 + kRows * n_lane * 4;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(score_tiles_kernel<kRandom, kPer>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return fail(APC_ERR_LAUNCH, "hipFuncSetAttribute(score_tiles_kernel): %s", hipGetErrorString(e));
  const int64_t per_block = (int64_t)n_lane * kPer;
  hipLaunchKernelGGL((score_tiles_kernel<kRandom, kPer>), dim3((unsigned)((n_assign + per_block - 1) / per_block)),
                     dim3(n_lane), lds, stream, p, per_arg, table, steps, tiles, n_tile, units, assign, stride, seed,
                     first, n_assign, clamp_inf, init, out);
  return check_launch("score_tiles_kernel");
}

}  // namespace

extern "C" {

int apc_score_tiles(const apc_edge* edges, int32_t n_edge, int32_t n_node, const int32_t* node_edge_off,
                    const int32_t* node_nstrat, const int32_t* node_nargs, const int64_t* node_comp_off,
                    int32_t first_node, int32_t explicit_rows, apc_score_step* steps, int64_t max_step,
                    apc_score_tile* tiles, int64_t max_tile, apc_score_unit* units, int64_t max_unit,
                    int32_t* n_step, int32_t* n_tile, int32_t* n_unit) {
  if (n_node < 0 || n_edge < 0 || first_node < 0 || first_node > n_node || !n_step || !n_tile || !n_unit || !steps ||
      !tiles || !units || (n_node > first_node && (!node_edge_off || !node_nstrat || !node_nargs || !node_comp_off)) ||
      (n_edge > 0 && !edges))
    return fail(APC_ERR_INVALID, "apc_score_tiles: null argument or first_node out of range%s");
  *n_step = *n_tile = *n_unit = 0;
  try {
    int64_t s = 0, t = -1, u = 0;
    int used = 0, n_row = 0;
    bool any_edge = false;
    struct Placed { int lds, n; };
    std::unordered_map<int64_t, Placed> at;  // (source, kind) -> where, within the tile
    std::unordered_map<int32_t, int> row_of;
    auto end_tile = [&]() {
      apc_score_tile& tile = tiles[t];
      tile.step1 = (int32_t)s;
      tile.unit1 = (int32_t)u;
      tile.n_row = n_row;
      for (int r = n_row; r < kRows; ++r) tile.row[r] = n_row ? tile.row[0] : first_node;
    };
    auto new_tile = [&]() -> bool {
      if (t >= 0) end_tile();
      if (++t >= max_tile) return false;
      memset(&tiles[t], 0, sizeof(tiles[t]));
      tiles[t].step0 = (int32_t)s;
      tiles[t].unit0 = (int32_t)u;
      used = n_row = 0;
      at.clear();
      row_of.clear();
      return true;
    };
    // LDS doubles that n elements from src of a kind (0 table, 1 per_arg, 2 default_vals) would
    // still take in this tile
    auto needs = [&](int64_t src, int kind, int n) {
      auto found = at.find(src * 3 + kind);
      return found != at.end() && found->second.n >= n ? 0 : (n + 1) / 2 * 2;
    };
    auto place = [&](int64_t src, int kind, int n) -> int {  // -1: no room for units
      auto found = at.find(src * 3 + kind);
      if (found != at.end() && found->second.n >= n) return found->second.lds;
      const int to = used;
      const int chunk = kind == 0 ? kUnitDoubles : kUnitSingles;
      for (int done = 0; done < n; done += chunk) {
        if (u >= max_unit) return -1;
        apc_score_unit& unit = units[u++];
        unit.src = src + done;
        unit.lds = (uint16_t)(to + done);
        unit.n = (uint16_t)std::min(chunk, n - done);
        unit.kind = kind;
      }
      used += (n + 1) / 2 * 2;
      at[src * 3 + kind] = Placed{to, n};
      return to;
    };
    auto row = [&](int32_t v) -> int {
      auto found = row_of.find(v);
      if (found != row_of.end()) return found->second;
      tiles[t].row[n_row] = v;
      row_of.emplace(v, n_row);
      return n_row++;
    };
    if (!new_tile()) return fail(APC_ERR_INVALID, "apc_score_tiles: max_tile is too small%s");
    for (int v = first_node; v < n_node; ++v) {
      const int e0 = node_edge_off[v], e1 = node_edge_off[v + 1];
      if (e0 < 0 || e0 > e1 || e1 > n_edge) return fail(APC_ERR_INVALID, "apc_score_tiles: node_edge_off is no list of offsets%s");
      if (node_nstrat[v] < 1 || node_nstrat[v] > 256) return 0;  // a choice does not fit its byte
      for (int e = e0; e < (e1 > e0 ? e1 : e0 + 1); ++e) {
        const apc_edge* const ed = e < e1 ? edges + e : nullptr;
        const bool starts = e == e0;
        int matrix = 0, kind = 0;
        int64_t src = 0;
        if (ed) {
          if (ed->flags & APC_EDGE_COMPRESSED) return 0;
          if (ed->sdst != node_nstrat[v] || ed->ssrc < 1 || ed->src_node >= v) return 0;
          if (ed->src_node >= 0 && ed->ssrc > 256) return 0;
          const int64_t size = (int64_t)ed->ssrc * ed->sdst;
          if (size > kTileDoubles - 256) return 0;  // its matrix and a node's terms do not fit a buffer
          matrix = (int)size;
          kind = ed->table_off >= 0 ? 0 : 2;
          src = kind == 0 ? ed->table_off : ed->default_off;
          if (src < 0 || (kind == 0 && (src & 1))) return 0;
          any_edge = true;
        }
        // a tile's room: doubles, and with explicit choices rows
        int need = (ed ? needs(src, kind, matrix) : 0) + needs(node_comp_off[v], 1, node_nstrat[v]);
        int rows = 0;
        if (explicit_rows) {
          if (!row_of.count(v)) ++rows;
          if (ed && ed->src_node >= 0 && !row_of.count(ed->src_node)) ++rows;
        }
        if (used + need > kTileDoubles || n_row + rows > kRows || (explicit_rows && s - tiles[t].step0 >= kTileSteps))
          if (!new_tile()) return fail(APC_ERR_INVALID, "apc_score_tiles: max_tile or max_unit is too small%s");
        if (s >= max_step) return fail(APC_ERR_INVALID, "apc_score_tiles: max_step is too small%s");
        apc_score_step& r = steps[s];
        memset(&r, 0, sizeof(r));
        r.node = v;
        r.nstrat = node_nstrat[v];
        r.nargs = node_nargs[v] > 1 ? node_nargs[v] : 1;
        r.src_node = -1;
        r.row_src = -1;
        r.row_node = explicit_rows ? row(v) : v & (kRows - 1);
        if (starts) r.flags |= APC_STEP_FIRST;
        int placed = r.pa = place(node_comp_off[v], 1, node_nstrat[v]);  // again, where a node goes on in another tile
        if (ed) {
          r.flags |= APC_STEP_EDGE;
          r.ssrc = ed->ssrc;
          r.src_node = ed->src_node;
          if (ed->src_node >= 0 && (ed->flags & APC_EDGE_SCORE_TRANSITION)) r.flags |= APC_STEP_TRANSITION;
          r.mat = place(src, kind, matrix);
          if (r.mat < 0) placed = -1;
          if (ed->src_node >= 0) {
            if (explicit_rows) r.row_src = row(ed->src_node);
            else if (ed->src_node >= first_node && v - ed->src_node < kRows) r.row_src = ed->src_node & (kRows - 1);
          }
        }
        if (placed < 0) return fail(APC_ERR_INVALID, "apc_score_tiles: max_unit is too small%s");
        ++s;
      }
    }
    end_tile();
    tiles[0].any_edge = any_edge;
    if (s == 0) return 0;
    *n_step = (int32_t)s;
    *n_tile = (int32_t)(t + 1);
    *n_unit = (int32_t)u;
  } catch (const std::exception&) {
    return fail(APC_ERR_INVALID, "apc_score_tiles: out of host memory%s");
  }
  return 0;
}

int apc_score_from_tiles(const apc_problem* p, const double* per_arg, const double* table, const apc_score_step* steps,
                         int32_t n_step, const apc_score_tile* tiles, int32_t n_tile, const apc_score_unit* units,
                         void* call_steps, const uint16_t* assign, uint64_t seed, int64_t first,
                         int64_t n_assign, const int32_t* node_gid, int32_t clamp_inf, const double* init, double* out,
                         void* stream) {
  if (int rc = validate_problem(p)) return rc;
  if (n_assign <= 0) return 0;
  if (!per_arg || !steps || !tiles || !units || !call_steps || !out || !p->node_multiplier || n_step <= 0 || n_tile <= 0 ||
      (p->table_size > 0 && !table))
    return fail(APC_ERR_INVALID, "apc_score_from_tiles: null argument or an empty layout%s");
  const dim3 step_grid((unsigned)((n_step + kBlock - 1) / kBlock));
  if (assign)
    hipLaunchKernelGGL(score_steps_kernel<false>, step_grid, dim3(kBlock), 0, (hipStream_t)stream, *p, steps, n_step,
                       node_gid, call_steps);
  else
    hipLaunchKernelGGL(score_steps_kernel<true>, step_grid, dim3(kBlock), 0, (hipStream_t)stream, *p, steps, n_step,
                       node_gid, call_steps);
  if (int rc = check_launch("score_steps_kernel")) return rc;
  // One workgroup per CU, of as many lanes as the batch has for it; from 1 024 on, two or four
  // assignments per lane.
  const int most = assign ? 2 : 4;  // assignments a lane's registers hold; explicit choices take some
  const int64_t kChunk = (int64_t)256 * kMaxLanes * most;
  for (int64_t a0 = 0; a0 < n_assign; a0 += kChunk) {
    const int64_t n = n_assign - a0 < kChunk ? n_assign - a0 : kChunk;
    const int64_t share = (n + 255) / 256;
    const int per = share <= kMaxLanes ? 1 : share <= 2 * kMaxLanes ? 2 : 4;
    int n_lane = (int)(((share + per - 1) / per + 63) / 64 * 64);
    if (n_lane < 128) n_lane = 128;
    const uint16_t* asg = assign ? assign + a0 : nullptr;
    const double* in = init ? init + a0 * 6 : nullptr;
    int rc;
#define APC_TILES(R, K)                                                                                             \
  launch_tiles<R, K>(*p, per_arg, table, call_steps, tiles, n_tile, units, asg, n_assign, seed, first + a0, n,      \
                     (int)clamp_inf, in, out + a0 * 6, n_lane, (hipStream_t)stream)
    if (assign) rc = per == 1 ? APC_TILES(false, 1) : APC_TILES(false, 2);
    else rc = per == 1 ? APC_TILES(true, 1) : per == 2 ? APC_TILES(true, 2) : APC_TILES(true, 4);
#undef APC_TILES
    if (rc) return rc;
  }
  return 0;
}

}  // extern "C"

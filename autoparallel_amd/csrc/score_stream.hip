// Batch scoring of graphs with large blocks from the block table, as a stream of pieces through LDS (gfx950), and its
// C ABI.
//
// One workgroup per CU has the matrix of the current edge in LDS and draws from there (the reasons stand at
// score_table_kernel, which does the same edge by edge).  That walk was bound by waits, 2.2 us per edge: everything it
// looks up on the way (records, index lists, per-argument terms) comes by loads whose wait is one for the copy of the
// next matrix too, a matrix of several tiles waits for each of them, and matrices above 128 KB were read in place, at
// 8 cycles a draw and CU.  Here a launch in front writes what every step needs into records and side images; the walk
// then is a list of pieces of at most 64 KB, whatever edge they belong to, and nothing else is waited for: the records of
// 64 pieces are in the lanes' registers (lane i: piece t + i), per-argument terms and index lists arrive with an edge's
// first piece.  The pieces lie in a ring of 160 KB, one behind the other, and are asked for as soon as the ring has room
// (apc_score_pieces works out where and when): with one piece under way at a time a copy is its latency, 0.8 us a piece
// whatever its size.
// Measured, MI355X, window of the planner DAG of 1 600 nodes (2 967 edges, 194 MB of matrices), edge by edge and as a
// stream: calls with carried sums, repeated on one set of inputs, 196 608 random assignments 5.27 -> 4.21 ms, 524 288
// 6.54 -> 5.48, 2^20 9.48 -> 7.40; on inputs that change from call to call, so that the matrices come from memory,
// 524 288 7.3 -> 5.9.  What bounds it: with the fewest lanes the copies (3.2 ms by themselves: 0.9 us latency over the
// 75 KB that are under way beside a piece in use; four consecutive buffers of 32 KB reach 1.8 ms), at 2^20 instructions,
// two hashes per edge and assignment first of all.  Not better, at 524 288: pieces of 44 KB (9% longer), a piece asked for
// by one wavefront (16%) or by all of them (23%).
// Sums run in node order, then argument order, as in score_kernel: the same bits.
#include <algorithm>

#include "apc_device.h"
#include "score_tiles.h"

namespace {

using namespace apc_tiles;

constexpr int kPieceDoubles = APC_SCORE_PIECE;  // 64 KB
constexpr int kSideBytes = APC_SCORE_SIDE_BYTES;
constexpr int kRingBytes = 160 * 1024;
constexpr int kAheadMost = 16;  // pieces under way
static_assert(2 * (kPieceDoubles * 8 + kSideBytes) <= kRingBytes, "a piece and the next one");

typedef const __attribute__((address_space(1))) double* global_f64_ptr_t;
typedef const __attribute__((address_space(3))) uint16_t* lds_u16_ptr_t;
typedef const __attribute__((address_space(3))) double* lds_f64_ptr_t;

enum : uint32_t {
  kFirstOfNode = APC_PIECE_FIRST_OF_NODE, kFirst = APC_PIECE_FIRST, kLast = APC_PIECE_LAST,  // of its edge
  kEdge = 8, kSource = 16, kTransition = 32, kInPlace = 64,
};

// What the walk has to know about a piece.
struct WalkRec {
  uint32_t flags, ask;           // pieces asked for when the ring has let go of the one before: all in front of this number
  uint32_t side, mat;            // in LDS, bytes
  uint32_t base, n;              // elements of its matrix in front of it and in it
  uint32_t nstrat, key_node, ssrc, key_src;
  uint32_t row;                  // length of a matrix row
  int32_t mult, nargs;
  uint32_t at_lo, at_hi;         // of a matrix that is read in place
  uint32_t reserved;
};
// And what its copy has to.
struct AskRec {
  uint32_t from_lo, from_hi, chunks, mat;  // of the matrix: where it is, in 16-byte pieces, where to in LDS
  uint32_t item, side_kb, side, reserved;  // its item's side image, if the item begins with this piece
};
static_assert(sizeof(WalkRec) == 64 && sizeof(AskRec) == 32 && sizeof(apc_score_piece) == 32, "layout");
// A side image: per-argument terms by choice, then the matrix row of every choice and the column of every choice of the
// producer, 16 bits each.

__global__ void __launch_bounds__(kBlock)
score_pieces_kernel(apc_problem p, const double* __restrict__ per_arg, const double* __restrict__ table,
                    const apc_score_piece* __restrict__ pieces, const int32_t* __restrict__ node_gid,
                    char* __restrict__ sides, WalkRec* __restrict__ walk, AskRec* __restrict__ ask) {
  const int t = (int)blockIdx.x, tid = threadIdx.x;
  const apc_score_piece q = pieces[t];
  if (tid == 0) {
    WalkRec r = {};
    AskRec a = {};
    r.flags = (uint32_t)q.flags;
    r.ask = (uint32_t)q.ask;
    r.side = a.side = (uint32_t)q.lds;
    const int side_bytes = 10 * p.node_nstrat[q.node] + (q.edge >= 0 ? 2 * p.edges[q.edge].ssrc : 0);
    if (q.flags & APC_PIECE_FIRST) a.side_kb = (uint32_t)((side_bytes + 1023) >> 10);
    r.mat = a.mat = (uint32_t)q.lds + a.side_kb * 1024u;
    a.item = (uint32_t)q.item;
    r.base = (uint32_t)q.base;
    r.n = (uint32_t)q.n;
    r.nstrat = (uint32_t)p.node_nstrat[q.node];
    r.key_node = fold16(node_key(node_gid ? node_gid[q.node] : q.node));
    r.mult = p.node_multiplier[q.node];
    r.nargs = p.node_nargs[q.node] > 1 ? p.node_nargs[q.node] : 1;
    if (q.edge >= 0) {
      const apc_edge ed = p.edges[q.edge];
      r.flags |= kEdge;
      r.row = ed.flags & APC_EDGE_COMPRESSED ? (uint32_t)ed.flags >> APC_EDGE_USRC_SHIFT : (uint32_t)ed.ssrc;
      if (ed.src_node >= 0) {
        r.flags |= kSource | (ed.flags & APC_EDGE_SCORE_TRANSITION ? kTransition : 0u);
        r.ssrc = (uint32_t)ed.ssrc;
        r.key_src = fold16(node_key(node_gid ? node_gid[ed.src_node] : ed.src_node));
      }
      if (ed.table_off < 0) {
        const uint64_t at = (uint64_t)(uintptr_t)(p.default_vals + ed.default_off);
        r.flags |= kInPlace;
        r.at_lo = (uint32_t)at;
        r.at_hi = (uint32_t)(at >> 32);
      } else {
        const uint64_t from = (uint64_t)(uintptr_t)(table + ed.table_off + q.base);
        a.from_lo = (uint32_t)from;
        a.from_hi = (uint32_t)(from >> 32);
        a.chunks = (uint32_t)(q.n + 1) >> 1;
      }
    }
    walk[t] = r;
    ask[t] = a;
  }
  if (!(q.flags & APC_PIECE_FIRST)) return;
  char* const side = sides + (size_t)q.item * kSideBytes;
  const int S = p.node_nstrat[q.node];
  uint16_t* const rows = reinterpret_cast<uint16_t*>(side + 8 * S);
  uint16_t* const cols = rows + S;
  for (int i = tid; i < S; i += kBlock) reinterpret_cast<double*>(side)[i] = per_arg[p.node_comp_off[q.node] + i];
  if (q.edge < 0) return;
  const apc_edge ed = p.edges[q.edge];
  const bool squeezed = (ed.flags & APC_EDGE_COMPRESSED) != 0;
  for (int i = tid; i < S; i += kBlock) rows[i] = (uint16_t)(squeezed ? p.list_uidx[(size_t)ed.dst_list + i] : i);
  for (int i = tid; i < ed.ssrc; i += kBlock) cols[i] = (uint16_t)(squeezed ? p.list_uidx[(size_t)ed.src_list + i] : i);
}

template <int kPer>
__global__ void __launch_bounds__(1024)
score_stream_kernel(const WalkRec* __restrict__ walk, const AskRec* __restrict__ asks, int n_piece,
                    const char* __restrict__ sides, uint64_t seed, int64_t first, int64_t n_assign, int clamp_inf,
                    const double* __restrict__ init, double* __restrict__ out) {
  extern __shared__ __align__(16) char s_mem[];  // the ring
  const int n_lane = blockDim.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), n_wave = n_lane >> 6;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)s_mem;
  const int64_t lanes = (int64_t)gridDim.x * n_lane;
  const int64_t t_raw = (int64_t)blockIdx.x * n_lane + tid;
  const int64_t t_first = t_raw < n_assign ? t_raw : 0;
  // assignment k of this lane; a lane past the end repeats another one and stores nothing
  auto asg = [&](int k) -> int64_t {
    const int64_t ak = t_raw + k * lanes;
    return ak < n_assign ? ak : t_first;
  };
  double t_compute[kPer], t_comm[kPer], obj[kPer], pa[kPer], raw[kPer];
  uint32_t n_trans[kPer], n_forbidden[kPer], h0[kPer], o[kPer], at[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    t_compute[k] = t_comm[k] = obj[k] = pa[k] = raw[k] = 0.0;
    n_trans[k] = n_forbidden[k] = o[k] = at[k] = 0;
    if (init) {
      const double* r = init + asg(k) * 6;
      t_compute[k] = r[1]; t_comm[k] = r[2]; obj[k] = r[4];
    }
    h0[k] = fold16(assignment_hash(seed, first + asg(k)));
    // the loads of init end here, not where the sums are first added to
    asm volatile("" : "+v"(t_compute[k]), "+v"(t_comm[k]), "+v"(obj[k]));
  }
  auto draw = [&](int k, uint32_t key, uint32_t nstrat) -> uint32_t {  // plain_draw by the node's key
    return folded_draw(h0[k], key, nstrat);
  };
  // by 32-bit addresses: a pointer that may go elsewhere makes flat loads, and those wait for the copies, too
  auto lds_f64 = [](uint32_t at) -> double { return *(lds_f64_ptr_t)(uintptr_t)at; };
  auto lds_u16 = [](uint32_t at) -> uint32_t { return *(lds_u16_ptr_t)(uintptr_t)at; };
  u32x4_t rec[4], ask[2];  // of 64 pieces each, lane i: the i-th
  auto word = [&](int i, int s) -> uint32_t { return (uint32_t)__builtin_amdgcn_readlane((int)rec[i >> 2][i & 3], s); };
  auto ask_word = [&](int i, int s) -> uint32_t { return (uint32_t)__builtin_amdgcn_readlane((int)ask[i >> 2][i & 3], s); };
  // A piece is asked for by four wavefronts, each four in their turn: what that takes besides the loads would cost
  // sixteen four times as much.
  const int n_team = n_wave >> 2, team = wave >> 2, member = wave & 3;
  int n_asked = 0, turn = 0;  // pieces asked for, and whose turn the next one is
  auto ask_for = [&](int upto) {  // nothing waits here, except for the next 64 records
    for (; n_asked < upto; ++n_asked) {
      const int s = n_asked & 63;
      if (s == 0) {
        const u32x4_t* const r = reinterpret_cast<const u32x4_t*>(asks + min(n_asked + lane, n_piece - 1));
        ask[0] = r[0];
        ask[1] = r[1];
        asm volatile("" : "+v"(ask[0]), "+v"(ask[1]));  // waited for here, not on every pass through the loop
      }
      if (turn == team) {
        const uint32_t side_kb = ask_word(5, s);
        const char* const side = sides + (size_t)ask_word(4, s) * kSideBytes + lane * 16;
        const uint32_t to_side = lds0 + ask_word(6, s);
        for (uint32_t c = (uint32_t)member; c < side_kb; c += 4) load16_lds(side + c * 1024, to_side + c * 1024u);
        const uint32_t chunks = ask_word(2, s), to = lds0 + ask_word(3, s);
        const char* const from = reinterpret_cast<const char*>((uint64_t)ask_word(1, s) << 32 | ask_word(0, s)) + lane * 16;
        uint32_t c = (uint32_t)member * 256u;
        for (; c + 256 <= chunks; c += 1024) load16x4_lds(from + c * 16, to + c * 16u);
        for (const uint32_t end = min(c + 256u, chunks); c < end; c += 64)
          if (c + lane < chunks) load16_lds(from + c * 16, to + c * 16u);
      }
      turn = turn + 1 == n_team ? 0 : turn + 1;
    }
  };
  int awaited = 0;  // whose piece is t
  for (int t = 0; t < n_piece; ++t) {
    const int s = t & 63;
    if (s == 0) {
      const u32x4_t* const r = reinterpret_cast<const u32x4_t*>(walk + min(t + lane, n_piece - 1));
#pragma unroll
      for (int i = 0; i < 4; ++i) rec[i] = r[i];
      asm volatile("" : "+v"(rec[0]), "+v"(rec[1]), "+v"(rec[2]), "+v"(rec[3]));
    }
    if (n_asked == t) {  // there was no room for this piece beside the one before
      if (t > 0) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      ask_for(t + 1);
    }
    if (awaited == team) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // piece t has arrived,
    awaited = awaited + 1 == n_team ? 0 : awaited + 1;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // for everyone; and the piece before is done with
    ask_for((int)word(1, s));
    const uint32_t flags = word(0, s);
    const uint32_t mat = lds0 + word(3, s);
    if (flags & kFirst) {
      const uint32_t side = lds0 + word(2, s);
      const uint32_t nstrat = word(6, s);
      if (flags & kFirstOfNode) {
        const uint32_t key = word(7, s);
        const double fargs = (double)(int)word(12, s);
#pragma unroll
        for (int k = 0; k < kPer; ++k) o[k] = draw(k, key, nstrat);
#pragma unroll
        for (int k = 0; k < kPer; ++k) pa[k] = lds_f64(side + o[k] * 8u);
#pragma unroll
        for (int k = 0; k < kPer; ++k) t_compute[k] += pa[k] * fargs;
      }
      if (flags & kEdge) {
        const uint32_t rows = side + 8 * nstrat, cols = rows + 2 * nstrat;
        const uint32_t row = word(10, s);
        uint32_t j[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) j[k] = 0;
        if (flags & kSource) {
          const uint32_t key = word(9, s), ssrc = word(8, s);
#pragma unroll
          for (int k = 0; k < kPer; ++k) j[k] = draw(k, key, ssrc);
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) at[k] = __umul24(lds_u16(rows + o[k] * 2u), row) + lds_u16(cols + j[k] * 2u);
      }
    }
    if (!(flags & kEdge)) continue;
    if (flags & kInPlace) {
      const global_f64_ptr_t matrix = (global_f64_ptr_t)((uint64_t)word(14, s) << 32 | word(13, s));
#pragma unroll
      for (int k = 0; k < kPer; ++k) raw[k] = matrix[at[k]];
      // waited for here, not on every pass through the loop
#pragma unroll
      for (int k = 0; k < kPer; ++k) asm volatile("" : "+v"(raw[k]));
    } else if ((flags & (kFirst | kLast)) == (kFirst | kLast)) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) raw[k] = lds_f64(mat + at[k] * 8u);
    } else {
      const uint32_t base = word(4, s), n = word(5, s);
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const uint32_t local = at[k] - base;
        if (local < n) raw[k] = lds_f64(mat + local * 8u);
      }
    }
    if (!(flags & kLast)) continue;
    // what the build makes of a matrix element, added up
    const int mult = (int)word(11, s);
    const uint32_t counts = flags & kTransition ? 1u : 0u;
    const bool has_src = (flags & kSource) != 0;
    double c[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const uint32_t hi = (uint32_t)((uint64_t)__double_as_longlong(raw[k]) >> 32);
      c[k] = (fabs(raw[k]) + pa[k]) +
             __longlong_as_double((long long)((uint64_t)((uint32_t)((int32_t)hi >> 31) & 0x3FF00000u) << 32));
      const bool finite = __builtin_amdgcn_class(c[k], kFinite);
      c[k] = finite || !clamp_inf ? c[k] : 10000.0;
      n_forbidden[k] += finite ? 0u : 1u;
      const double more = t_comm[k] + fabs(raw[k]);
      t_comm[k] = has_src && __builtin_amdgcn_class(raw[k], kFinite) ? more : t_comm[k];
      n_trans[k] += (hi >> 31) & counts;
    }
    if (mult != 1) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) c[k] *= (double)mult;
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) obj[k] += c[k];
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing is in flight towards LDS when the workgroup ends
  bool any_edge = false;
  for (int t = lane; t < n_piece && !any_edge; t += 64) any_edge = walk[t].flags & kEdge;
  any_edge = __ballot(any_edge) != 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    if (t_raw + k * lanes >= n_assign) continue;
    const double t_trans = add_ones(init ? init[asg(k) * 6 + 3] : 0.0, n_trans[k]);
    double forbidden = init ? init[asg(k) * 6 + 5] : 0.0;
    if (any_edge) forbidden += 0.0;  // a walk adds 0.0 or 1.0 per edge: a carried -0.0 loses its sign
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

template <int kPer>
int launch_stream(const WalkRec* walk, const AskRec* asks, int n_piece, const char* sides, uint64_t seed, int64_t first,
                  int64_t n_assign, int clamp_inf, const double* init, double* out, int n_lane, hipStream_t stream) {
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(score_stream_kernel<kPer>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, kRingBytes);
  if (e != hipSuccess) return fail(APC_ERR_LAUNCH, "hipFuncSetAttribute(score_stream_kernel): %s", hipGetErrorString(e));
  const int64_t per_block = (int64_t)n_lane * kPer;
  hipLaunchKernelGGL((score_stream_kernel<kPer>), dim3((unsigned)((n_assign + per_block - 1) / per_block)), dim3(n_lane),
                     kRingBytes, stream, walk, asks, n_piece, sides, seed, first, n_assign, clamp_inf, init, out);
  return check_launch("score_stream_kernel");
}

}  // namespace

extern "C" {

int apc_score_pieces(const apc_edge* edges, int32_t n_edge, int32_t n_node, const int32_t* node_edge_off,
                     const int32_t* node_nstrat, const int32_t* msize, int32_t first_node, apc_score_piece* pieces,
                     int64_t max_piece, int32_t* n_piece, int32_t* n_item) {
  if (n_node < 0 || n_edge < 0 || first_node < 0 || first_node > n_node || !pieces || !n_piece || !n_item ||
      (n_node > first_node && (!node_edge_off || !node_nstrat)) || (n_edge > 0 && (!edges || !msize)))
    return fail(APC_ERR_INVALID, "apc_score_pieces: null argument or first_node out of range%s");
  *n_piece = *n_item = 0;
  int64_t t = 0;
  int32_t item = 0;
  auto side_kb = [&](int v, int e) { return (10 * node_nstrat[v] + (e >= 0 ? 2 * edges[e].ssrc : 0) + 1023) / 1024; };
  for (int v = first_node; v < n_node; ++v) {
    const int e0 = node_edge_off[v], e1 = node_edge_off[v + 1];
    if (e0 < 0 || e0 > e1 || e1 > n_edge) return fail(APC_ERR_INVALID, "apc_score_pieces: node_edge_off is no list of offsets%s");
    for (int e = e0; e < (e1 > e0 ? e1 : e0 + 1); ++e, ++item) {
      const int edge = e < e1 ? e : -1;
      if (node_nstrat[v] < 1 || node_nstrat[v] > kSideBytes / 10 || (edge >= 0 && edges[edge].ssrc > kSideBytes / 2) ||
          side_kb(v, edge) * 1024 > kSideBytes)
        return 0;  // its side image does not fit
      const int64_t size = edge >= 0 && edges[edge].table_off >= 0 ? msize[edge] : 0;
      if (size < 0 || (size > 0 && (edges[edge].table_off & 1))) return 0;
      int64_t base = 0;
      do {
        if (t >= max_piece) return fail(APC_ERR_INVALID, "apc_score_pieces: max_piece is too small%s");
        apc_score_piece& q = pieces[t++];
        memset(&q, 0, sizeof(q));
        q.node = v;
        q.edge = edge;
        q.item = item;
        q.base = (int32_t)base;
        q.n = (int32_t)std::min<int64_t>(size - base, kPieceDoubles);
        q.flags = (e == e0 && base == 0 ? APC_PIECE_FIRST_OF_NODE : 0) | (base == 0 ? APC_PIECE_FIRST : 0);
        base += kPieceDoubles;
        if (base >= size) q.flags |= APC_PIECE_LAST;
      } while (base < size);
    }
  }
  // Where in the ring, and when: behind the last one, or at the start where that does not fit, as soon as the
  // pieces still in use leave the room.
  auto bytes = [&](int64_t i) {
    const apc_score_piece& q = pieces[i];
    return (q.flags & APC_PIECE_FIRST ? side_kb(q.node, q.edge) * 1024 : 0) + (q.n * 8 + 1023) / 1024 * 1024;
  };
  int64_t next = 0;  // to be placed
  int at = 0;        // behind the last one placed
  for (int64_t i = 0; i < t; ++i) {  // pieces from i on are in use, or on their way
    if (next == i) at = 0;           // none is
    for (; next < t && next < i + kAheadMost; ++next) {
      const int size = bytes(next);
      if (next > i) {
        const int from = pieces[i].lds, last = pieces[next - 1].lds;  // in use: from .. at, round the end if last < from
        if (last >= from) {
          if (at + size > kRingBytes) {
            if (size > from) break;
            at = 0;
          }
        } else if (at + size > from) {
          break;
        }
      }
      pieces[next].lds = at;
      at += size;
    }
    pieces[i].ask = (int32_t)next;
  }
  *n_piece = (int32_t)t;
  *n_item = item;
  return 0;
}

int apc_score_stream(const apc_problem* p, const double* per_arg, const double* table, const apc_score_piece* pieces,
                     int32_t n_piece, int32_t n_item, void* scratch, uint64_t seed, int64_t first, int64_t n_assign,
                     const int32_t* node_gid, int32_t clamp_inf, const double* init, double* out, void* stream) {
  if (int rc = validate_problem(p)) return rc;
  if (n_assign <= 0) return 0;
  if (!per_arg || !pieces || !scratch || !out || !p->node_multiplier || n_piece <= 0 || n_item <= 0 ||
      (p->table_size > 0 && !table))
    return fail(APC_ERR_INVALID, "apc_score_stream: null argument or no pieces%s");
  char* const sides = static_cast<char*>(scratch);
  WalkRec* const walk = reinterpret_cast<WalkRec*>(sides + (size_t)n_item * kSideBytes);
  AskRec* const asks = reinterpret_cast<AskRec*>(walk + n_piece);
  hipLaunchKernelGGL(score_pieces_kernel, dim3((unsigned)n_piece), dim3(kBlock), 0, (hipStream_t)stream, *p, per_arg,
                     table, pieces, node_gid, sides, walk, asks);
  if (int rc = check_launch("score_pieces_kernel")) return rc;
  const int64_t kChunk = (int64_t)256 * 1024 * 4;
  for (int64_t a0 = 0; a0 < n_assign; a0 += kChunk) {
    const int64_t n = n_assign - a0 < kChunk ? n_assign - a0 : kChunk;
    const int64_t share = (n + 255) / 256;  // of a CU
    const int per = share <= 1024 ? 1 : share <= 2048 ? 2 : 4;
    int n_lane = (int)(((share + per - 1) / per + 63) / 64 * 64);
    if (n_lane < 256) n_lane = 256;
    const double* in = init ? init + a0 * 6 : nullptr;
#define APC_STREAM(K)                                                                                                \
  launch_stream<K>(walk, asks, n_piece, sides, seed, first + a0, n, (int)clamp_inf, in, out + a0 * 6, n_lane,         \
                   (hipStream_t)stream)
    const int rc = per == 1 ? APC_STREAM(1) : per == 2 ? APC_STREAM(2) : APC_STREAM(4);
#undef APC_STREAM
    if (rc) return rc;
  }
  return 0;
}

}  // extern "C"

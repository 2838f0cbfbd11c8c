// Scoring of small batches from the block table (gfx950), and its C ABI.
//
// As score_fold_kernel (score.hip, where the reasons for its shape stand): a workgroup takes 1 << kShift assignments, its
// first kTermLanes lanes gather the terms of a tile of edges and nodes, one (row, assignment) pair a lane, and the
// wavefronts behind them add the tile before up meanwhile, in node order, then argument order: the same bits.  That
// kernel looks a pair's edge up field by field, a dozen loads each of which it waits for.  Here a launch in front writes
// one record per edge and per node with all a pair needs, and nothing is waited for where it is asked for: records a tile
// (with explicit choices two) ahead, choices a tile ahead, and a tile's terms are formed while the next tile's
// entries are on their way.
// Measured, MI355X, fields and records, us: 2 000 random assignments of the 12-layer GPT-2 graph 50 -> 33, of the
// Llama-3-8B graph 143 -> 94, 100 93 -> 64, 32 768 1 188 -> 629; 16 384 explicit ones of a 1 600-node window of the
// planner DAG 811 -> 567, 2 000 165 -> 126.  What bounds it: few assignments, the chain of additions (4.6 ns a term, of
// which 3.6 are the addition's latency); 2 000 and more, the gathering lanes' instructions (0.43 busy at 2 000, three
// hashes per edge and node); explicit ones on large blocks, the misses of a draw's entry.
#include "apc_device.h"

namespace {

constexpr int kTermLanes = 768;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
// a pointer made of a number is one to anywhere: its loads are flat ones, which a wait for LDS waits for, too
typedef const __attribute__((address_space(1))) double* global_f64_ptr_t;

struct FoldEdge {
  uint32_t mat_lo, mat_hi;  // its matrix
  uint32_t row;             // length of a matrix row
  uint32_t terms;           // the node's per-argument terms
  uint32_t node, src;       // what the draws start from, or the rows of explicit choices
  uint32_t sdst;            // strategies of the node
  int32_t mult;
  uint32_t dst_list, src_list, flags;
  uint32_t ssrc;            // and of the producer, 32 bits each: a node's number of them has no other bound
};
struct FoldNode { uint32_t terms, node, nstrat; int32_t nargs; };
constexpr uint32_t kSource = 1, kTransition = 2, kSqueezed = 4;
static_assert(sizeof(FoldEdge) == 48 && sizeof(FoldNode) == 16, "layout");

__global__ void __launch_bounds__(kBlock)
fold_records_kernel(apc_problem p, const double* __restrict__ table, const int32_t* __restrict__ node_gid, int first_node,
                    int e_first, int random, FoldEdge* __restrict__ edges, FoldNode* __restrict__ nodes) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  auto key = [&](int v) -> uint32_t { return random ? fold16(node_key(node_gid ? node_gid[v] : v)) : (uint32_t)v; };
  if (e_first + i < p.n_edge) {
    const apc_edge ed = p.edges[e_first + i];
    const bool squeezed = (ed.flags & APC_EDGE_COMPRESSED) != 0, has_src = ed.src_node >= 0;
    const uint64_t mat = ed.table_off >= 0 ? (uint64_t)(uintptr_t)table + (uint64_t)ed.table_off * 8u
                                           : (uint64_t)(uintptr_t)p.default_vals + (uint64_t)ed.default_off * 8u;
    FoldEdge r;
    r.mat_lo = (uint32_t)mat;
    r.mat_hi = (uint32_t)(mat >> 32);
    r.row = squeezed ? (uint32_t)ed.flags >> APC_EDGE_USRC_SHIFT : (uint32_t)ed.ssrc;
    r.terms = (uint32_t)ed.comp_base;
    r.node = key(ed.node);
    r.src = has_src ? key(ed.src_node) : 0u;
    r.sdst = (uint32_t)ed.sdst;
    r.mult = p.node_multiplier[ed.node];
    r.dst_list = squeezed ? ed.dst_list : 0u;
    r.src_list = squeezed ? ed.src_list : 0u;
    r.flags = (has_src ? kSource : 0u) | (has_src && (ed.flags & APC_EDGE_SCORE_TRANSITION) ? kTransition : 0u) |
              (squeezed ? kSqueezed : 0u);
    r.ssrc = (uint32_t)ed.ssrc;
    edges[i] = r;
  }
  if (first_node + i < p.n_node) {
    const int v = first_node + i, nargs = p.node_nargs[v];
    nodes[i] = FoldNode{(uint32_t)p.node_comp_off[v], key(v), (uint32_t)p.node_nstrat[v], nargs > 1 ? nargs : 1};
  }
}

// kTwo: for two workgroups per CU
template <bool kRandom, int kShift, bool kLists, int kUnroll, bool kTwo>
__global__ void __launch_bounds__(kTermLanes + 192, kTwo ? 8 : 4)
score_terms_kernel(const FoldEdge* __restrict__ edges, int n_edges, const FoldNode* __restrict__ nodes, int n_nodes,
                   const double* __restrict__ per_arg, const int32_t* __restrict__ list_uidx, int clamp_inf,
                   const uint16_t* __restrict__ assign, int64_t stride, uint64_t seed, int64_t first, int64_t n_assign,
                   const double* __restrict__ init, double* __restrict__ out) {
  constexpr int kGroup = 1 << kShift;
  constexpr int kTile = kTermLanes * kUnroll;  // (row, assignment) pairs of a tile
  constexpr int kRows = kTile >> kShift;       // edges (and nodes) of a tile
  // two rows of an assignment side by side, which spares the adding wavefront half its reads, where that one is
  // what a tile takes
  constexpr bool kPaired = !kTwo;
  extern __shared__ __align__(16) double s_terms[];  // [2][3][kTile]
  __shared__ double s_sum[3][kGroup];
  __shared__ uint32_t s_count[2][kGroup];  // transitions, forbidden entries
  const int tid = threadIdx.x;
  const bool gathers = tid < kTermLanes;  // else: adds up
  const int fold = tid - kTermLanes;
  const int al = (gathers ? tid : fold) & (kGroup - 1);
  const int sum = fold >> kShift;  // of a lane that adds up: 0 compute, 1 comm, 2 objective; idle beyond
  const int64_t a_raw = (int64_t)blockIdx.x * kGroup + al;
  const int64_t a = a_raw < n_assign ? a_raw : n_assign - 1;  // lanes past the end repeat the last one
  if (tid < 2 * kGroup) s_count[tid >> kShift][tid & (kGroup - 1)] = 0;
  const int n_max = n_edges > n_nodes ? n_edges : n_nodes;
  const int n_tiles = (n_max + kRows - 1) / kRows;
  uint32_t n_trans = 0, n_forbidden = 0;
  double acc = 0.0;
  if (init && !gathers && sum < 3) acc = init[a * 6 + (sum == 0 ? 1 : sum == 1 ? 2 : 4)];
  if (gathers) {
    const uint32_t h0 = fold16(assignment_hash(seed, first + a));
    const uint16_t* const my_assign = assign + a;
    struct Rec { u32x4_t e[3], n; };                        // a pair's edge and node
    struct Choices { uint32_t o, j, v; };                   // of its edge's node and producer, and of its node
    struct Values { double raw, pa, term; uint32_t flags; int32_t mult, nargs; };
    auto row_of = [&](int t, int u) -> int {
      const int row = t * kRows + ((u * kTermLanes + tid) >> kShift);
      return kShift == 6 ? __builtin_amdgcn_readfirstlane(row) : row;
    };
    auto load_rec = [&](int t, int u) -> Rec {
      const int row = row_of(t, u);
      const u32x4_t* const e = reinterpret_cast<const u32x4_t*>(edges + max(min(row, n_edges - 1), 0));
      Rec r;
      // The node's record in front of the edge's where 4 to 32 lanes read the same ones: 2 000, 4 000 and 8 000 random
      // assignments of the Llama-3-8B graph 113, 195 and 353 -> 93, 162 and 301 us, but 16 000 489 -> 504.
      constexpr bool kNodeFirst = kShift >= 2 && kShift < 6;
      if (kNodeFirst) r.n = *reinterpret_cast<const u32x4_t*>(nodes + min(row, n_nodes - 1));
      r.e[0] = e[0];
      r.e[1] = e[1];
      r.e[2] = e[2];
      if (!kNodeFirst) r.n = *reinterpret_cast<const u32x4_t*>(nodes + min(row, n_nodes - 1));
      return r;
    };
    auto draw = [&](uint32_t key, uint32_t nstrat) -> uint32_t {  // plain_draw by the node's key
      return folded_draw(h0, key, nstrat);
    };
    auto choose = [&](const Rec& r) -> Choices {
      Choices c;
      if (kRandom) {
        c.o = draw(r.e[1][0], r.e[1][2]);
        c.j = draw(r.e[1][1], r.e[2][3]);
        c.v = draw(r.n[1], r.n[2]);
      } else {
        c.o = my_assign[(size_t)r.e[1][0] * stride];
        c.j = my_assign[(size_t)r.e[1][1] * stride];
        c.v = my_assign[(size_t)r.n[1] * stride];
      }
      return c;
    };
    auto ask = [&](const Rec& r, const Choices& c) -> Values {
      const uint32_t flags = r.e[2][2], j = flags & kSource ? c.j : 0u;
      uint32_t d = c.o, s = j;
      if (kLists) {
        const bool squeezed = (flags & kSqueezed) != 0;
        const uint32_t ud = (uint32_t)list_uidx[squeezed ? (size_t)r.e[2][0] + c.o : 0];
        const uint32_t us = (uint32_t)list_uidx[squeezed ? (size_t)r.e[2][1] + j : 0];
        d = squeezed ? ud : d;
        s = squeezed ? us : s;
      }
      Values v;
      v.raw = ((global_f64_ptr_t)((uint64_t)r.e[0][1] << 32 | r.e[0][0]))[d * r.e[0][2] + s];
      v.pa = per_arg[r.e[0][3] + c.o];
      v.term = per_arg[r.n[0] + c.v];
      v.flags = flags;
      v.mult = (int32_t)r.e[1][3];
      v.nargs = (int32_t)r.n[3];
      return v;
    };
    auto put = [&](int t, int u, const Values& v) {
      const int row = (u * kTermLanes + tid) >> kShift;
      double* const s_t = s_terms + (t & 1) * 3 * kTile + 
                          (kPaired ? (((row >> 1) << kShift) + al) * 2 + (row & 1) : (row << kShift) + al);
      // as item_store forms an entry from its matrix element
      const uint32_t trans = (uint32_t)((uint64_t)__double_as_longlong(v.raw) >> 63);
      const double cm = fabs(v.raw);
      double c = (cm + v.pa) + __longlong_as_double((long long)((uint64_t)((0u - trans) & 0x3FF00000u) << 32));
      const bool finite = __builtin_amdgcn_class(c, kFinite);
      c = finite || !clamp_inf ? c : 10000.0;
      const bool live = t * kRows + row < n_edges;
      n_forbidden += live && !finite;
      n_trans += live && (v.flags & kTransition) ? trans : 0u;
      const double comm = (v.flags & kSource) && __builtin_amdgcn_class(v.raw, kFinite) ? cm : 0.0;
      // behind the last row: -0.0, which changes no sum
      s_t[0] = t * kRows + row < n_nodes ? v.term * (double)v.nargs : -0.0;
      s_t[kTile] = live ? comm : -0.0;
      s_t[2 * kTile] = live ? c * (double)v.mult : -0.0;
    };
    Rec rec[kUnroll], ahead[kUnroll];
    Choices chosen[kUnroll];
    Values asked[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      rec[u] = load_rec(0, u);
      if (!kRandom) {
        ahead[u] = load_rec(1, u);
        chosen[u] = choose(rec[u]);
      }
      asked[u] = Values{0.0, 0.0, 0.0, 0u, 0, 0};
    }
    for (int t = 0; t <= n_tiles + 1; ++t) {
      if (t <= n_tiles) {
        Values now[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          if (kRandom) chosen[u] = choose(rec[u]);
          now[u] = ask(rec[u], chosen[u]);
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          if (kRandom) {
            rec[u] = load_rec(t + 1, u);
          } else {
            rec[u] = ahead[u];
            chosen[u] = choose(rec[u]);
            ahead[u] = load_rec(t + 2, u);
          }
        }
        if (t > 0) {
#pragma unroll
          for (int u = 0; u < kUnroll; ++u) put(t - 1, u, asked[u]);
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) asked[u] = now[u];
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    if (n_trans) atomicAdd(&s_count[0][al], n_trans);
    if (n_forbidden) atomicAdd(&s_count[1][al], n_forbidden);
  } else {
    for (int t = 0; t <= n_tiles + 1; ++t) {
      if (t > 1 && sum < 3) {  // tile t - 2
        const double* __restrict__ s_t = s_terms + ((t & 1) * 3 + sum) * kTile;
        // The chain of additions is what a small batch takes: 3.6 ns each, and every other instruction of this one
        // wavefront 2.8.  So a read brings two terms, and the next kPairs reads are on their way while these are added.
        constexpr int kPairs = kRows % 16 == 0 ? 8 : kRows % 8 == 0 ? 4 : 6, kParts = kRows / 2 / kPairs;
        static_assert(kParts * kPairs * 2 == kRows, "whole parts");
        const int left = n_max - (t - 2) * kRows;
        const int parts = left < kRows ? (left + 2 * kPairs - 1) / (2 * kPairs) : kParts;
        double2_t x[kPairs], y[kPairs];
        auto read = [&](double2_t (&to)[kPairs], int part) {
#pragma unroll
          for (int i = 0; i < kPairs; ++i) {
            const int pair = part * kPairs + i;
            if (kPaired) to[i] = reinterpret_cast<const double2_t*>(s_t)[(pair << kShift) + al];
            else to[i] = double2_t{s_t[((2 * pair) << kShift) + al], s_t[((2 * pair + 1) << kShift) + al]};
          }
        };
        auto add = [&](const double2_t (&from)[kPairs]) {
#pragma unroll
          for (int i = 0; i < kPairs; ++i) {
            acc += from[i].x;
            acc += from[i].y;
          }
        };
        read(x, 0);
        int q = 0;
        for (; q + 2 <= parts; q += 2) {
          read(y, q + 1);
          add(x);
          read(x, q + 2 < parts ? q + 2 : q);
          add(y);
        }
        if (q < parts) add(x);
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    if (sum < 3) s_sum[sum][al] = acc;
  }
  __syncthreads();
  if (tid < kGroup && a_raw < n_assign) {
    // counts: onto the carried sums as so many ones
    const double t_trans = add_ones(init ? init[a * 6 + 3] : 0.0, s_count[0][tid]);
    double forbidden = init ? init[a * 6 + 5] : 0.0;
    if (n_edges > 0) forbidden += 0.0;  // a walk adds 0.0 or 1.0 per edge: a carried -0.0 loses its sign
    forbidden = add_ones(forbidden, s_count[1][tid]);
    const double t_compute = s_sum[0][tid], t_comm = s_sum[1][tid];
    double* r = out + a * 6;
    r[0] = (t_compute + t_comm) + t_trans;
    r[1] = t_compute;
    r[2] = t_comm;
    r[3] = t_trans;
    r[4] = s_sum[2][tid];
    r[5] = forbidden;
  }
}

template <bool kRandom, int kShift, bool kLists, int kUnroll, bool kTwo, typename... Args>
int launch_terms_k(int64_t n_assign, hipStream_t stream, Args... args) {
  constexpr int kLds = 2 * kTermLanes * kUnroll * 3 * 8;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(score_terms_kernel<kRandom, kShift, kLists, kUnroll, kTwo>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  if (e != hipSuccess) return fail(APC_ERR_LAUNCH, "hipFuncSetAttribute(score_terms_kernel): %s", hipGetErrorString(e));
  const int fold_lanes = ((3 << kShift) + 63) / 64 * 64;
  hipLaunchKernelGGL((score_terms_kernel<kRandom, kShift, kLists, kUnroll, kTwo>),
                     dim3((unsigned)((n_assign + (1 << kShift) - 1) >> kShift)), dim3(kTermLanes + fold_lanes), kLds, stream,
                     args...);
  return check_launch("score_terms_kernel");
}

template <bool kRandom, bool kLists, typename... Args>
int launch_terms(int64_t n_assign, hipStream_t stream, Args... args) {
  // The smallest groups with a workgroup per CU: a tile's copies of records, and the additions, cost a group the same
  // however small.  In us, at 5 000, 8 000 and 12 000 explicit assignments of the Llama-3-8B graph 334, 347 and 574, in
  // groups half as large 422, 424 and 674.  Beyond 256 groups of 64 two workgroups share a CU, of one row a lane:
  // 32 768 random assignments 649 us, with two rows 917; 16 384 492, with one row 561.  Explicit ones take one row
  // everywhere: the choices of two do not fit the registers (8 000: 716).
  constexpr int kU = kRandom ? 2 : 1;
  if (n_assign > 16384) return launch_terms_k<kRandom, 6, kLists, 1, true>(n_assign, stream, args...);
  if (n_assign <= 256) return launch_terms_k<kRandom, 0, kLists, kU, false>(n_assign, stream, args...);
  if (n_assign <= 512) return launch_terms_k<kRandom, 1, kLists, kU, false>(n_assign, stream, args...);
  if (n_assign <= 1024) return launch_terms_k<kRandom, 2, kLists, kU, false>(n_assign, stream, args...);
  if (n_assign <= 2048) return launch_terms_k<kRandom, 3, kLists, kU, false>(n_assign, stream, args...);
  if (n_assign <= 4096) return launch_terms_k<kRandom, 4, kLists, kU, false>(n_assign, stream, args...);
  if (n_assign <= 8192) return launch_terms_k<kRandom, 5, kLists, kU, false>(n_assign, stream, args...);
  return launch_terms_k<kRandom, 6, kLists, kU, false>(n_assign, stream, args...);
}

}  // namespace

extern "C" int apc_score_terms(const apc_problem* p, const double* per_arg, const double* table, void* scratch,
                               const uint16_t* assign, uint64_t seed, int64_t first, int64_t n_assign,
                               const int32_t* node_gid, int32_t first_node, int32_t first_edge, int32_t clamp_inf,
                               const double* init, double* out, void* stream) {
  if (int rc = validate_problem(p)) return rc;
  if (n_assign <= 0) return 0;
  if (!per_arg || !scratch || !out || !p->node_multiplier || (p->table_size > 0 && !table))
    return fail(APC_ERR_INVALID, "apc_score_terms: null argument%s");
  if (first_node < 0 || first_node >= p->n_node || first_edge < 0 || first_edge >= p->n_edge)
    return fail(APC_ERR_INVALID, "apc_score_terms: nothing to score, or first_node or first_edge out of range%s");
  if ((n_assign >> 6) >= 0x7FFFFFFF) return fail(APC_ERR_INVALID, "apc_score_terms: too many assignments for one launch%s");
  const int n_edges = p->n_edge - first_edge, n_nodes = p->n_node - first_node;
  FoldEdge* const edges = static_cast<FoldEdge*>(scratch);
  FoldNode* const nodes = reinterpret_cast<FoldNode*>(edges + n_edges);
  const int n_max = n_edges > n_nodes ? n_edges : n_nodes;
  hipLaunchKernelGGL(fold_records_kernel, dim3((unsigned)((n_max + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     (hipStream_t)stream, *p, table, node_gid, (int)first_node, (int)first_edge, assign == nullptr, edges,
                     nodes);
  if (int rc = check_launch("fold_records_kernel")) return rc;
#define APC_TERMS(R, L)                                                                                                \
  launch_terms<R, L>(n_assign, (hipStream_t)stream, (const FoldEdge*)edges, n_edges, (const FoldNode*)nodes, n_nodes,  \
                     per_arg, p->list_uidx, (int)clamp_inf, assign, n_assign, seed, first, n_assign, init, out)
  const bool lists = p->list_uidx != nullptr;
  if (assign) return lists ? APC_TERMS(false, true) : APC_TERMS(false, false);
  return lists ? APC_TERMS(true, true) : APC_TERMS(true, false);
#undef APC_TERMS
}

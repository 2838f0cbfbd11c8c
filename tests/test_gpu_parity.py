"""Parity of the HIP path (through the C ABI) against the CPU oracle and the
golden vectors written by the reference's own cost functions.

Bar: bit-exact for every fp64 cost entry and every flag (the north-star
tolerance is 1e-9 relative; the kernels restate the same binary64 operations
in the same order, so equality of bit patterns is what is asserted)."""
import json

import numpy as np
import pytest
import torch

from autoparallel_amd import graphgen, opprog, packed
from autoparallel_amd.packed import GraphBuilder, NodeDesc
from helpers import bits_equal, first_mismatch, graph_from_pairs
from oracle import cost_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def CostEngine():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from autoparallel_amd.engine import CostEngine as CE

    return CE


def _check_build(CE, g, use_table, clamp=False):
    print(f"  build: E={g.num_entries} table={use_table}", flush=True)
    # use_table: True / False, or the name of a table mode
    kw = dict(table_mode=use_table) if isinstance(use_table, str) else dict(use_table=use_table)
    eng = CE(g, **kw).build(clamp_inf=clamp)
    if isinstance(use_table, str):
        assert eng.table_mode == use_table
    got = eng.results()
    ref = O.GraphOracle(g).build()
    want_cost = O.clamp_inf(ref["cost"])[0] if clamp else ref["cost"]
    assert bits_equal(got["compute"], ref["compute"]), first_mismatch(got["compute"], ref["compute"])
    assert bits_equal(got["comm"], ref["comm"]), first_mismatch(got["comm"], ref["comm"])
    assert bits_equal(got["cost"], want_cost), first_mismatch(got["cost"], want_cost)
    assert ((got["flags"] & 1) == ref["transition"]).all()
    assert (((got["flags"] >> 1) & 1) == ~np.isfinite(ref["cost"])).all()
    return eng, got, ref


# ---------------------------------------------------------------------------
# golden vectors of the reference, through the C ABI
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("lut", [False, True])
@pytest.mark.parametrize("use_table", [True, False, "compressed"])
def test_golden_comm_vectors(CostEngine, golden, use_table, lut):
    n_cases = int(golden["comm_ncases"][0])
    checked = 0
    for k in range(n_cases):
        mesh = [int(x) for x in golden[f"comm_{k}_mesh"]]
        shape = [int(x) for x in golden[f"comm_{k}_shape"]]
        stride = [int(x) for x in golden[f"comm_{k}_stride"]]
        itemsize = int(golden[f"comm_{k}_itemsize"][0])
        src, tgt, want = golden[f"comm_{k}_src"], golden[f"comm_{k}_tgt"], golden[f"comm_{k}_cost"]
        src_t = sorted({tuple(int(x) for x in r) for r in src})
        tgt_t = sorted({tuple(int(x) for x in r) for r in tgt})
        g = graph_from_pairs(mesh, 8, shape, stride, itemsize, src_t, tgt_t)
        print(f"golden case {k}: mesh={mesh} shape={shape} pairs={len(want)}", flush=True)
        kw = dict(table_mode=use_table) if isinstance(use_table, str) else dict(use_table=use_table)
        eng = CostEngine(g, lut=lut, **kw).build(clamp_inf=False)  # lut: per-source terms in LDS, or the fold per element
        comm = eng.results()["comm"]
        e = 1  # the consumer's edge
        base, ssrc = int(g.edge_off[e]), int(g.edge_ssrc[e])
        si = {t: i for i, t in enumerate(src_t)}
        ti = {t: i for i, t in enumerate(tgt_t)}
        idx = np.asarray([base + ti[tuple(int(x) for x in t)] * ssrc + si[tuple(int(x) for x in s)]
                          for s, t in zip(src, tgt)])
        assert bits_equal(comm[idx], want), (k, first_mismatch(comm[idx], want))
        checked += len(want)
    assert checked > 20000


def test_golden_runtime_vectors(CostEngine, golden):
    """estimate_strategy_runtime_cost of the reference on hand-built fx nodes."""
    d = json.loads(bytes(golden["rt_json"]).decode())
    DT = {"torch.float64": (0, 8), "torch.float32": (1, 4), "torch.float16": (2, 2),
          "torch.bfloat16": (3, 2), "torch.int8": (4, 1), "torch.int64": (5, 8)}
    progs = {
        "mm": lambda s, i: opprog.mm(i), "mm_f32": lambda s, i: opprog.mm(i),
        "bmm": lambda s, i: opprog.bmm(i), "addmm": lambda s, i: opprog.addmm(i),
        "add": lambda s, i: opprog.pointwise(len(s[0]), i),
        "mul_bcast": lambda s, i: opprog.pointwise(len(s[0]), i),
        "small_add": lambda s, i: opprog.pointwise(len(s[0]), i),
        "silu": lambda s, i: opprog.pointwise(len(s[0]), i),
        "sum_dim": lambda s, i: opprog.reduction(len(s[0]), [2], True, i),
        "mean_dim": lambda s, i: opprog.reduction(len(s[0]), [-1], True, i),
        "einsum_fwd": lambda s, i: opprog.einsum_fwd(len(s[0]), i),
        "einsum_bwd": lambda s, i: opprog.einsum_bwd(len(s[0]), i),
        "softmax": lambda s, i: opprog.same_as_arg(0, len(s[0]), i),
        "embedding": lambda s, i: opprog.embedding(len(s[1]), i),
        "sdpa_flash": lambda s, i: opprog.sdpa_flash_fwd(i),
        "view": lambda s, i: None,
    }
    b = GraphBuilder(d["mesh"], 8)
    want = []
    # group the cases of one op into one node (one strategy per case)
    by_op = {}
    for i, name in enumerate(d["names"]):
        by_op.setdefault(name, []).append(i)
    for name, idxs in by_op.items():
        shapes, dtypes = d["shapes"][idxs[0]], d["dtypes"][idxs[0]]
        metas = []
        for shape, dt in zip(shapes, dtypes):
            stride = list(torch.empty(shape, device="meta").stride())
            metas.append(b.meta(shape, stride, DT[dt][1], DT[dt][0]))
        # producers: one placeholder-like node per argument, with the strategies' specs
        prods = []
        for a, m in enumerate(metas):
            specs = [b.spec(m, d["placements"][i][a]) for i in idxs]
            uniq = list(dict.fromkeys(specs))
            prods.append(b.add_node(NodeDesc(f"{name}_arg{a}", in_specs=[[s] for s in uniq],
                                             out_specs=[[s] for s in uniq], inputs=[],
                                             default_rows=[[[0.0]] for _ in uniq])))
        in_specs = [[b.spec(m, d["placements"][i][a]) for a, m in enumerate(metas)] for i in idxs]
        prog = progs[name](shapes, DT[dtypes[0]][1])
        b.add_node(NodeDesc(name, in_specs=in_specs, out_specs=[[r[0]] for r in in_specs], inputs=prods,
                            op=packed.OP_PROGRAM if prog is not None else packed.OP_ZERO, program=prog))
        want.append((len(b.nodes) - 1, [float.fromhex(d["cost_hex"][i]) for i in idxs]))
    b.share_compute_slots = False
    g = b.pack()
    eng = CostEngine(g).build(clamp_inf=False)
    compute = eng.results()["compute"]
    for v, vals in want:
        off = int(g.node_comp_off[v])
        got = compute[off:off + len(vals)]
        assert bits_equal(got, np.asarray(vals)), (g.node_names[v], got, vals)


# ---------------------------------------------------------------------------
# whole graphs against the oracle
# ---------------------------------------------------------------------------
GRAPHS = {
    "llama_2d": lambda: graphgen.llama_graph((8, 8), 1, 1024, 8, 4, 2048, 8192, 512, 16),
    "llama_2d_real_dims": lambda: graphgen.llama_graph((8, 8), 1, 4096, 32, 8, 14336, 128256, 8192, 64),
    "gpt2_1d": lambda: graphgen.gpt2_graph((8,), n_layers=2),
    "llama_3d": lambda: graphgen.llama_graph((2, 4, 2), 1, 512, 8, 4, 1024, 4096, 256, 16),
    "llama_odd_mesh": lambda: graphgen.llama_graph((3, 5), 1, 960, 15, 5, 1920, 3000, 240, 30),
    "stress_3d": lambda: graphgen.stress_graph(150, (4, 8, 8), seed=1, s_max=48),
    "llama70b_1layer_3d": lambda: graphgen.config_llama3_70b(1),  # config 3 dims on (4,8,8)
    "moe_1layer_real_dims": lambda: graphgen.config_moe(1),  # config 4 dims on (8,8), local_map nodes
    "moe_tiny": lambda: graphgen.moe_graph((2, 4), 2, 64, 4, 8, 2, 32, 256, 32, 8),
    "pairs_4d": lambda: _pairs_graph((2, 3, 2, 4), (48, 36, 40), 300),
    "pairs_3d_noncontig": lambda: _pairs_graph((4, 8, 8), (256, 8192, 64), 250, stride=(64, 16384, 1)),
}


def _pairs_graph(mesh, shape, n, stride=None, seed=3):
    """One edge whose rows/columns are random placement tuples over
    {R, S(d), P(sum), P(avg)} on a mesh of any rank."""
    rng = np.random.default_rng(seed)
    opts = [0x00] + [0x40 | d for d in range(len(shape))] + [0x80, 0x81]
    draw = lambda: sorted({tuple(int(x) for x in rng.choice(opts, size=len(mesh))) for _ in range(n)})
    if stride is None:
        stride = graphgen.contiguous_stride(shape)
    return graph_from_pairs(mesh, 8, shape, stride, 2, draw(), draw(), dtype=packed.DT_BF16)


# every graph through the table path; direct evaluation and the compressed
# table (matrices by distinct spec word, read by gather) on the smaller ones
CASES = [(n, True) for n in GRAPHS] + [
    (n, False) for n in ("llama_2d", "gpt2_1d", "llama_odd_mesh", "stress_3d", "pairs_4d", "pairs_3d_noncontig",
                         "moe_tiny")
] + [
    (n, "compressed") for n in ("llama_2d", "gpt2_1d", "llama_3d", "stress_3d", "moe_tiny", "pairs_3d_noncontig")
]


@pytest.mark.parametrize("name,use_table", CASES)
def test_graph_parity(CostEngine, name, use_table):
    g = GRAPHS[name]()
    print(f"graph {name}", flush=True)
    _check_build(CostEngine, g, use_table)


def test_moe_local_map_nodes_and_dispatch_volume(CostEngine):
    """Config 4: the routed-expert region is a single-strategy node priced at
    zero compute whose inputs are redistributed into the declared placements;
    the Zipf-weighted dispatch all-to-all is priced by the collective entry
    point (benchmark extension, not part of the entry parity)."""
    import ctypes as C

    from autoparallel_amd import _lib
    from autoparallel_amd.engine import make_model

    g = graphgen.config_moe(1)
    eng, got, ref = _check_build(CostEngine, g, True)
    lm = [v for v, n in enumerate(g.node_names) if n.startswith("local_map_moe")]
    assert len(lm) == 2  # forward and backward region
    for v in lm:
        assert int(g.node_nstrat[v]) == 1 and int(g.node_op[v]) == packed.OP_ZERO
        assert got["compute"][int(g.node_comp_off[v])] == 0.0
        for e in range(int(g.node_edge_off[v]), int(g.node_edge_off[v + 1])):
            blk = got["comm"][int(g.edge_off[e]): int(g.edge_off[e]) + int(g.edge_ssrc[e])]
            assert np.isfinite(blk).any() and (blk[np.isfinite(blk)] >= 0).all()
            assert (blk == 0).any()  # the producer can already hold the declared placement
    nbytes = graphgen.moe_dispatch_bytes(16, 64, 6, 32 * 4096, 2048, 2, 8, 8, seed=0)
    assert nbytes.shape == (16,) and (nbytes > 0).all()
    lib = _lib.load()
    m = make_model((8, 8), 8, "AMD Instinct MI355X")
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    kind, dim = d(np.full(16, 1, np.int32)), d(np.full(16, 1, np.int32))
    nb, out = d(nbytes), torch.empty(16, dtype=torch.float64, device="cuda")
    assert lib.apc_collective_costs(C.byref(m), 16, kind.data_ptr(), nb.data_ptr(), dim.data_ptr(), out.data_ptr(), None) == 0
    torch.cuda.synchronize()
    topo = O.Topo((8, 8), 8)
    want = np.asarray([O.collective_comm_cost("all_to_all", int(b), topo, 1) for b in nbytes])
    assert bits_equal(out.cpu().numpy(), want)


def test_graph_replay_matches_eager(CostEngine):
    """The build captured in a HIP graph: every replay, with eager work and
    synchronisations in between, gives the eager bits."""
    g = GRAPHS["llama_2d"]()
    eng = CostEngine(g)
    eng.build(clamp_inf=True)
    want = {k: v.copy() for k, v in eng.results().items()}
    graph = eng.capture_build(clamp_inf=True)
    for rep in range(4):
        for t in (eng.comm, eng.cost, eng.compute, eng.per_arg):
            t.fill_(-1.0)
        eng.flags.fill_(255)
        if eng.table is not None:
            eng.table.fill_(-7.0)
        torch.cuda.synchronize()
        graph.replay()
        got = eng.results()
        slots = g.entry_slots()
        for k in ("comm", "cost", "flags"):
            assert bits_equal(got[k][slots], want[k][slots]), (rep, k)
        assert bits_equal(got["compute"], want["compute"]) and bits_equal(got["per_arg"], want["per_arg"])
        # eager work between replays
        eng.build(clamp_inf=False)
        torch.cuda.synchronize()


def test_timed_launch_is_the_same_launch(CostEngine):
    import ctypes as C

    g = GRAPHS["llama_2d"]()
    eng = CostEngine(g).build(clamp_inf=True)
    want = eng.results()
    timer = C.c_void_p()
    assert eng.lib.apc_timer_create(3, C.byref(timer)) == 0
    eng.cost.fill_(-1.0)
    for k in range(3):
        eng.edge_costs_timed(timer, k, clamp_inf=True)
    got = eng.results()
    slots = g.entry_slots()
    assert bits_equal(got["cost"][slots], want["cost"][slots])
    ms = C.c_float()
    for k in range(3):
        assert eng.lib.apc_timer_elapsed_ms(timer, k, C.byref(ms)) == 0
        assert 0.0 < ms.value < 100.0
    assert eng.lib.apc_timer_elapsed_ms(timer, 3, C.byref(ms)) != 0  # slot out of range
    with pytest.raises(Exception):
        eng.edge_costs_timed(timer, 7)
    assert eng.lib.apc_timer_destroy(timer) == 0


def test_clamp_inf(CostEngine):
    _check_build(CostEngine, GRAPHS["llama_2d"](), True, clamp=True)


def test_deterministic(CostEngine):
    g = GRAPHS["llama_2d"]()
    a = CostEngine(g).build().results()
    b = CostEngine(g).build().build().results()
    for k in ("comm", "cost", "compute"):
        assert bits_equal(a[k], b[k])
    assert (a["flags"] == b["flags"]).all()


def test_prefetch_discount(CostEngine):
    g = GRAPHS["llama_2d"]()
    for scale in (0.0, 0.25):
        eng, got, ref = _check_build(CostEngine, g, True, clamp=True)
        n = eng.apply_prefetch_discount(scale)
        cost0, _ = O.clamp_inf(ref["cost"])
        comm2, cost2, n2 = O.prefetch_discount(g, ref["comm"], ref["transition"], ref["compute"], cost0, scale)
        got2 = eng.results()
        assert n == n2 > 0
        assert bits_equal(got2["comm"], comm2) and bits_equal(got2["cost"], cost2)


def test_objective_coeffs(CostEngine):
    g = GRAPHS["gpt2_1d"]()
    g.node_multiplier = (np.arange(g.num_nodes) % 3 + 1).astype(np.int32)
    eng, got, ref = _check_build(CostEngine, g, True, clamp=True)
    obj = eng.objective_coeffs().cpu().numpy()
    slots, keys = g.entry_slots(), g.entry_keys()
    want = got["cost"][slots] * g.node_multiplier[keys[:, 0]]
    assert bits_equal(obj[slots], want)


def test_scoring(CostEngine):
    g = GRAPHS["llama_2d"]()
    eng, got, ref = _check_build(CostEngine, g, True, clamp=True)
    rng = np.random.default_rng(1)
    A = 37
    assign = np.stack([rng.integers(0, g.node_nstrat) for _ in range(A)], axis=1).astype(np.int16)
    assign[:, 0] = 0
    out = eng.score(torch.from_numpy(np.ascontiguousarray(assign)).cuda()).cpu().numpy()
    cost, bad = O.clamp_inf(ref["cost"])
    for a in range(A):
        want = O.score_assignment(g, ref["comm"], ref["transition"], ref["compute"], assign[:, a])
        obj, viol = O.ilp_objective(g, cost, bad, assign[:, a])
        assert tuple(out[a, :4]) == tuple(float(x) for x in want), (a, out[a], want)
        assert out[a, 4] == obj and out[a, 5] == viol
    # large batches take the lane-per-assignment kernel: same bits as the wave kernel
    big = np.tile(assign, (1, 900))[:, :33000]
    out_big = eng.score(torch.from_numpy(np.ascontiguousarray(big)).cuda()).cpu().numpy()
    assert bits_equal(out_big[:A].ravel(), out.ravel()) and bits_equal(out_big[A:2 * A].ravel(), out.ravel())
    r_small = eng.score_random(seed=3, first=0, count=50).cpu().numpy()
    r_big = eng.score_random(seed=3, first=0, count=33000).cpu().numpy()
    assert bits_equal(r_big[:50].ravel(), r_small.ravel())
    # on-device generated assignments: same draw on the host
    out = eng.score_random(seed=11, first=5, count=9).cpu().numpy()
    for i in range(9):
        asg = eng.random_assignment(11, 5 + i)
        assert (asg < g.node_nstrat).all()
        want = O.score_assignment(g, ref["comm"], ref["transition"], ref["compute"], asg)
        assert tuple(out[i, :4]) == tuple(float(x) for x in want)


def test_device_scorers_on_a_hand_made_plan(CostEngine):
    """Every device scorer against totals worked out by hand from the text of the reference's
    _compute_solution_cost (helpers.hand_made_plan): the entry arrays of an engine are overwritten with
    the literal numbers of that case, so nothing of the cost model is involved."""
    from helpers import hand_made_plan

    g, comm, transition, compute, assign, want = hand_made_plan()
    eng = CostEngine(g, use_table=False).build(clamp_inf=True)
    nargs = np.repeat(g.node_nargs, 2).astype(np.float64)
    per_arg = compute / nargs
    eng.per_arg.copy_(torch.from_numpy(per_arg))
    eng.compute.copy_(torch.from_numpy(compute))
    eng.comm.copy_(torch.from_numpy(comm))
    # cost as the build forms it, (comm + per_arg) + transition, clamped; flags: transition | non-finite << 1
    cost = np.zeros(g.num_slots)
    flags = transition.copy()
    for e in range(g.num_edges):
        v, off, ssrc, sdst = int(g.edge_node[e]), int(g.edge_off[e]), int(g.edge_ssrc[e]), int(g.edge_sdst[e])
        for o in range(sdst):
            for j in range(ssrc):
                c = (comm[off + o * ssrc + j] + per_arg[int(g.node_comp_off[v]) + o]) + float(transition[off + o * ssrc + j])
                if not np.isfinite(c):
                    c, flags[off + o * ssrc + j] = 10000.0, flags[off + o * ssrc + j] | 2
                cost[off + o * ssrc + j] = c
    eng.cost.copy_(torch.from_numpy(cost))
    eng.flags.copy_(torch.from_numpy(flags))
    eng.mark_results_edited()
    # objective: the selected cost of every argument row, placeholders' own rows included;
    # one selected variable is forbidden (C <- Q)
    obj = 2.0 + 4.0 + (0.5 + 16.0) + 10000.0 + (0.25 + 64.0 + 1.0) + (0.125 + 256.0 + 1.0)
    col = np.asarray(assign, np.int16)[:, None]
    for count in (1, 70, 33000, 140000):  # terms side by side, lanes over records
        out = eng.score(torch.from_numpy(np.ascontiguousarray(np.tile(col, (1, count)))).cuda()).cpu().numpy()
        assert tuple(out[0, :4]) == want and tuple(out[-1, :4]) == want, (count, eng.last_score_backend, out[0])
        assert out[0, 4] == obj and out[0, 5] == 1.0 and bits_equal(out[0], out[-1])


def test_scoring_from_interleaved_records(CostEngine, monkeypatch):
    """apc_score_packed against the scorers that read the three entry arrays:
    explicit assignments, drawn ones, a window with continued sums; and the
    records follow the entry arrays when those are rewritten.  (The scorers
    that come before it for a graph with large blocks are switched off here;
    test_gpu_scoring_large_blocks.py covers them.)"""
    from autoparallel_amd import engine as engine_mod

    monkeypatch.setattr(engine_mod, "_SCORE_FROM_TABLE", False)
    monkeypatch.setattr(engine_mod, "_SCORE_COMPACT", False)
    for name in ("stress_3d", "llama_2d"):
        g = GRAPHS[name]()
        eng = CostEngine(g).build(clamp_inf=True)
        n = 40000
        rng = np.random.default_rng(2)
        assign = np.stack([rng.integers(0, g.node_nstrat) for _ in range(64)], axis=1).astype(np.int16)
        big = torch.from_numpy(np.ascontiguousarray(np.tile(assign, (1, n // 64 + 1))[:, :n])).cuda()
        gid = np.arange(g.num_nodes, dtype=np.int32) + 1000
        half = torch.rand(n, 6, dtype=torch.float64, device="cuda")

        def run():
            return [eng.score(big), eng.score_random(3, 5, n), eng.score_random_window(3, 0, n, gid, 7, init=half)]

        eng.packed_scoring = False
        want = run()
        eng.packed_scoring = True
        got = run()
        for a, b in zip(got, want):
            assert torch.equal(a.view(torch.int64), b.view(torch.int64))
        assert eng._recs_valid
        if name == "llama_2d":
            eng = CostEngine(g).build(clamp_inf=True)
            eng.packed_scoring = True
            before = eng.score_random(3, 5, n)
            assert eng.apply_prefetch_discount(0.25) > 0 and not eng._recs_valid
            after = eng.score_random(3, 5, n)
            eng.packed_scoring = False
            assert torch.equal(after.view(torch.int64), eng.score_random(3, 5, n).view(torch.int64))
            assert not torch.equal(after, before)


# ---------------------------------------------------------------------------
# edge cases
# ---------------------------------------------------------------------------
def _edge_case_graph():
    """Missing specs with default rows, a tuple-valued producer consumed
    directly and through getitem, an explicit-flops node, a node with more than
    8 arguments, strategies > 64, single-entry blocks."""
    b = GraphBuilder((2, 4), 8)
    m = b.meta((64, 48), (48, 1), 2, packed.DT_BF16)
    mt = b.meta((64, 48), (1, 64), 2, packed.DT_BF16)
    opts = O.create_all_options((64, 48), (2, 4))
    specs = [b.spec(m, o) for o in opts]
    ph = b.add_node(NodeDesc("x", in_specs=[[s] for s in specs], out_specs=[[s] for s in specs],
                             inputs=[], default_rows=[[[0.0]] for _ in specs]))
    one = b.add_node(NodeDesc("scalar", in_specs=[[specs[0]]], out_specs=[[specs[0]]], inputs=[],
                              default_rows=[[[0.0]]]))
    # tuple producer: two outputs, second one None in some strategies
    tup_out = [[s, (b.spec(mt, o) if i % 3 else -1)] for i, (s, o) in enumerate(zip(specs, opts))]
    tup = b.add_node(NodeDesc("tuple_op", in_specs=[[s] for s in specs], out_specs=tup_out, inputs=[ph],
                              op=packed.OP_PROGRAM, program=opprog.same_as_arg(0, 2, 2, n_out=2),
                              tuple_output=True))
    uniq1 = list(dict.fromkeys(o[1] for o in tup_out))
    gi = b.add_node(NodeDesc("getitem1", in_specs=[[s] for s in uniq1], out_specs=[[s] for s in uniq1],
                             inputs=[tup], getitem_index=1,
                             default_rows=[[[float(i + j) for j in range(len(specs))]] for i in range(len(uniq1))]))
    direct = b.add_node(NodeDesc("uses_tuple", in_specs=[[specs[0]], [specs[1]]], out_specs=[[specs[0]], [specs[1]]],
                                 inputs=[tup],
                                 default_rows=[[[1.5] * len(specs)], [[2.5] * len(specs)]]))
    # explicit flops/bytes, with a None input spec (non-tensor arg)
    b.add_node(NodeDesc("explicit", in_specs=[[specs[0], -1], [specs[2], -1]], out_specs=[[specs[0]], [specs[2]]],
                        inputs=[ph, one], op=packed.OP_EXPLICIT, flops=[10**12, 0], nbytes=[10**9, 10**3],
                        default_rows=[[[0.0] * len(specs), [7.0]], [[0.0] * len(specs), [8.0]]]))
    # 10 arguments: beyond the staged fast path of the node kernel
    b.add_node(NodeDesc("many_args", in_specs=[[s] * 10 for s in specs[:5]], out_specs=[[s] for s in specs[:5]],
                        inputs=[ph] * 10, op=packed.OP_PROGRAM, program=opprog.pointwise(2, 2)))
    # > 64 strategies on both sides
    big = [specs[i % len(specs)] for i in range(150)]
    pb = b.add_node(NodeDesc("big_prod", in_specs=[[s] for s in big], out_specs=[[s] for s in big], inputs=[ph],
                             op=packed.OP_PROGRAM, program=opprog.pointwise(2, 2)))
    b.add_node(NodeDesc("big_cons", in_specs=[[s, s] for s in big[:131]], out_specs=[[s] for s in big[:131]],
                        inputs=[pb, pb], op=packed.OP_PROGRAM, program=opprog.mm(2)))
    return b.pack()


@pytest.mark.parametrize("use_table", [True, False, "compressed"])
def test_edge_cases(CostEngine, use_table):
    g = _edge_case_graph()
    eng, got, ref = _check_build(CostEngine, g, use_table)
    # the default rows really were used
    e = [i for i in range(g.num_edges) if g.node_names[g.edge_node[i]] == "uses_tuple"][0]
    b0 = int(g.edge_off[e])
    assert got["comm"][b0] == 1.5


@pytest.mark.parametrize("mode", ["full", "compressed"])
def test_work_items_of_512_entries(CostEngine, mode):
    """Large problems use work items of 512 entries: same bits."""
    for make in (GRAPHS["llama_2d"], GRAPHS["stress_3d"], _edge_case_graph):
        g = make()
        eng = CostEngine(g, table_mode=mode, item_entries=512).build(clamp_inf=False)
        assert eng.problem.item_entries == 512
        assert eng.problem.n_item < CostEngine(g, table_mode=mode, item_entries=256).problem.n_item
        got = eng.results()
        ref = O.GraphOracle(g).build()
        assert bits_equal(got["comm"], ref["comm"]) and bits_equal(got["cost"], ref["cost"])
        assert ((got["flags"] & 1) == ref["transition"]).all()
    from autoparallel_amd import _lib
    with pytest.raises(_lib.ApcError):
        CostEngine(g, table_mode="direct", item_entries=512, lut=False).build()


def _sized_blocks_graph(sizes):
    """A chain of producer/consumer pairs whose edge blocks have the given (S_src, S_dst):
    rows shorter than, exactly and longer than a wavefront, single rows and single columns,
    behind small blocks, so that blocks start at every offset inside a 64-slot group."""
    import itertools

    b = GraphBuilder((2, 2, 2, 2), 8)
    m = b.meta((8, 16, 32, 64), (32768, 2048, 64, 1), 4, packed.DT_F32)
    codes = [0x00, 0x40, 0x41, 0x42, 0x43, 0x80]
    tuples = list(itertools.product(codes, repeat=4))  # 1 296 distinct placement tuples
    rng = np.random.default_rng(7)
    for k, (ssrc, sdst) in enumerate(sizes):
        src = [b.spec(m, tuples[i]) for i in rng.choice(len(tuples), ssrc, replace=False)]
        dst = [b.spec(m, tuples[i]) for i in rng.choice(len(tuples), sdst, replace=False)]
        p = b.add_node(NodeDesc(f"p{k}", in_specs=[[x] for x in src], out_specs=[[x] for x in src], inputs=[],
                                default_rows=[[[0.0]] for _ in src]))
        b.add_node(NodeDesc(f"c{k}", in_specs=[[x] for x in dst], out_specs=[[x] for x in dst], inputs=[p]))
    return b.pack()


@pytest.mark.parametrize("mode", ["full", "compressed"])
@pytest.mark.parametrize("item_entries", [256, 512])
def test_entry_kernel_on_blocks_of_chosen_sizes(CostEngine, mode, item_entries):
    """The wave-per-item kernel picks the row values of an entry three ways (two candidate rows
    for rows of 64 entries and more, one lane per row below, a load per entry for items of more
    than 64 rows) and repeats an entry of the block in the lanes that fall outside it: blocks on
    every side of those limits, every entry against the oracle."""
    sizes = [(63, 5), (3, 2), (64, 7), (5, 1), (65, 9), (128, 1), (1, 300), (512, 3), (7, 200), (2, 700),
             (200, 64), (64, 64), (9, 60), (8, 65), (300, 2), (1, 1), (130, 130)]
    g = _sized_blocks_graph(sizes)
    assert len({int(o) % 64 for o in g.edge_off[:-1]}) >= 3  # blocks start at several offsets of a 64-slot group
    eng = CostEngine(g, table_mode=mode, item_entries=item_entries).build(clamp_inf=False)
    got = eng.results()
    ref = O.GraphOracle(g).build()
    assert bits_equal(got["comm"], ref["comm"]), first_mismatch(got["comm"], ref["comm"])
    assert bits_equal(got["cost"], ref["cost"]), first_mismatch(got["cost"], ref["cost"])
    assert ((got["flags"] & 1) == ref["transition"]).all()
    assert (((got["flags"] >> 1) & 1) == ~np.isfinite(ref["cost"])).all()


@pytest.mark.parametrize("mode", ["full", "compressed"])
@pytest.mark.parametrize("item_entries", [256, 512])
def test_entry_kernel_with_an_output_left_out(CostEngine, mode, item_entries):
    """With all three outputs apc_edge_costs runs a wavefront per work item, nothing
    predicated; with one left out, the loop kernel.  Same bits in what both write,
    and the one left out stays untouched."""
    for make in (GRAPHS["llama_2d"], GRAPHS["stress_3d"], _edge_case_graph):
        g = make()
        eng = CostEngine(g, table_mode=mode, item_entries=item_entries).build(clamp_inf=True)
        want = eng.results()
        slots = np.zeros(g.num_slots, bool)  # the slots that hold an entry; blocks are padded to 16
        for e in range(g.num_edges):
            slots[int(g.edge_off[e]): int(g.edge_off[e]) + int(g.edge_sdst[e]) * int(g.edge_ssrc[e])] = True
        for skip in (None, "comm", "flags"):
            eng.comm.fill_(-7.0)
            eng.cost.fill_(-7.0)
            eng.flags.fill_(0x55)
            eng.edge_costs(clamp_inf=True, want_comm=skip != "comm", want_flags=skip != "flags")
            got = eng.results()
            assert bits_equal(got["cost"][slots], want["cost"][slots])
            if skip == "comm":
                assert (got["comm"] == -7.0).all()
            else:
                assert bits_equal(got["comm"][slots], want["comm"][slots])
            if skip == "flags":
                assert (got["flags"] == 0x55).all()
            else:
                assert (got["flags"][slots] == want["flags"][slots]).all()
            # neither kernel writes between the blocks (the lanes of the unpredicated one that
            # fall outside a block repeat an entry of the block)
            assert (got["cost"][~slots] == -7.0).all() and (got["flags"][~slots] == 0x55).all()


@pytest.mark.parametrize("rank,n_args", [(1, 15), (2, 16)])
def test_more_arguments_than_the_node_record_holds(CostEngine, rank, n_args):
    """Arguments past the 14 runs kept in a node's record are found through the
    edge table: with rank-1 tensors the local sizes are still staged in LDS, with
    rank 2 and 16 arguments they are read on demand."""
    b = GraphBuilder((2, 4), 8)
    shape = (64, 48)[:rank]
    m = b.meta(shape, graphgen.contiguous_stride(shape), 2, packed.DT_BF16)
    opts = O.create_all_options(shape, (2, 4))
    specs = [b.spec(m, o) for o in opts]
    phs = [b.add_node(NodeDesc(f"x{k}", in_specs=[[s] for s in specs], out_specs=[[s] for s in specs], inputs=[],
                               default_rows=[[[0.0]] for _ in specs])) for k in range(3)]
    rng = np.random.default_rng(rank)
    S = 40
    in_specs = [[specs[int(rng.integers(len(specs)))] for _ in range(n_args)] for _ in range(S)]
    out_specs = [[specs[int(rng.integers(len(specs)))]] for _ in range(S)]
    b.add_node(NodeDesc("wide", in_specs=in_specs, out_specs=out_specs,
                        inputs=[phs[k % 3] for k in range(n_args)], op=packed.OP_PROGRAM,
                        program=opprog.pointwise(rank, 2)))
    g = b.pack()
    assert g.max_node_args == n_args > packed.PackedGraph.REC_ARGS
    _check_build(CostEngine, g, True)
    _check_build(CostEngine, g, False)


@pytest.mark.parametrize("mode", ["full", "compressed"])
def test_problem_without_the_derived_records(CostEngine, mode):
    """A caller of the C ABI may leave out every record the host derives for the
    prepare launch (table units, spec records, product terms, node records): the
    kernels then walk the arrays those were made from.  Same bits either way."""
    g = graphgen.llama_graph((2, 2, 4), 1, 64, 4, 2, 128, 256, 32, 16)
    eng = CostEngine(g, table_mode=mode, lut=False).build(clamp_inf=False)  # the kernels with one element per lane
    want = eng.results()
    ref = O.GraphOracle(g).build()
    assert bits_equal(want["comm"], ref["comm"]) and bits_equal(want["compute"], ref["compute"])
    for drop in (("table_units",), ("spec_recs",), ("prog_terms", "n_prog_term"),
                 ("comp_recs",), ("table_units", "spec_recs", "prog_terms", "n_prog_term", "comp_recs")):
        e2 = CostEngine(g, table_mode=mode, lut=False)
        for f in drop:
            setattr(e2.problem, f, 0 if f == "n_prog_term" else None)
        got = e2.build(clamp_inf=False).results()
        for k in ("comm", "cost", "compute", "per_arg"):
            assert bits_equal(got[k], want[k]), (drop, k, first_mismatch(got[k], want[k]))
        assert (got["flags"] == want["flags"]).all()


def test_node_program_paths(CostEngine):
    """The node estimate by product terms, by the interpreter (a term over more
    factors than a term record names), with an argument whose strategies see
    different tensors (the record's meta hint then misses), a missing spec and a
    broadcast output, all in one graph."""
    b = GraphBuilder((2, 4), 8)
    big = (4,) * 8
    m8 = b.meta(big, graphgen.contiguous_stride(big), 2, packed.DT_BF16)
    ma = b.meta((64, 48), (48, 1), 2, packed.DT_BF16)
    mb = b.meta((64, 1), (1, 1), 4, packed.DT_F32)
    mc = b.meta((32, 48), (48, 1), 2, packed.DT_BF16)
    o8 = [b.spec(m8, o) for o in O.create_all_options(big, (2, 4))[:12]]
    oa = [b.spec(ma, o) for o in O.create_all_options((64, 48), (2, 4))]
    ob = [b.spec(mb, o) for o in O.create_all_options((64, 1), (2, 4))]
    oc = [b.spec(mc, o) for o in O.create_all_options((32, 48), (2, 4))]
    x8 = b.add_node(NodeDesc("x8", [[s] for s in o8], [[s] for s in o8], inputs=[], default_rows=[[[0.0]] for _ in o8]))
    xa = b.add_node(NodeDesc("xa", [[s] for s in oa], [[s] for s in oa], inputs=[], default_rows=[[[0.0]] for _ in oa]))
    xb = b.add_node(NodeDesc("xb", [[s] for s in ob], [[s] for s in ob], inputs=[], default_rows=[[[0.0]] for _ in ob]))
    # eight factors in one term: interpreted word by word
    prog8 = opprog.program([(2, [(0, d) for d in range(8)])], [(2, [opprog.argnumel(0)])])
    b.add_node(NodeDesc("eight", [[s] for s in o8], [[s] for s in o8], inputs=[x8], op=packed.OP_PROGRAM, program=prog8))
    # broadcast add of [64, 48] and [64, 1]; argument 0 sees tensor ma or mc by strategy
    mixed = [[(oa + oc)[k % (len(oa) + len(oc))], ob[k % len(ob)], -1] for k in range(70)]
    rows = [[[0.0] * len(oa), [0.0] * len(ob), [0.0]] for _ in range(70)]
    b.add_node(NodeDesc("bcast_add", mixed, [[r[0]] for r in mixed], inputs=[xa, xb, None], op=packed.OP_PROGRAM,
                        program=opprog.pointwise(2, 2), default_rows=rows, nargs=3))
    g = b.pack()
    rec = g.comp_records()
    by_node = {int(r["node"]): r for r in rec}
    assert by_node[3]["n_term"] == 0 and by_node[4]["n_term"] > 0 and by_node[4]["term_flags"] & 1
    for mode in (True, False, "compressed"):
        _check_build(CostEngine, g, mode)


@pytest.mark.parametrize("mode", ["full", "direct"])
def test_xgmi_topology_on_the_device(CostEngine, mode):
    """With the xGMI link constants selected, the device and the oracle still
    agree bit for bit, every all_to_all entry changes and nothing else does
    that has no collective on a dim whose constants moved."""
    from autoparallel_amd import cost_models as cm

    cfg = cm.mi355x_topo_config()
    g = graphgen.llama_graph((8, 8), 1, 1024, 8, 4, 2048, 8192, 512, 16)
    got = CostEngine(g, table_mode=mode, topo_config=cfg).build(clamp_inf=False).results()
    ref = O.GraphOracle(g, xgmi=cfg).build()
    assert bits_equal(got["comm"], ref["comm"]), first_mismatch(got["comm"], ref["comm"])
    assert bits_equal(got["cost"], ref["cost"])
    plain = O.GraphOracle(g).build()
    assert bits_equal(got["compute"], plain["compute"])  # the compute estimate does not see the links
    finite = np.isfinite(plain["comm"])
    assert (ref["comm"][finite] != plain["comm"][finite]).any()
    assert ((ref["comm"] == 0) == (plain["comm"] == 0)).all() and (np.isfinite(ref["comm"]) == finite).all()


@pytest.mark.parametrize("name", ["llama_2d", "llama_3d", "llama_odd_mesh", "moe_tiny", "pairs_4d", "pairs_3d_noncontig",
                                  "stress_3d"])
def test_lookup_table_kernels(CostEngine, name):
    """The tile kernels (terms per source spec in LDS) against the oracle, for the
    block table in both layouts and for direct evaluation, with the inf clamp on
    the direct path; and the edge cases graph (missing specs, tuple outputs, default
    rows, an edge without a producer)."""
    g = GRAPHS[name]()
    ref = O.GraphOracle(g).build()
    for mode in ("full", "compressed", "direct"):
        eng = CostEngine(g, table_mode=mode, lut=True)
        assert eng._lut_tiles is not None
        got = eng.build(clamp_inf=False).results()
        assert bits_equal(got["comm"], ref["comm"]), (mode, first_mismatch(got["comm"], ref["comm"]))
        assert bits_equal(got["cost"], ref["cost"]), mode
        assert ((got["flags"] & 1) == ref["transition"]).all() and bits_equal(got["compute"], ref["compute"])
    clamped = CostEngine(g, table_mode="direct", lut=True).build(clamp_inf=True).results()
    assert bits_equal(clamped["cost"], O.clamp_inf(ref["cost"])[0])
    ge = _edge_case_graph()
    re_ = O.GraphOracle(ge).build()
    for mode in ("full", "compressed", "direct"):
        got = CostEngine(ge, table_mode=mode, lut=True).build(clamp_inf=False).results()
        assert bits_equal(got["comm"], re_["comm"]) and bits_equal(got["cost"], re_["cost"]), mode
        assert ((got["flags"] & 1) == re_["transition"]).all()


def test_build_all_takes_the_tile_route_from_the_problem(CostEngine):
    """One build entry point: apc_build_all through the C ABI with table == NULL
    evaluates by tiles when the problem carries lut_entry_tiles and entry by entry
    when it does not, and with a table builds it by tiles when the problem carries
    lut_table_tiles; the same bits each way, and as the entry points that take a
    tile list as an argument."""
    import ctypes as C

    import torch

    from autoparallel_amd import _lib

    g = graphgen.stress_graph(200, (4, 8, 8), seed=11, s_min=8, s_max=160)
    ref = O.GraphOracle(g).build()

    def run(eng, table):
        for t in (eng.comm, eng.cost, eng.flags):
            t.zero_()
        _lib.check(eng.lib.apc_build_all(
            C.byref(eng.problem), table, eng._ptr(eng.compute), eng._ptr(eng.per_arg), eng._ptr(eng.status),
            eng._ptr(eng.comm), eng._ptr(eng.cost), eng._ptr(eng.flags), 0, eng._stream()), "apc_build_all")
        eng.built = True
        return eng.results()

    for lut in (True, False):
        eng = CostEngine(g, table_mode="direct", lut=lut)
        assert (eng.problem.n_lut_entry_tile > 0) == lut and eng.problem.n_lut_table_tile == 0
        got = run(eng, None)
        assert bits_equal(got["comm"], ref["comm"]) and bits_equal(got["cost"], ref["cost"]), lut
        assert ((got["flags"] & 1) == ref["transition"]).all()
    # the explicit entry point with the same list
    eng = CostEngine(g, table_mode="direct", lut=True)
    eng.node_compute()
    tiles, n_tile = eng._lut_tiles
    for t in (eng.comm, eng.cost, eng.flags):
        t.zero_()
    _lib.check(eng.lib.apc_edge_costs_lut(C.byref(eng.problem), tiles, n_tile, eng._ptr(eng.per_arg), eng._ptr(eng.comm),
                                          eng._ptr(eng.cost), eng._ptr(eng.flags), 0, eng._stream()), "apc_edge_costs_lut")
    eng.built = True
    got = eng.results()
    assert bits_equal(got["comm"], ref["comm"]) and bits_equal(got["cost"], ref["cost"])
    for mode in ("full", "compressed"):
        tables = []
        for lut in (True, False):
            eng = CostEngine(g, table_mode=mode, lut=lut)
            assert (eng.problem.n_lut_table_tile > 0) == lut and eng.problem.n_lut_entry_tile == 0
            eng.table.zero_()  # the padding between matrices is nobody's to write
            got = run(eng, eng._ptr(eng.table))
            assert bits_equal(got["comm"], ref["comm"]) and bits_equal(got["cost"], ref["cost"]), (mode, lut)
            tables.append(eng.table.cpu().numpy())
        assert bits_equal(tables[0], tables[1]), mode
        torch.cuda.synchronize()


def test_unsupported_dtype_reports(CostEngine):
    b = GraphBuilder((2,), 8)
    m = b.meta((8, 8), (8, 1), 8, packed.DT_OTHER)
    s = b.spec(m, (0,))
    ph = b.add_node(NodeDesc("x", in_specs=[[s]], out_specs=[[s]], inputs=[], default_rows=[[[0.0]]]))
    b.add_node(NodeDesc("mm_i64", in_specs=[[s, s]], out_specs=[[s]], inputs=[ph, ph],
                        op=packed.OP_PROGRAM, program=opprog.mm(8)))
    eng = CostEngine(b.pack()).build()
    with pytest.raises(ValueError):
        eng.results()


def test_enumerate_input_options(CostEngine):
    import ctypes as C

    from autoparallel_amd import _lib
    from autoparallel_amd.engine import make_model

    lib = _lib.load()
    mesh = (4, 8, 8)
    shapes = [(256, 8192, 8192), (10, 3, 1000), (7,), (64, 32, 8192, 128), (), (4, 4)]
    model = make_model(mesh, 8, "AMD Instinct MI355X")
    rank = np.asarray([len(s) for s in shapes], np.int32)
    shp = np.ones((len(shapes), 8), np.int64)
    for i, s in enumerate(shapes):
        shp[i, :len(s)] = s
    ncand = (rank.astype(np.int64) + 1) ** len(mesh)
    off = np.zeros(len(shapes) + 1, np.int64)
    np.cumsum(ncand, out=off[1:])
    d = lambda a: torch.from_numpy(a).cuda()
    t_rank, t_shape, t_off = d(rank), d(shp), d(off)
    valid = torch.zeros(int(off[-1]), dtype=torch.uint8, device="cuda")
    plc = torch.zeros(int(off[-1]) * 4, dtype=torch.uint8, device="cuda")
    rc = lib.apc_enumerate_input_options(C.byref(model), len(shapes), t_rank.data_ptr(), t_shape.data_ptr(),
                                         t_off.data_ptr(), valid.data_ptr(), plc.data_ptr(), None)
    assert rc == 0
    torch.cuda.synchronize()
    valid, plc = valid.cpu().numpy(), plc.cpu().numpy().reshape(-1, 4)
    for i, s in enumerate(shapes):
        got = [tuple(int(x) for x in plc[j, :3]) for j in range(off[i], off[i + 1]) if valid[j]]
        assert got == O.create_all_options(s, mesh), s


# ---------------------------------------------------------------------------
# full benchmark size: properties that need no oracle pass over every entry
# ---------------------------------------------------------------------------
def test_full_size_properties(CostEngine):
    g = graphgen.config_llama3_8b()
    print(f"full size: E={g.num_entries}", flush=True)
    eng = CostEngine(g, use_table=True).build(clamp_inf=False)
    a = eng.results()
    d = CostEngine(g, use_table=False).build(clamp_inf=False).results()
    # table path and direct evaluation are the same function
    for k in ("comm", "cost", "compute"):
        assert bits_equal(a[k], d[k])
    assert (a["flags"] == d["flags"]).all()
    slots, keys = g.entry_slots(), g.entry_keys()
    comm, cost, fl = a["comm"][slots], a["cost"][slots], a["flags"][slots]
    pa = a["per_arg"][g.node_comp_off[keys[:, 0]] + keys[:, 2]]
    fin = np.isfinite(comm)
    # cost = (comm + per_arg) + transition, everywhere
    assert (cost[fin] == (comm[fin] + pa[fin]) + (fl[fin] & 1)).all()
    assert np.isinf(cost[~fin]).all() and ((fl[~fin] >> 1) == 1).all()
    # no transition => no communication
    assert (comm[(fl & 1) == 0] == 0.0).all()
    assert (comm >= 0).all()
    # the 32 identical layers have identical blocks: layer 3 vs layer 17
    per_layer = (g.num_nodes - 0) // 32
    # oracle on a sample of nodes (seconds), incl. first, last and middle nodes
    orc = O.GraphOracle(g)
    sample = sorted(set(list(range(0, 40)) + list(range(g.num_nodes - 40, g.num_nodes)) +
                        list(range(g.num_nodes // 2, g.num_nodes // 2 + 60))))
    ref = orc.build(nodes=sample)
    for v in sample:
        for e in range(int(g.node_edge_off[v]), int(g.node_edge_off[v + 1])):
            b0 = int(g.edge_off[e])
            n = int(g.edge_sdst[e]) * int(g.edge_ssrc[e])
            assert bits_equal(a["comm"][b0:b0 + n], ref["comm"][b0:b0 + n])
            assert bits_equal(a["cost"][b0:b0 + n], ref["cost"][b0:b0 + n])


@pytest.mark.parametrize("name", ["llama3_8b", "llama3_70b_8layers", "moe_16l", "llama3_70b", "stress_3k"])
def test_full_size_every_entry_against_compiled_oracle(CostEngine, name):
    """Every entry of the benchmark graphs (not a sample) against the compiled C
    restatement, itself bit-identical to the Python oracle on the test graphs
    (tests/test_oracle_c.py); and the other table layouts give the same bits."""
    from oracle import c_oracle

    g = {"llama3_8b": lambda: graphgen.config_llama3_8b(), "llama3_70b_8layers": lambda: graphgen.config_llama3_70b(8),
         "moe_16l": lambda: graphgen.config_moe(), "llama3_70b": lambda: graphgen.config_llama3_70b(),
         "stress_3k": lambda: graphgen.stress_graph(3000, (4, 8, 8), seed=0)}[name]()
    print(f"  {name}: E={g.num_entries}", flush=True)
    want = c_oracle.COracle(g).build(threads=16)
    eng = CostEngine(g).build(clamp_inf=False)
    got = eng.results()
    assert bits_equal(got["comm"], want["comm"]), first_mismatch(got["comm"], want["comm"])
    assert bits_equal(got["cost"], want["cost"]), first_mismatch(got["cost"], want["cost"])
    assert bits_equal(got["compute"], want["compute"])
    assert ((got["flags"] & 1) == want["transition"]).all()
    del got, want
    if g.num_entries > 10**8:  # the largest config once, in the layout the engine picks
        return
    for kw in (dict(table_mode="compressed", item_entries=512), dict(table_mode="full", item_entries=512),
               dict(table_mode="compressed", item_entries=256)):
        other = CostEngine(g, **kw).build(clamp_inf=False)
        assert torch.equal(other.comm.view(torch.int64), eng.comm.view(torch.int64)), kw
        assert torch.equal(other.cost.view(torch.int64), eng.cost.view(torch.int64)), kw
        assert torch.equal(other.flags, eng.flags), kw
        del other


@pytest.mark.parametrize("seed", range(12))
def test_seeded_graphs_on_many_meshes_every_layout(CostEngine, seed):
    """Seeded random graphs on 1-D to 4-D meshes (powers of two and not), in every
    table layout and work-item size the engine has: every entry against the
    compiled C restatement.  (The same loop over 240 further seeds, 1 440 builds
    and 5.3e9 entries, was run once on the device with the kernels as they are
    now, and over 360 seeds with the kernels before them, without a mismatch.)"""
    from oracle import c_oracle

    meshes = [(8,), (64,), (2, 4), (8, 8), (3, 5), (4, 8, 8), (2, 2, 2), (6, 10), (2, 3, 4), (16, 4), (2, 2, 2, 2), (4, 4, 4, 2)]
    g = graphgen.stress_graph([120, 300, 700][seed % 3], meshes[seed % len(meshes)], seed=1000 + seed, s_min=2,
                              s_max=[40, 120, 260][(seed // 3) % 3])
    want = c_oracle.COracle(g).build(threads=16)
    for mode, items, lut in (("direct", 256, False), ("direct", 256, True), ("full", 256, False), ("full", 512, True),
                             ("compressed", 256, True), ("compressed", 512, False)):
        got = CostEngine(g, table_mode=mode, item_entries=items, lut=lut).build(clamp_inf=False).results()
        assert bits_equal(got["comm"], want["comm"]), (mode, items, lut, first_mismatch(got["comm"], want["comm"]))
        assert bits_equal(got["cost"], want["cost"]), (mode, items, lut)
        assert bits_equal(got["compute"], want["compute"]), (mode, items, lut)
        assert ((got["flags"] & 1) == want["transition"]).all(), (mode, items, lut)


# ---------------------------------------------------------------------------
# scalar cost-model entry points in batch form
# ---------------------------------------------------------------------------
def _model(mesh, order_mode=0):
    from autoparallel_amd.engine import make_model

    return make_model(mesh, 8, "AMD Instinct MI355X", order_mode)


def test_forward_order_mode_matches_redistribute_cost(CostEngine, golden):
    """redistribute_cost(src, tgt, [0..ndim)) of the reference: order_mode 1."""
    for k in (2, 3, 10):  # two 2-D cases (where the orders differ) and a 3-D one
        mesh = [int(x) for x in golden[f"comm_{k}_mesh"]]
        shape = [int(x) for x in golden[f"comm_{k}_shape"]]
        stride = [int(x) for x in golden[f"comm_{k}_stride"]]
        src, tgt, want = golden[f"comm_{k}_src"], golden[f"comm_{k}_tgt"], golden[f"comm_{k}_cost_fwd"]
        src_t = sorted({tuple(int(x) for x in r) for r in src})
        tgt_t = sorted({tuple(int(x) for x in r) for r in tgt})
        g = graph_from_pairs(mesh, 8, shape, stride, int(golden[f"comm_{k}_itemsize"][0]), src_t, tgt_t)
        for use_table in (True, False):
            comm = CostEngine(g, use_table=use_table, order_mode=1).build(clamp_inf=False).results()["comm"]
            base, ssrc = int(g.edge_off[1]), int(g.edge_ssrc[1])
            si = {t: i for i, t in enumerate(src_t)}
            ti = {t: i for i, t in enumerate(tgt_t)}
            idx = np.asarray([base + ti[tuple(int(x) for x in t)] * ssrc + si[tuple(int(x) for x in s)]
                              for s, t in zip(src, tgt)])
            assert bits_equal(comm[idx], want), (k, use_table, first_mismatch(comm[idx], want))


def test_batch_scalar_entry_points(CostEngine, golden):
    import ctypes as C

    from autoparallel_amd import _lib

    lib = _lib.load()
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    # compute_read_write_time against the reference's values
    for key_b, key_t in (("rw_bytes", "rw_time"), ("rw_fbytes", "rw_ftime")):
        b = d(golden[key_b].astype(np.float64))
        out = torch.empty_like(b)
        m = _model((8, 8))
        assert lib.apc_rw_times(C.byref(m), b.numel(), b.data_ptr(), out.data_ptr(), None) == 0
        torch.cuda.synchronize()
        assert bits_equal(out.cpu().numpy(), golden[key_t])
    # _get_sharded_shape_stride against the reference's values
    mesh = [int(x) for x in golden["shard_mesh"]]
    n = golden["shard_rank"].shape[0]
    pad8 = lambda a: np.concatenate([a, np.zeros((n, 8 - a.shape[1]), np.int64)], axis=1)
    rank = d(golden["shard_rank"].astype(np.int32))
    shape, stride = d(pad8(golden["shard_shape"])), d(pad8(golden["shard_stride"]))
    plc = d(np.concatenate([golden["shard_plc"], np.zeros((n, 1), np.uint8)], axis=1))
    o_shape, o_stride = torch.zeros_like(shape), torch.zeros_like(stride)
    m = _model(mesh)
    assert lib.apc_local_shapes(C.byref(m), n, rank.data_ptr(), shape.data_ptr(), stride.data_ptr(),
                                plc.data_ptr(), o_shape.data_ptr(), o_stride.data_ptr(), None) == 0
    torch.cuda.synchronize()
    assert (o_shape.cpu().numpy()[:, :4] == golden["shard_out_shape"]).all()
    assert (o_stride.cpu().numpy()[:, :4] == golden["shard_out_stride"]).all()
    # collective_comm_cost against the oracle (itself checked against torch's functions)
    rng = np.random.default_rng(5)
    q = 500
    kind = rng.integers(0, 5, q).astype(np.int32)
    nbytes = rng.integers(0, 2**36, q).astype(np.int64)
    dim = rng.integers(0, 3, q).astype(np.int32)
    out = torch.empty(q, dtype=torch.float64, device="cuda")
    mesh = (4, 8, 8)
    m = _model(mesh)
    tk, tb, td = d(kind), d(nbytes), d(dim)
    assert lib.apc_collective_costs(C.byref(m), q, tk.data_ptr(), tb.data_ptr(), td.data_ptr(), out.data_ptr(), None) == 0
    torch.cuda.synchronize()
    topo = O.Topo(mesh, 8)
    names = ["allgather", "all_to_all", "allreduce", "reduce_scatter", "unknown"]
    want = np.asarray([O.collective_comm_cost(names[k], int(b), topo, int(dd)) for k, b, dd in zip(kind, nbytes, dim)])
    assert bits_equal(out.cpu().numpy(), want)


# ---------------------------------------------------------------------------
# ILP: the plan from the HIP coefficients is the plan from the oracle's
# ---------------------------------------------------------------------------
def test_solved_plan_identical(CostEngine):
    from autoparallel_amd.sharding_problem import Coefficients, PackedShardingOptimizer
    from test_sharding_problem import oracle_coefficients

    g = graphgen.gpt2_graph((4,), n_layers=1, dim=64, n_heads=2, ffn_dim=128, vocab=256, seq=32, batch=8)
    gpu = PackedShardingOptimizer(g)
    ref_coef, raw = oracle_coefficients(g)
    assert bits_equal(gpu.coef.cost, ref_coef.cost) and bits_equal(gpu.coef.comm, ref_coef.comm)
    assert (gpu.coef.flags == ref_coef.flags).all() and bits_equal(gpu.coef.per_arg, ref_coef.per_arg)
    cpu = PackedShardingOptimizer(g, coefficients=ref_coef)
    s_gpu, s_cpu = gpu.get_solution(), cpu.get_solution()
    assert (s_gpu == s_cpu).all() and gpu.objective_value == cpu.objective_value
    # the scorer on the device agrees with the oracle on the solved plan
    got = gpu.compute_solution_cost(s_gpu)
    want = O.score_assignment(g, raw["comm"], raw["transition"], raw["compute"], s_gpu)
    assert (got["total"], got["compute"], got["comm"], got["transition"]) == tuple(float(x) for x in want)
    # prefetch discount through the optimizer, then re-solve: never more expensive
    base = gpu.objective_value
    assert gpu.apply_prefetch_discount(0.0) > 0
    gpu.get_solution()
    assert gpu.objective_value <= base + 1e-9


def test_memory_constraint(CostEngine):
    from autoparallel_amd.sharding_problem import PackedShardingOptimizer

    g = graphgen.gpt2_graph((4,), n_layers=1, dim=64, n_heads=2, ffn_dim=128, vocab=256, seq=32, batch=8)
    opt = PackedShardingOptimizer(g)
    params = [p for p, _ in g.roles.param_grad]
    ratios = opt._memory_ratios(params)
    for p, r in zip(params, ratios):
        run = int(g.node_out_list[p])
        for o in range(int(g.node_nstrat[p])):
            w = int(g.lists[run + o])
            rk = int(g.meta_rank[w >> 12])
            shape = [int(x) for x in g.meta_shape[w >> 12, :rk]]
            plc = [int(x) for x in g.tuple_plc[w & 0xFFF, : g.ndim]]
            ls, _ = O.sharded_shape_stride(shape, [1] * rk, plc, [int(x) for x in g.mesh_shape])
            assert r[o] == np.prod(ls) / np.prod(shape)
    # parameters sharded as much as possible: every parameter at its smallest ratio
    opt.add_parameter_memory_constraint(0.0, 0.0)
    sol = opt.get_solution()
    for p, r in zip(params, ratios):
        assert r[sol[p]] == r.min()
    assert "memory_constraint_high" in opt.prob.constraints


def test_saved_problem_carries_the_memory_ratios(CostEngine, tmp_path, monkeypatch):
    """The ratios that weigh the memory budget rows come from the device; the saved file holds
    them, so the problem read back is solved under its budget without another device call."""
    from autoparallel_amd import _lib
    from autoparallel_amd.sharding_problem import PackedShardingOptimizer

    g = graphgen.gpt2_graph((4,), n_layers=1, dim=64, n_heads=2, ffn_dim=128, vocab=256, seq=32, batch=8)
    opt = PackedShardingOptimizer(g)
    opt.add_parameter_memory_constraint(0.0, 0.0)
    sol = opt.get_solution()
    path = str(tmp_path / "budget.npz")
    opt.save(path)
    params = [p for p, _ in g.roles.param_grad]
    want = opt._memory_ratios(params)
    monkeypatch.setattr(_lib, "load", lambda: (_ for _ in ()).throw(AssertionError("no device call expected")))
    back = PackedShardingOptimizer.load(path)
    assert all(np.array_equal(a, b) for a, b in zip(back._memory_ratios(params), want))
    assert np.array_equal(back.resolve(), sol) and "memory_constraint_high" in back.prob.constraints
    assert np.isclose(back.objective_value, opt.objective_value, rtol=1e-12)

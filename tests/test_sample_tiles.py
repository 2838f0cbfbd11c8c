"""The layout of a feasible draw in tiles (apc_sample_tiles, host) and the draw over it: every choice and count of the
walk with a lane per assignment."""
import ctypes as C
import itertools

import numpy as np
import pytest
import torch

from autoparallel_amd import _lib, graphgen, packed
from autoparallel_amd import engine as engine_mod

TILE = np.dtype([(k, "<i4") for k in ("node0", "n_node", "edge0", "n_edge", "seq0", "n_far")]
                + [("far", "<i4", 24), ("reserved", "<i4", 10)])
RING = 64


def _layout(off, src, ssrc, nstrat, first_node):
    a = [np.ascontiguousarray(x, np.int32) for x in (off, src, ssrc, nstrat)]
    n = len(nstrat)
    tiles, row, n_tile = np.zeros(n, TILE), np.zeros(max(len(src), 1), np.uint8), C.c_int32()
    _lib.check(_lib.load().apc_sample_tiles(n, len(src), *[x.ctypes.data for x in a], first_node, tiles.ctypes.data, n,
                                            row.ctypes.data, C.byref(n_tile)), "apc_sample_tiles")
    return tiles[:n_tile.value], row


def _many_args(n=300, seed=1, strategies=64, widest=6):
    """Nodes of up to 64 strategies with none to 32 argument rows, among them rows of the node in front more than once,
    of nodes far behind and of no producer."""
    b = packed.GraphBuilder((2, 2), 4)
    m = b.meta((8, 16, 32), (512, 32, 1), 4, packed.DT_F32)
    tuples = list(itertools.product([0x00, 0x40, 0x41, 0x42, 0x80, 0x81, 0x82, 0x83], repeat=2))
    rng = np.random.default_rng(seed)

    def specs(k):
        return [b.spec(m, tuples[i]) for i in rng.choice(len(tuples), k, replace=False)]

    at = []
    for v in range(n):
        s = specs(int(rng.choice([1, 5, 31, 32, 33, strategies - 1, strategies])))
        rows = 32 if v % 97 == 50 else int(rng.integers(0, widest))
        if rows == 0 or not at:
            at.append(b.add_node(packed.NodeDesc(f"n{v}", in_specs=[[x] for x in s], out_specs=[[x] for x in s], inputs=[],
                                                 default_rows=[[[0.0]] for _ in s])))
            continue
        back = np.where(rng.random(rows) < 0.4, 1, rng.integers(1, v + 1, rows))  # how far in front of it
        at.append(b.add_node(packed.NodeDesc(f"n{v}", in_specs=[[x] * rows for x in s], out_specs=[[x] for x in s],
                                             inputs=[at[v - int(d)] for d in back])))
    return b.pack(), None, 0


GRAPHS = {
    "many_args": _many_args,
    "gpt2": lambda: (graphgen.gpt2_graph((2, 3), 2, vocab=4096, seq=512, batch=64), None, 0),
    "llama_8x8": lambda: (graphgen.llama_graph((8, 8), 1, 1024, 8, 4, 2048, 8192, 512, 16), None, 0),
}


@pytest.mark.parametrize("name,first_node", [("many_args", 0), ("many_args", 70), ("gpt2", 0), ("llama_8x8", 0), ("llama_8x8", 3)])
def test_layout(name, first_node):
    g = GRAPHS[name]()[0]
    tiles, row = _layout(g.node_edge_off, g.edge_src_node, g.edge_ssrc, g.node_nstrat, first_node)
    v = first_node
    for i, t in enumerate(tiles):
        assert t["node0"] == v and t["seq0"] == v - first_node and 0 < t["n_node"] <= 32 and t["n_edge"] <= 32
        e0, e1 = int(g.node_edge_off[v]), int(g.node_edge_off[v + t["n_node"]])
        assert (t["edge0"], t["edge0"] + t["n_edge"]) == (e0, e1) and t["n_far"] <= 24 and (t["far"][t["n_far"]:] == 0).all()
        asked = first_node if i == 0 else int(tiles[i - 1]["node0"])  # older choices are asked for when that tile begins
        for e in range(e0, e1):
            u, at = int(g.edge_src_node[e]), int(row[e])
            consumer = int(g.edge_node[e])
            if u < 0:
                assert at == 255
            elif at < RING:  # still there, also while the node in front is drawn
                assert u >= first_node and at == (u - first_node) % RING and consumer - u < RING
            else:
                assert t["far"][at - RING] == u and at - RING < t["n_far"] and u < asked
        v += int(t["n_node"])
    assert v == g.num_nodes
    level = np.zeros(v, int)  # nodes of the longest chain that ends in a node
    for u in range(first_node, v):
        src = g.edge_src_node[g.node_edge_off[u]:g.node_edge_off[u + 1]]
        level[u] = 1 + max((level[x] for x in src if x >= first_node), default=0)
    assert tiles[0]["reserved"][0] == level.max() and (tiles[1:]["reserved"] == 0).all()


def test_layout_leaves_other_graphs_alone():
    off, one = [0, 0, 1], [2, 2]
    assert len(_layout(off, [0], [2], one, 0)[0]) == 1
    assert len(_layout(off, [1], [2], one, 0)[0]) == 0  # a producer that is not in front of its consumer
    assert len(_layout(off, [0], [65], [65, 2], 0)[0]) == 0
    assert len(_layout([0, 0, 33], [0] * 33, [2] * 33, one, 0)[0]) == 0
    assert len(_layout(off, [0], [2], one, 2)[0]) == 0


# workgroups of one wavefront to sixteen, and two launches; filters, given choices of earlier nodes, other ids
@pytest.mark.gpu
@pytest.mark.parametrize("name,count", [(name, count) for name in GRAPHS for count in (1, 65, 1000)]
                         + [("many_args", 70001), ("gpt2", 262144), ("gpt2", 262145)])
def test_draws_equal_the_lane_walks(name, count, monkeypatch):
    g, gid, first_node = GRAPHS[name]()
    eng = engine_mod.CostEngine(g).build()
    rng = np.random.default_rng(count)
    filters = {v: rng.random(int(g.node_nstrat[v])) < 0.7 for v in range(first_node, g.num_nodes, 3)}
    given = (rng.integers(0, 1 << 20, (g.num_nodes, count)) % g.node_nstrat[:, None]).astype(np.int16)

    def draws():
        out = []
        for row_filter in (None, filters):
            for ids, begin in ((gid, first_node), (None if gid is None else gid * 3, first_node)) + (
                    ((np.arange(g.num_nodes) + 9, 40),) if count < 70001 else ()):
                assign = torch.from_numpy(given).cuda().view(torch.uint16)
                a, f = eng.sample_feasible(3, 17, count, node_gid=ids, first_node=begin, assign=assign, row_filter=row_filter)
                out += [a.view(torch.int16).cpu(), f.cpu()]
        return out

    monkeypatch.setattr(engine_mod, "_SAMPLE_TILES_US", (0.0, 0.0, 0.0))  # also where steps would be faster
    assert eng._sample_tiles(first_node) is not None
    got = draws()
    assert eng.last_sample_backend == "tiles"
    monkeypatch.setattr(engine_mod, "_SAMPLE_TILES", False)
    monkeypatch.setattr(engine_mod, "_SAMPLE_LANES_FROM", {2: 0, 16: 0})
    want = draws()
    assert eng.last_sample_backend == "lanes"
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    if name == "many_args":
        assert max(int(f.max()) for f in want[1::2]) > 0  # nodes that fall back do occur


# small batches of a graph with work for sixteen wavefronts go in steps, larger ones and decoders by tiles, the smallest
# graphs in steps of two; the same draws
@pytest.mark.gpu
@pytest.mark.parametrize("name,first_node,count,route", [
    ("dag", 0, 100, "steps"), ("dag", 0, 16385, "steps"), ("dag", 0, 49152, "steps"), ("dag", 0, 49153, "tiles"),
    ("dag", 90, 33, "steps"), ("small_dag", 0, 32768, "steps"), ("small_dag", 0, 65537, "tiles"), ("smallest_dag", 0, 65536, "steps"),
    ("smallest_dag", 0, 131072, "steps"), ("smallest_dag", 0, 196608, "tiles"), ("gpt2", 0, 1, "tiles"),
    ("llama_8x8", 0, 65, "tiles")])
def test_which_graphs_are_drawn_in_steps(name, first_node, count, route, monkeypatch):
    g = {"dag": lambda: graphgen.stress_graph(400, (2, 2, 4), seed=1, s_min=2, s_max=20),
         "small_dag": lambda: graphgen.stress_graph(60, (2, 2, 4), seed=1, s_min=2, s_max=20),
         "smallest_dag": lambda: graphgen.stress_graph(30, (2, 2, 4), seed=1, s_min=2, s_max=20),
         **{k: lambda k=k: GRAPHS[k]()[0] for k in GRAPHS}}[name]()
    eng = engine_mod.CostEngine(g).build()
    gen = torch.Generator(device="cuda").manual_seed(count)
    nstrat = torch.from_numpy(g.node_nstrat.astype(np.int32)).cuda()[:, None]
    given = (torch.randint(0, 1 << 30, (g.num_nodes, count), device="cuda", generator=gen, dtype=torch.int32)
             % nstrat).to(torch.int16).view(torch.uint16)

    def draw():
        a, f = eng.sample_feasible(3, 17, count, first_node=first_node, assign=given.clone())
        return a.view(torch.int16), f, eng.last_sample_backend

    got = draw()
    assert got[2] == route
    monkeypatch.setattr(engine_mod, "_SAMPLE_TILES", False)
    monkeypatch.setattr(engine_mod, "_SAMPLE_LANES_FROM", {2: 0, 16: 0})
    want = draw()
    assert want[2] == "lanes" and torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])

"""The list of pieces of a walk over large matrices (apc_score_pieces, host): every argument row in order, and a ring in
which nothing is overwritten before it is done with; and the scores over it have the bits of the walk over records."""
import ctypes as C

import numpy as np
import pytest
import torch

from autoparallel_amd import _lib, graphgen
from autoparallel_amd import engine as engine_mod

PIECE = np.dtype([(k, "<i4") for k in ("node", "edge", "item", "flags", "base", "n", "lds", "ask")])
RING = 160 * 1024

GRAPHS = {
    "window": lambda: graphgen.stress_dag_window(2000, 600, 700, (4, 8, 8), seed=0)[0],  # up to 300 KB a matrix
    "stress": lambda: graphgen.stress_graph(40, (4, 8, 8), seed=3, s_min=2, s_max=400),
    "moe_8x8": lambda: graphgen.moe_graph((8, 8), 1, vocab=4096, seq=512, batch=64),  # edges without a producer
}


def _pieces(g, first_node, msize):
    edges = np.ascontiguousarray(g.edge_records(True))
    off, nstrat = [np.ascontiguousarray(x, np.int32) for x in (g.node_edge_off, g.node_nstrat)]
    out = np.zeros(g.num_nodes + int((msize // 8192 + 1).sum()), PIECE)
    n, items = C.c_int32(), C.c_int32()
    _lib.check(_lib.load().apc_score_pieces(
        edges.ctypes.data, g.num_edges, g.num_nodes, off.ctypes.data, nstrat.ctypes.data, msize.ctypes.data, first_node,
        out.ctypes.data, len(out), C.byref(n), C.byref(items)), "apc_score_pieces")
    return edges, out[:n.value], items.value


@pytest.mark.parametrize("name,first_node,scale", [("window", 0, 1), ("window", 20, 1), ("stress", 7, 3), ("moe_8x8", 0, 1)])
def test_pieces(name, first_node, scale):
    g = GRAPHS[name]()
    msize = (g.edge_ssrc.astype(np.int64) * g.edge_sdst // scale).astype(np.int32)
    edges, pieces, n_item = _pieces(g, first_node, msize)
    want = []
    for v in range(first_node, g.num_nodes):
        e0, e1 = int(g.node_edge_off[v]), int(g.node_edge_off[v + 1])
        for e in range(e0, e1) if e1 > e0 else [-1]:
            size = int(msize[e]) if e >= 0 and edges["table_off"][e] >= 0 else 0
            parts = range(0, max(size, 1), 8192)
            want += [(v, e, b, min(size - b, 8192), (b == 0 and e in (-1, e0)) + 2 * (b == 0) + 4 * (b == parts[-1]))
                     for b in parts]
    assert [tuple(int(q[k]) for k in ("node", "edge", "base", "n", "flags")) for q in pieces] == want
    assert (np.diff(pieces["item"]) == ((pieces["flags"][1:] & 2) != 0)).all() and n_item == pieces["item"][-1] + 1
    side = 10 * g.node_nstrat[pieces["node"]].astype(np.int64) + 2 * np.where(pieces["edge"] >= 0, g.edge_ssrc[pieces["edge"]], 0)
    size = np.where(pieces["flags"] & 2, -(-side // 1024), 0) * 1024 + -(-pieces["n"] // 128) * 1024
    assert (pieces["lds"] >= 0).all() and (pieces["lds"] + size <= RING).all() and (pieces["lds"] % 1024 == 0).all()
    assert (np.diff(pieces["ask"]) >= 0).all() and pieces["ask"].max() <= len(pieces)
    for t in range(len(pieces)):  # what is in use or under way while piece t is drawn from
        live = np.arange(t, max(int(pieces["ask"][t]), t + 1))
        order = live[np.argsort(pieces["lds"][live], kind="stable")]
        assert (pieces["lds"][order][:-1] + size[order][:-1] <= pieces["lds"][order][1:]).all()
        assert live[-1] < t + 16


def test_pieces_leave_other_graphs_alone():
    g = graphgen.stress_graph(6, (4, 8, 8), seed=4, s_min=1030, s_max=1100)
    assert len(_pieces(g, 0, np.full(g.num_edges, 100, np.int32))[1]) == 0
    sizes = engine_mod.matrix_sizes(g, False)
    assert engine_mod.piece_counts(g, sizes, 0) is None and engine_mod.piece_counts(g, sizes, g.num_nodes) is None


@pytest.mark.parametrize("compressed", [False, True])
@pytest.mark.parametrize("first_node", [0, 9])
@pytest.mark.parametrize("name", [*GRAPHS, "widest", "wider"])
def test_counts_are_those_of_the_list(name, first_node, compressed):
    """What the choice of a scorer asks, without a list: at the largest counts of strategies that a list takes, too."""
    wide = {"widest": 682, "wider": 683}  # 12 bytes of a side image a strategy, of 8 192
    g = GRAPHS[name]() if name in GRAPHS else graphgen.stress_graph(12, (4, 8, 8), seed=4, s_min=wide[name], s_max=wide[name])
    edges = np.ascontiguousarray(g.edge_records(compressed))
    off, nstrat = [np.ascontiguousarray(x, np.int32) for x in (g.node_edge_off, g.node_nstrat)]
    sizes = engine_mod.matrix_sizes(g, compressed)
    msize = sizes.astype(np.int32)
    out, n, items = np.zeros(g.num_nodes + int((msize // 8192 + 1).sum()), PIECE), C.c_int32(), C.c_int32()
    _lib.check(_lib.load().apc_score_pieces(
        edges.ctypes.data, g.num_edges, g.num_nodes, off.ctypes.data, nstrat.ctypes.data, msize.ctypes.data, first_node,
        out.ctypes.data, len(out), C.byref(n), C.byref(items)), "apc_score_pieces")
    assert engine_mod.piece_counts(g, sizes, first_node) == ((n.value, items.value) if n.value else None)
    assert (n.value == 0) == (name == "wider")


# one assignment a lane up to 2^18, then two, then four, then a second launch; a workgroup of five wavefronts
@pytest.mark.gpu
@pytest.mark.parametrize("name,count", [(name, count) for name in GRAPHS for count in (1, 70001, 262145, 524289)]
                         + [("moe_8x8", 2**20 + 65)])
def test_scores_have_the_bits_of_the_walk_over_records(name, count, monkeypatch):
    g = GRAPHS[name]()
    eng = engine_mod.CostEngine(g)
    eng.large_blocks = True
    gid = np.arange(g.num_nodes, dtype=np.int32) * 7 + 1
    gen = torch.Generator(device="cuda").manual_seed(count)
    init = torch.rand((count, 6), dtype=torch.float64, device="cuda", generator=gen) * 1e6
    init[::3] = -0.0

    def scores(backend):
        out = []
        for score in (lambda: eng.score_random(11, 5, count), lambda: eng.score_random_window(11, 5, count, gid, 5, init=init)):
            out.append(score().view(torch.int64))
            assert eng.last_score_backend == backend
        return out

    monkeypatch.setattr(engine_mod, "_SCORE_LANES_FROM", 1)
    monkeypatch.setattr(engine_mod, "_SCORE_TABLE_FROM", 0)
    monkeypatch.setattr(engine_mod, "_SCORE_TABLE_US", (1e9, 0, 0, 0, 0, 0))  # the stream, also where edge by edge is faster
    for clamp in (True, False):
        eng.build(clamp_inf=clamp)
        assert eng._score_pieces(0) is not None and eng._score_pieces(5) is not None
        got = scores("block_table")
        monkeypatch.setattr(engine_mod, "_SCORE_STREAM", False)  # edge by edge
        assert all(torch.equal(a, b) for a, b in zip(got, scores("block_table")))
        monkeypatch.setattr(engine_mod, "_SCORE_STREAM", True)
        monkeypatch.setattr(engine_mod, "_SCORE_FROM_TABLE", False)
        assert all(torch.equal(a, b) for a, b in zip(got, scores("compact_records")))
        monkeypatch.setattr(engine_mod, "_SCORE_FROM_TABLE", True)
        eng.set_node_multiplier(np.arange(g.num_nodes) % 3 - 1)  # the list is kept, the multipliers are the call's

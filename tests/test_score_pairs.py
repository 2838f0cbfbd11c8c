"""Images of finished entries (apc_pair_tiles, host): every argument row once, entries that do not overlap, and slots that
hold the choices a step reads; and the scores from them have the bits of the walk over records."""
import ctypes as C

import numpy as np
import pytest
import torch

from autoparallel_amd import _lib, graphgen
from autoparallel_amd import engine as engine_mod

STEP = np.dtype([(k, "<i4") for k in ("node", "edge", "pairs", "terms", "row_node", "row_src")])
TILE = np.dtype([("step0", "<i4"), ("step1", "<i4"), ("n_row", "<i4"), ("n_unit", "<i4"), ("row", "<i4", 12),
                 ("slot", "u1", 12), ("reserved", "<i4")])

GRAPHS = {
    "moe_8x8": lambda: graphgen.moe_graph((8, 8), 1, vocab=4096, seq=512, batch=64),  # edges without a producer
    "gpt2_2x3": lambda: graphgen.gpt2_graph((2, 3), 1, vocab=4096, seq=512, batch=64),
    "stress_57": lambda: graphgen.stress_graph(60, (8, 8), seed=2, s_min=1, s_max=57),  # up to 3 249 entries an edge
}


def _tiles(g, first_node):
    edges = np.ascontiguousarray(g.edge_records(False))
    off, nstrat = [np.ascontiguousarray(x, np.int32) for x in (g.node_edge_off, g.node_nstrat)]
    most = g.num_nodes + g.num_edges
    steps, tiles = np.zeros(most, STEP), np.zeros(most, TILE)
    n_step, n_tile = C.c_int32(), C.c_int32()
    _lib.check(_lib.load().apc_pair_tiles(
        edges.ctypes.data, g.num_edges, g.num_nodes, off.ctypes.data, nstrat.ctypes.data, first_node, steps.ctypes.data,
        most, tiles.ctypes.data, most, C.byref(n_step), C.byref(n_tile)), "apc_pair_tiles")
    return steps[:n_step.value], tiles[:n_tile.value]


@pytest.mark.parametrize("first_node", [0, 7])
@pytest.mark.parametrize("name", GRAPHS)
def test_tiles(name, first_node):
    g = GRAPHS[name]()
    assert (STEP.itemsize, TILE.itemsize) == (_lib.PAIR_STEP_BYTES, _lib.PAIR_TILE_BYTES)
    steps, tiles = _tiles(g, first_node)
    want = []
    for v in range(first_node, g.num_nodes):
        e0, e1 = int(g.node_edge_off[v]), int(g.node_edge_off[v + 1])
        want += [(v, e) for e in range(e0, e1)] or [(v, -1)]
    assert [(int(s["node"]), int(s["edge"])) for s in steps] == want
    assert (tiles["step0"][1:] == tiles["step1"][:-1]).all() and tiles["step0"][0] == 0 and tiles["step1"][-1] == len(steps)
    held, scored = {}, set()
    for t in tiles:
        assert 0 < t["step1"] - t["step0"] <= 64 and t["n_row"] <= 12 and t["n_unit"] <= 3328
        assert ((0 <= t["row"]) & (t["row"] < g.num_nodes)).all()
        for r in range(t["n_row"]):
            assert t["slot"][r] < 12
            held[int(t["slot"][r])] = int(t["row"][r])
        at = 0
        for s in steps[t["step0"]:t["step1"]]:
            v, e = int(s["node"]), int(s["edge"])
            src = int(g.edge_src_node[e]) if e >= 0 else -1
            assert held[int(s["row_node"])] == v
            assert held[int(s["row_src"])] == src if src >= 0 else s["row_src"] == -1
            if e >= 0:
                assert s["pairs"] == at
                at += int(g.node_nstrat[v]) * (int(g.edge_ssrc[e]) if src >= 0 else 1)
            if v not in scored:
                assert s["terms"] == at
                at += (int(g.node_nstrat[v]) + 1) // 2
                scored.add(v)
            else:
                assert s["terms"] == -1
        assert t["n_unit"] == at
    assert scored == set(range(first_node, g.num_nodes))


def test_graphs_of_another_form_are_left_alone():
    for g in (graphgen.stress_graph(6, (4, 8, 8), seed=4, s_min=58, s_max=60),  # 58 * 58 entries and terms: over a buffer
              graphgen.stress_graph(6, (4, 8, 8), seed=4, s_min=257, s_max=258)):
        assert len(_tiles(g, 0)[1]) == 0
    g = GRAPHS["gpt2_2x3"]()
    assert len(_tiles(g, g.num_nodes)[1]) == 0  # nothing to score


# one assignment a lane up to 2^18, then two, then four, then a second launch; a workgroup without a whole wavefront.
# Multipliers 1: costs that carry their flag in the sign; -1, 0, 1: tiles that name it; clamped or infinite
@pytest.mark.gpu
@pytest.mark.parametrize("name,count", [(name, count) for name in GRAPHS for count in (1, 70001, 262145, 524289)]
                         + [("gpt2_2x3", 2**20 + 65)])
def test_scores_have_the_bits_of_the_walk_over_records(name, count, monkeypatch):
    g = GRAPHS[name]()
    eng = engine_mod.CostEngine(g, table_mode="full")
    eng.large_blocks = False
    gid = np.arange(g.num_nodes, dtype=np.int32) * 7 + 1
    called = []
    score_pairs = eng.lib.apc_score_pairs
    monkeypatch.setattr(eng, "lib", type("Lib", (), {
        "__getattr__": lambda self, k: getattr(_lib.load(), k),
        "apc_score_pairs": staticmethod(lambda *a: called.append(1) or score_pairs(*a))})())

    def scores():
        return [score().view(torch.int64) for score in (
            lambda: eng.score_random(11, 5, count), lambda: eng.score_random_window(11, 5, count, gid, 5))]

    monkeypatch.setattr(engine_mod, "_SCORE_LANES_FROM", 1)
    monkeypatch.setattr(engine_mod, "_SCORE_TERMS_ABOVE", False)
    monkeypatch.setattr(engine_mod, "_SCORE_PAIRS_TILES", 1)
    monkeypatch.setattr(engine_mod, "_SCORE_PAIRS_FROM", (0, 0))
    for mult in (np.ones(g.num_nodes, np.int32), np.arange(g.num_nodes, dtype=np.int32) % 3 - 1):
        eng.set_node_multiplier(mult)  # the layout is kept, the multipliers are the call's
        for clamp in (True, False):
            eng.build(clamp_inf=clamp)
            called.clear()
            got = scores()
            assert len(called) == 2
            monkeypatch.setattr(engine_mod, "_SCORE_PAIRS", False)  # over matrices
            assert all(torch.equal(a, b) for a, b in zip(got, scores()))
            monkeypatch.setattr(engine_mod, "_SCORE_PAIRS", True)
            monkeypatch.setattr(engine_mod, "_SCORE_FROM_TILES", False)  # over records
            assert all(torch.equal(a, b) for a, b in zip(got, scores()))
            monkeypatch.setattr(engine_mod, "_SCORE_FROM_TILES", True)
            assert len(called) == 2

"""The layout of a walk in tiles (apc_score_tiles, host) brings in what every step reads, and the
scores from it have the bits of the walk over records."""
import ctypes as C

import numpy as np
import pytest
import torch

from autoparallel_amd import _lib, graphgen, packed
from autoparallel_amd import engine as engine_mod

STEP = np.dtype([(k, "<i4") for k in ("node", "src", "nstrat", "ssrc", "nargs", "flags", "mat", "pa", "row_node",
                                      "row_src")] + [("reserved", "<i4", 6)])
UNIT = np.dtype([("src", "<i8"), ("lds", "<u2"), ("n", "<u2"), ("kind", "<i4")])
TILE = np.dtype([(k, "<i4") for k in ("step0", "step1", "unit0", "unit1", "n_row", "any_edge")]
                + [("row", "<i4", 16), ("reserved", "<i4", 10)])
DOUBLES = 5120

def _default_rows(n=6, strategies=250, columns=11, rows=3):
    """Nodes with argument rows without a producer, whose default values fill a tile each: the terms of a node are placed
    in every tile that it goes on in."""
    b = packed.GraphBuilder((2, 2), 4)
    m = b.meta((64, 96), (96, 1), 4, packed.DT_F32)
    tuples = [(x, y) for x in (0x00, 0x40, 0x41, 0x80) for y in (0x00, 0x40, 0x41, 0x80)]
    specs = [b.spec(m, tuples[o % 16]) for o in range(strategies)]
    for v in range(n):
        b.add_node(packed.NodeDesc(
            f"n{v}", in_specs=[[x] * rows for x in specs], out_specs=[[x] for x in specs], inputs=[],
            default_rows=[[[0.5 * j + a + o * v for j in range(columns)] for a in range(rows)] for o in range(strategies)]))
    return b.pack()


GRAPHS = {
    "default_rows": _default_rows,
    "gpt2_2x3": lambda: graphgen.gpt2_graph((2, 3), 1, vocab=4096, seq=512, batch=64),
    "moe_8x8": lambda: graphgen.moe_graph((8, 8), 1, vocab=4096, seq=512, batch=64),
    "stress_60": lambda: graphgen.stress_graph(150, (2, 2, 4), seed=4, s_min=2, s_max=60),
}


def _layout(g, first_node, explicit):
    edges = np.ascontiguousarray(g.edge_records(False))
    a = [np.ascontiguousarray(x, t) for x, t in ((g.node_edge_off, np.int32), (g.node_nstrat, np.int32),
                                                 (g.node_nargs, np.int32), (g.node_comp_off, np.int64))]
    most = g.num_nodes + g.num_edges
    room = 2 * most + g.num_entries + g.num_compute
    steps, tiles, units = np.zeros(most, STEP), np.zeros(most, TILE), np.zeros(room, UNIT)
    n = [C.c_int32() for _ in range(3)]
    _lib.check(_lib.load().apc_score_tiles(
        edges.ctypes.data, g.num_edges, g.num_nodes, *[x.ctypes.data for x in a], first_node, explicit,
        steps.ctypes.data, most, tiles.ctypes.data, most, units.ctypes.data, room, *[C.byref(x) for x in n]),
        "apc_score_tiles")
    return edges, steps[:n[0].value], tiles[:n[1].value], units[:n[2].value]


@pytest.mark.parametrize("explicit", [0, 1])
@pytest.mark.parametrize("first_node", [0, 5])
@pytest.mark.parametrize("name", list(GRAPHS))
def test_layout(name, first_node, explicit):
    g = GRAPHS[name]()
    edges, steps, tiles, units = _layout(g, first_node, explicit)
    room = engine_mod.score_tile_room(g)
    assert max(len(steps), len(tiles)) <= room[0] and len(units) <= room[1]
    assert (STEP.itemsize, TILE.itemsize, UNIT.itemsize) == (64, 128, 16)
    table_size = int(g.block_table(False)[1][-1])
    e, v, ring, at = int(g.node_edge_off[first_node]), first_node - 1, {}, 0
    for t in tiles:
        assert t["step0"] == at and t["step1"] > at and t["unit1"] > t["unit0"]
        at = int(t["step1"])
        buf = np.full(DOUBLES, -1, np.int64)  # what a place of the buffer holds: element * 3 + array
        for u in units[t["unit0"]:t["unit1"]]:
            n = int(u["n"])
            assert u["lds"] % 2 == 0 and 0 < n <= (128 if u["kind"] == 0 else 32) and u["lds"] + n <= DOUBLES
            if u["kind"] == 0:  # copied in pairs, 16 bytes aligned
                assert u["src"] % 2 == 0 and u["src"] + (n + 1) // 2 * 2 <= table_size
            buf[u["lds"]:u["lds"] + n] = (u["src"] + np.arange(n)) * 3 + u["kind"]
        for s in steps[t["step0"]:t["step1"]]:
            if s["flags"] & 1:
                v += 1
                k = np.arange(int(g.node_nstrat[v]))
                assert s["nstrat"] == len(k) and s["nargs"] == max(1, g.node_nargs[v])
                assert (buf[s["pa"] + k] == (g.node_comp_off[v] + k) * 3 + 1).all()
                if explicit:
                    assert s["row_node"] < t["n_row"] <= 16 and t["row"][s["row_node"]] == v
                else:
                    assert s["row_node"] == v % 16
                    ring[v % 16] = v
            assert s["node"] == v
            if s["flags"] & 2:
                ed = edges[e]
                e += 1
                assert ed["node"] == v and ed["src_node"] == s["src"] and ed["ssrc"] == s["ssrc"]
                k = np.arange(int(ed["ssrc"]) * int(ed["sdst"]))
                src, kind = (ed["table_off"], 0) if ed["table_off"] >= 0 else (ed["default_off"], 2)
                assert (buf[s["mat"] + k] == (src + k) * 3 + kind).all()
                if s["row_src"] >= 0:
                    assert s["src"] == (t["row"][s["row_src"]] if explicit else ring[int(s["row_src"])])
                else:
                    assert s["src"] < 0 or not explicit
    assert at == len(steps) and v == g.num_nodes - 1 and e == g.num_edges


def test_layout_leaves_other_graphs_alone():
    g = graphgen.stress_graph(60, (2, 2, 4), seed=4, s_min=200, s_max=700)
    assert len(_layout(g, 0, 0)[1]) == 0


# one assignment a lane up to 2^18, then two, then four (two, and a second launch, if explicit); past 2^20
# random ones take a second launch too.  As batches are walked where there is room for the images, where there is none,
# and where there is none for a record per step either.
@pytest.mark.gpu
@pytest.mark.parametrize("room", ["images", "steps", "none"])
@pytest.mark.parametrize("name,count", [(name, count) for name in GRAPHS for count in (1, 129, 33000, 200000, 262145, 524289)]
                         + [("gpt2_2x3", 2**20 + 65)])
def test_scores_have_the_bits_of_the_walk_over_records(name, count, room, monkeypatch):
    g = GRAPHS[name]()
    eng = engine_mod.CostEngine(g, table_mode="full").build()
    eng.large_blocks = False
    mult = np.arange(g.num_nodes) % 3 + 1
    gid = np.arange(g.num_nodes, dtype=np.int32) * 7 + 1
    gen = torch.Generator(device="cuda").manual_seed(count)
    nstrat = torch.from_numpy(g.node_nstrat.astype(np.int32)).cuda()[:, None]
    assign = (torch.randint(0, 1 << 30, (g.num_nodes, count), device="cuda", generator=gen, dtype=torch.int32)
              % nstrat).to(torch.int16)
    init = torch.rand((count, 6), dtype=torch.float64, device="cuda", generator=gen) * 1e6

    def scores(*backends):
        out = []
        for score, backend in zip((
                lambda: eng.score_random(11, 5, count), lambda: eng.score(assign),
                lambda: eng.score_random_window(11, 5, count, gid, 5, init=init),
                lambda: eng.score_window(assign, 5, init=init)), backends):
            out.append(score().view(torch.int64))
            assert backend in (eng.last_score_backend, eng.last_score_entry)
        return out

    monkeypatch.setattr(engine_mod, "_SCORE_LANES_FROM", 1)
    monkeypatch.setattr(engine_mod, "_SCORE_TERMS_ABOVE", False)
    monkeypatch.setattr(engine_mod, "_SCORE_PAIRS_TILES", 1)
    monkeypatch.setattr(engine_mod, "_SCORE_IMAGES_TILES", 1)
    by_entry = {  # random, explicit, and both with carried sums
        "images": ("apc_score_images" if count <= 131072 else "apc_score_pairs", "apc_score_images",
                   "apc_score_images" if count <= 196608 else "apc_score_from_tiles", "apc_score_images"),
        "steps": ("apc_score_from_tiles",) * 4, "none": ("compact_records",) * 4}[room]
    if name == "stress_60" or name == "default_rows":  # a matrix may be too large for an image of finished entries
        by_entry = (("block_table_tiles",) if room == "images" else by_entry[:1]) + by_entry[1:]
    if room != "images":
        steps = (g.num_nodes + g.num_edges) * _lib.SCORE_STEP_BYTES
        scratch = eng._scratch
        monkeypatch.setattr(eng, "_scratch", lambda nbytes: scratch(nbytes) if room == "steps" and nbytes <= steps else None)
        monkeypatch.setattr(engine_mod, "_SCORE_IMAGES_UP_TO", 1 << 62)
    for clamp in (True, False):
        eng.build(clamp_inf=clamp)
        got = scores(*by_entry)
        monkeypatch.setattr(engine_mod, "_SCORE_FROM_TILES", False)
        want = scores(*["compact_records"] * 4)
        monkeypatch.setattr(engine_mod, "_SCORE_FROM_TILES", True)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        eng.set_node_multiplier(mult)  # the layout is kept, the multipliers are the call's


# a lane per assignment from tile images: rows of explicit choices brought in 16, 4 and 2 bytes a lane (by
# their number and where they start), two tiles ahead and one (from 768 lanes a workgroup), one launch and two;
# workgroups without a whole wavefront, and rows that end inside one
@pytest.mark.gpu
@pytest.mark.parametrize("name,count,skip", [
    ("moe_8x8", 8, 0), ("moe_8x8", 1002, 0), ("moe_8x8", 131080, 0), ("gpt2_2x3", 131080, 2), ("gpt2_2x3", 131082, 0),
    ("gpt2_2x3", 131080, 1), ("stress_60", 163848, 0), ("stress_60", 196616, 0), ("moe_8x8", 196618, 0),
    ("gpt2_2x3", 262160, 0), ("stress_60", 262154, 0)])
def test_images_have_the_bits_of_the_walk_over_records(name, count, skip, monkeypatch):
    g = GRAPHS[name]()
    eng = engine_mod.CostEngine(g, table_mode="full")
    eng.large_blocks = False
    eng.set_node_multiplier(np.arange(g.num_nodes) % 3 - 1)  # -1, 0, 1
    eng.build()
    gid = np.arange(g.num_nodes, dtype=np.int32) * 7 + 1
    gen = torch.Generator(device="cuda").manual_seed(count)
    nstrat = torch.from_numpy(g.node_nstrat.astype(np.int32)).cuda()[:, None]
    given = torch.empty(g.num_nodes * count + skip, dtype=torch.int16, device="cuda")[skip:].view(g.num_nodes, count)
    given.copy_(torch.randint(0, 1 << 30, (g.num_nodes, count), device="cuda", generator=gen, dtype=torch.int32) % nstrat)
    init = torch.rand((count, 6), dtype=torch.float64, device="cuda", generator=gen) * 1e6
    init[::3] = -0.0

    def scores(backend):
        out = []
        for score in (lambda: eng.score_random(11, 5, count), lambda: eng.score(given),
                      lambda: eng.score_random_window(11, 5, count, gid, 5, init=init),
                      lambda: eng.score_window(given, 5, init=init)):
            out.append(score().view(torch.int64))
            assert eng.last_score_backend == backend
        return out

    monkeypatch.setattr(engine_mod, "_SCORE_LANES_FROM", 1)
    monkeypatch.setattr(engine_mod, "_SCORE_TERMS_ABOVE", False)
    monkeypatch.setattr(engine_mod, "_SCORE_PAIRS_TILES", 1)
    monkeypatch.setattr(engine_mod, "_SCORE_IMAGES_TILES", 1)
    monkeypatch.setattr(engine_mod, "_SCORE_IMAGES_UP_TO", 1 << 20)
    monkeypatch.setattr(engine_mod, "_SCORE_PAIRS", False)
    got = scores("block_table_tiles")
    monkeypatch.setattr(engine_mod, "_SCORE_FROM_TILES", False)
    assert all(torch.equal(a, b) for a, b in zip(got, scores("compact_records")))

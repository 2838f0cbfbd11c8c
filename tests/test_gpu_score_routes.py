"""Which entry point scores a batch by default, on both sides of every line between two of them, and that the sums are
the same bits there as from the entry arrays."""
import numpy as np
import pytest
import torch

from autoparallel_amd import engine as engine_mod
from autoparallel_amd import graphgen
from autoparallel_amd.engine import CostEngine

pytestmark = pytest.mark.gpu

# blocks that images of finished entries take many of at a time and few (2.6), and large ones
GRAPHS = {
    "small": lambda: graphgen.gpt2_graph((4,), 4, vocab=4096, seq=512, batch=64),
    "middling": lambda: graphgen.stress_graph(130, (2, 2, 4), seed=1, s_min=34, s_max=38),
    "tiny": lambda: graphgen.stress_graph(30, (2, 2, 4), seed=1, s_min=2, s_max=20),  # 39 edges, three tiles
    "tiled": lambda: graphgen.stress_graph(100, (2, 2, 4), seed=1, s_min=10, s_max=60),  # 3.4 edges a tile
    "smallest": lambda: graphgen.gpt2_graph((4,), 1, vocab=4096, seq=512, batch=64),
    "large": lambda: graphgen.stress_graph(60, (2, 2, 4), seed=1, s_min=95, s_max=110),  # two pieces a matrix
    "larger": lambda: graphgen.stress_graph(200, (2, 2, 4), seed=1, s_min=95, s_max=100),
    "untiled": lambda: graphgen.stress_graph(30, (2, 2, 4), seed=1, s_min=2, s_max=150),  # small on average only
    "in_place": lambda: graphgen.stress_graph(40, (2, 2, 4), seed=1, s_min=140, s_max=170),  # three or four pieces a matrix
    "widest": lambda: graphgen.stress_graph(8, (2, 2, 4), seed=1, s_min=820, s_max=900),  # no list of pieces
}


@pytest.fixture(scope="module")
def engines():
    return {name: CostEngine(make(), table_mode="full").build() for name, make in GRAPHS.items()}


# kind: random, the same with carried sums, explicit
ROUTES = [
    ("small", "random", 256, "apc_score_fold_table"), ("small", "explicit", 257, "apc_score_terms"),
    ("smallest", "random", 257, "apc_score_fold_table"), ("smallest", "explicit", 1024, "apc_score_fold_table"),
    ("smallest", "carried", 2048, "apc_score_fold_table"), ("smallest", "random", 2049, "apc_score_terms"),
    ("large", "carried", 16384, "apc_score_fold_table"), ("large", "explicit", 16385, "apc_score_terms"),
    ("larger", "random", 640, "apc_score_fold_table"), ("larger", "random", 641, "apc_score_terms"),
    ("tiny", "random", 16384, "apc_score_fold_table"), ("tiny", "explicit", 32768, "apc_score_fold_table"),
    ("tiny", "carried", 32769, "apc_score_terms"), ("tiny", "random", 131072, "apc_score_images"),
    ("tiny", "random", 196609, "apc_score_from_tiles"), ("tiny", "explicit", 262144, "apc_score_images"),
    ("tiny", "explicit", 262145, "apc_score_from_tiles"), ("small", "random", 3000, "apc_score_terms"), ("small", "explicit", 3000, "apc_score_terms"),
    ("small", "random", 81920, "apc_score_terms"), ("small", "random", 81921, "apc_score_pairs"),
    ("middling", "random", 114688, "apc_score_terms"), ("middling", "random", 114689, "apc_score_images"),
    ("middling", "random", 131072, "apc_score_images"), ("middling", "random", 131073, "apc_score_pairs"),
    ("small", "carried", 114688, "apc_score_terms"), ("small", "carried", 114689, "apc_score_images"),
    ("small", "carried", 196608, "apc_score_images"), ("small", "carried", 196609, "apc_score_from_tiles"),
    ("small", "explicit", 81920, "apc_score_terms"), ("small", "explicit", 81921, "apc_score_images"),
    ("small", "explicit", 262145, "apc_score_images"), ("tiled", "explicit", 114688, "apc_score_terms"),
    ("tiled", "explicit", 114689, "apc_score_images"),
    ("large", "random", 131072, "apc_score_terms"), ("large", "carried", 131072, "apc_score_terms"),
    ("large", "random", 262144, "apc_score_stream"), ("large", "carried", 262144, "apc_score_stream"),
    ("large", "explicit", 196607, "apc_score_terms"), ("large", "explicit", 196608, "apc_score_table"),
    ("in_place", "random", 240000, "apc_score_terms"), ("in_place", "random", 300000, "apc_score_table"),
    ("in_place", "carried", 300000, "apc_score_table"), ("in_place", "random", 1 << 20, "apc_score_stream"),
    ("widest", "random", 163839, "apc_score_terms"), ("widest", "random", 163840, "apc_score_table"),
    ("widest", "carried", 163839, "apc_score_terms"), ("widest", "carried", 163840, "apc_score_table"),
    ("untiled", "random", 131072, "apc_score_terms"), ("untiled", "random", 131073, "apc_score_compact"),
    ("untiled", "carried", 131072, "apc_score_terms"), ("untiled", "carried", 131073, "apc_score_compact"),
    ("untiled", "explicit", 163840, "apc_score_terms"), ("untiled", "explicit", 163841, "apc_score_compact"),
]


@pytest.mark.parametrize("name,kind,count,entry", ROUTES)
def test_routes(engines, name, kind, count, entry, monkeypatch):
    eng = engines[name]
    g = eng.g
    gen = torch.Generator(device="cuda").manual_seed(count)
    ids = np.arange(g.num_nodes, dtype=np.int32)
    if kind == "explicit":
        nstrat = torch.from_numpy(g.node_nstrat.astype(np.int32)).cuda()[:, None]
        assign = (torch.randint(0, 1 << 30, (g.num_nodes, count), device="cuda", generator=gen, dtype=torch.int32)
                  % nstrat).to(torch.int16)
    elif kind == "carried":
        init = torch.rand((count, 6), dtype=torch.float64, device="cuda", generator=gen)

    def score():
        out = (eng.score(assign) if kind == "explicit" else eng.score_random(11, 5, count) if kind == "random"
               else eng.score_random_window(11, 5, count, ids, 3, init=init))
        return out.view(torch.int64), eng.last_score_entry, eng.last_score_backend

    got = score()
    assert got[1] == entry and got[2].startswith("block_table") == (entry != "apc_score_compact")
    monkeypatch.setattr(engine_mod, "_SCORE_FROM_TABLE", False)
    monkeypatch.setattr(engine_mod, "_SCORE_SMALL_FROM_TABLE", False)
    want = score()
    assert want[2] == ("compact_records" if count >= 32768 else "entry_arrays") and torch.equal(got[0], want[0])


def test_no_list_of_pieces_is_made_to_choose_the_terms():
    eng = CostEngine(GRAPHS["large"](), table_mode="full").build()
    eng.score_random(11, 5, 131072)
    assert eng.last_score_entry == "apc_score_terms" and not eng._layouts["score_pieces"]
    eng.score_random(11, 5, 262144)
    assert eng.last_score_entry == "apc_score_stream" and eng._layouts["score_pieces"][0] is not None


@pytest.mark.parametrize("eager,entry", [(300000, "apc_score_table"), (1 << 20, "apc_score_stream")])
def test_a_recorded_batch_takes_the_walk_whose_layout_is_there(eager, entry):
    """Nothing can be copied to the device meanwhile: edge by edge, where that is faster and its records were made, else the
    stream, where its list was."""
    count = 300000
    eng = CostEngine(GRAPHS["in_place"](), table_mode="full").build()
    eng.score_random(11, 5, eager)
    assert eng.last_score_entry == entry
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = eng.score_random(11, 5, count)
    assert eng.last_score_entry == entry
    want = eng.score_random(11, 5, count)
    assert eng.last_score_entry == "apc_score_table"
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int64), want.view(torch.int64))
        want = eng.score_random(11, 5, count)

"""Scores follow the entry arrays, whatever a batch is scored from: edits in place, arrays put in
another's place, builds and edits replayed from a graph.  Wanted sums: those of a second engine that
adopted the arrays as they are (load_results), which has no block table to go by."""
import numpy as np
import pytest
import torch

from autoparallel_amd import engine as engine_mod
from autoparallel_amd import graphgen
from autoparallel_amd.engine import CostEngine

pytestmark = pytest.mark.gpu

COUNTS = [70, 40000, 140000]  # terms side by side, the same from the table, by tiles (or the table edge by edge)


@pytest.fixture(scope="module", params=["small_blocks", "large_blocks"])
def engines(request):
    g = graphgen.gpt2_graph((2, 3), 1, vocab=4096, seq=512, batch=64)
    eng, other = CostEngine(g, table_mode="full"), CostEngine(g, table_mode="full")
    eng.large_blocks = request.param == "large_blocks"
    return eng, other


def _bits(t):
    return t.cpu().numpy().view(np.uint64)


def _as_the_arrays_are(eng, other, count):
    other.load_results(**{k: getattr(eng, k).cpu().numpy() for k in ("comm", "cost", "flags", "compute", "per_arg")})
    return _bits(other.score_random(5, 9, count))


def _table_backend(eng, count):
    if count < 131072:
        return "block_table_terms"
    return "block_table" if eng.large_blocks else "block_table_tiles"


@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("array", ["cost", "comm"])
def test_edits_in_place_are_followed(engines, array, count):
    eng, other = engines
    eng.build()
    built = _bits(eng.score_random(5, 9, count))
    assert eng.last_score_backend == _table_backend(eng, count)
    assert (built == _as_the_arrays_are(eng, other, count)).all()
    for _ in range(2):  # again after records were made of the first edit
        getattr(eng, array).mul_(2.0)
        got = _bits(eng.score_random(5, 9, count))
        assert (got == _as_the_arrays_are(eng, other, count)).all() and not (got == built).all()
    eng.build()  # rewrites the arrays: the table stands for them again
    assert (_bits(eng.score_random(5, 9, count)) == built).all()
    assert eng.last_score_backend == _table_backend(eng, count)


@pytest.mark.parametrize("count", COUNTS[:2])
def test_arrays_without_edit_counters_are_read(engines, count):
    """Tensors made under inference mode count no edits: what is scored after a build is the arrays."""
    other = engines[1]
    with torch.inference_mode():
        eng = CostEngine(engines[0].g, table_mode="full").build()
        eng.cost.mul_(2.0)
        got = _bits(eng.score_random(5, 9, count))
        assert eng.last_score_backend == ("entry_arrays" if count < 32768 else "records")
    assert (got == _as_the_arrays_are(eng, other, count)).all()


@pytest.mark.parametrize("count", COUNTS)
def test_an_array_in_anothers_place_is_scored(engines, count):
    """The builds write the arrays the engine was made with; a tensor put in the place of one of them
    is what the scorers read, also where its edit counter is that of the array it replaced."""
    eng, other = engines
    eng.build()
    built, cost = _bits(eng.score_random(5, 9, count)), eng.cost
    keep = cost.data
    try:
        for put in (lambda: setattr(eng, "cost", cost * 2.0), lambda: setattr(cost, "data", keep * 2.0)):
            put()
            for _ in range(2):
                got = _bits(eng.score_random(5, 9, count))
                assert (got == _as_the_arrays_are(eng, other, count)).all() and not (got == built).all()
                eng.build()  # into ``keep``
            eng.cost, cost.data = cost, keep
    finally:
        eng.cost, cost.data = cost, keep
    eng.build()
    assert (_bits(eng.score_random(5, 9, count)) == built).all()
    assert eng.last_score_backend == _table_backend(eng, count)


def test_builds_ask_for_edits_only_where_a_caller_edits(engines, monkeypatch):
    eng = CostEngine(engines[0].g, table_mode="full").build()
    asked = []
    count = engine_mod._edit_count
    monkeypatch.setattr(engine_mod, "_edit_count", lambda t: asked.append(t) or count(t))
    eng.build()
    assert not asked
    built = _bits(eng.score_random(5, 9, 70))
    assert eng.last_score_backend == "block_table_terms"
    eng.cost.mul_(2.0)
    eng.build()  # the edit is overwritten before it was seen: until the next build the arrays are read
    assert (_bits(eng.score_random(5, 9, 70)) == built).all() and eng.last_score_backend == "entry_arrays"
    for rewrite in (lambda: None, lambda: eng.cost.mul_(2.0), lambda: _as_the_arrays_are(eng, eng, 70)):
        rewrite()
        eng.build()
        assert (_bits(eng.score_random(5, 9, 70)) == built).all() and eng.last_score_backend == "block_table_terms"


@pytest.mark.parametrize("count", COUNTS)
def test_replayed_builds_count(engines, count):
    """A recorded build leaves its own clamp in the arrays whenever it is replayed; scores follow,
    and where every recorded build has the last build's clamp the table goes on standing for them."""
    eng = CostEngine(engines[0].g, table_mode="full")
    eng.large_blocks = engines[0].large_blocks
    other = engines[1]
    graph = eng.capture_build(True)
    for _ in range(3):
        eng.build(True)
        assert (_bits(eng.score_random(5, 9, count)) == _as_the_arrays_are(eng, other, count)).all()
        assert eng.last_score_backend == _table_backend(eng, count)
        graph.replay()
        assert (_bits(eng.score_random(5, 9, count)) == _as_the_arrays_are(eng, other, count)).all()
        for change in (lambda: eng.build(False), lambda: eng.apply_prefetch_discount(0.5)):
            change()
            assert (_bits(eng.score_random(5, 9, count)) == _as_the_arrays_are(eng, other, count)).all()
            graph.replay()
            assert (_bits(eng.score_random(5, 9, count)) == _as_the_arrays_are(eng, other, count)).all()


def test_recorded_edits_and_entries_count(engines):
    eng = CostEngine(engines[0].g, table_mode="full")
    other = engines[1]
    for record in (lambda: eng.edge_costs(clamp_inf=False), lambda: (eng.cost.mul_(2.0), eng.mark_results_edited())):
        eng.build(True)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            record()
        for _ in range(2):
            eng.build(True)
            graph.replay()
            assert (_bits(eng.score_random(5, 9, 70)) == _as_the_arrays_are(eng, other, 70)).all()


@pytest.mark.parametrize("count", COUNTS)
def test_a_build_that_is_only_recorded_rewrites_nothing(engines, count):
    eng = CostEngine(engines[0].g, table_mode="full")
    eng.large_blocks = engines[0].large_blocks
    other = engines[1]
    for change in (lambda: eng.apply_prefetch_discount(0.5), lambda: eng.cost.mul_(2.0), lambda: eng.build(False)):
        eng.build(True)
        eng.score_random(5, 9, count)
        change()
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            eng.build(True)
        assert (_bits(eng.score_random(5, 9, count)) == _as_the_arrays_are(eng, other, count)).all()
        graph.replay()
        assert (_bits(eng.score_random(5, 9, count)) == _as_the_arrays_are(eng, other, count)).all()


@pytest.mark.parametrize("count", COUNTS)
def test_builds_and_scores_recorded_together(engines, count):
    """Replays give what the recorded build and edits leave, whatever was built eagerly before."""
    eng = CostEngine(engines[0].g, table_mode="full")
    eng.large_blocks = engines[0].large_blocks
    other = engines[1]
    eng.build(False)
    eng.score_random(5, 9, count)
    for record in (lambda: eng.build(True), lambda: eng.build(False), lambda: eng.build(True).cost.mul_(2.0),
                   lambda: (eng.build(True), eng.edge_costs(clamp_inf=False))):
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            record()
            out = eng.score_random(5, 9, count)
        for _ in range(3):
            graph.replay()
            assert (_bits(out) == _as_the_arrays_are(eng, other, count)).all()
            eng.build(False)


@pytest.mark.parametrize("explicit", [False, True])
def test_a_recorded_small_score_reads_the_arrays(engines, explicit):
    """Replays of a recorded score follow builds, edits and discounts between them."""
    eng, other = engines
    g = eng.g
    rng = np.random.default_rng(1)
    rows = (rng.integers(0, 1 << 20, (g.num_nodes, 70)) % g.node_nstrat[:, None]).astype(np.int16)
    assign = torch.from_numpy(rows).cuda()
    score = (lambda e: e.score(assign)) if explicit else (lambda e: e.score_random(5, 9, 70))
    eng.build()
    score(eng)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = score(eng)
    for change in (lambda: eng.build(True), lambda: eng.apply_prefetch_discount(0.5), lambda: eng.cost.mul_(2.0),
                   lambda: eng.build(False), lambda: eng.build(True)):
        change()
        graph.replay()
        _as_the_arrays_are(eng, other, 70)
        assert (_bits(out) == _bits(score(other))).all()
    assert torch.equal(out.view(torch.int64), score(eng).view(torch.int64))


def test_scores_and_draws_are_recorded_without_a_layout_at_hand(engines):
    """A layout cannot be copied to the device while a graph is recorded: a call whose layout is not
    there yet is recorded over another route, with the same results on every replay."""
    eng = CostEngine(engines[0].g, table_mode="full")
    g = eng.g
    n = 140000
    gen = torch.Generator(device="cuda").manual_seed(2)
    nstrat = torch.from_numpy(g.node_nstrat.astype(np.int32)).cuda()[:, None]
    assign = (torch.randint(0, 1 << 30, (g.num_nodes, n), device="cuda", generator=gen, dtype=torch.int32)
              % nstrat).to(torch.int16)
    drawn = torch.zeros((g.num_nodes, 300), dtype=torch.int16, device="cuda").view(torch.uint16)
    eng.build()
    eng.sample_feasible(3, 0, 300)
    eng.score_random(5, 9, 40000)
    torch.cuda.synchronize()
    calls = [lambda: eng.score_random(5, 9, n), lambda: eng.score(assign), lambda: eng.score_window(assign, 5),
             lambda: eng.sample_feasible(3, 0, 300, first_node=7, assign=drawn)[0].view(torch.int16).clone()]
    recorded = []
    for call in calls:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = call()
        recorded.append((graph, out))
    for _ in range(3):
        for call, (graph, out) in zip(calls, recorded):
            out.zero_()
            graph.replay()
            got = out.cpu().numpy().tobytes()
            want = call()
            torch.cuda.synchronize()
            assert got == want.cpu().numpy().tobytes()


def test_layouts_stay_where_they_are(engines):
    """A launch on another stream or in a graph may still read a layout when another first_node is
    asked for: none is let go or moved while the engine lives, and only so many are made."""
    eng = engines[0]
    eng.build()
    eng.sample_feasible(3, 0, 64)
    kinds = [lambda v: eng._score_tiles(v, False), lambda v: eng._score_tiles(v, True), eng._sample_steps]
    for kind in kinds:
        first = kind(0)
        for v in range(1, 40):
            kind(v)
        assert kind(0) is first
        assert sum(kind(v) is not None for v in range(40)) == engine_mod._LAYOUTS_KEPT

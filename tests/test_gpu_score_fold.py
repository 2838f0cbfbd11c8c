"""Small batches are scored in groups of 4 to 64 assignments whose terms are gathered side by
side; every row has to have the bits of the walk that takes one lane per assignment."""
import numpy as np
import pytest
import torch

from autoparallel_amd import engine as engine_mod
from autoparallel_amd import graphgen
from autoparallel_amd.engine import CostEngine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engines():
    model = graphgen.gpt2_graph((2, 3), 1, vocab=4096, seq=512, batch=64)
    window, gid, first_node = graphgen.stress_dag_window(2000, 600, 633, (2, 2), seed=0)
    return (CostEngine(model).build(), None, 0), (CostEngine(window).build(), gid, first_node)


def _bits(t):
    return t.cpu().numpy().view(np.uint64)


# 1 << shift assignments a workgroup: up to 1024, 4096, 8192, 16383, and beyond
@pytest.mark.parametrize("count", [1, 3, 5, 1024, 1025, 4096, 4097, 8193, 16383, 16385])
@pytest.mark.parametrize("which", [0, 1])
def test_groups_have_the_bits_of_the_lane_walk(engines, which, count, monkeypatch):
    eng, gid, first_node = engines[which]
    g = eng.g
    rng = np.random.default_rng(count)
    assign = torch.from_numpy((rng.integers(0, 1 << 20, (g.num_nodes, count)) % g.node_nstrat[:, None]).astype(np.int16)).cuda()
    init = torch.from_numpy(rng.integers(0, 1000, (count, 6)).astype(np.float64)).cuda()
    ids = np.arange(g.num_nodes, dtype=np.int32) if gid is None else gid

    def all_scores():
        return [_bits(x) for x in (
            eng.score_random(11, 5, count), eng.score(assign),
            eng.score_random_window(11, 5, count, ids, first_node, init=init),
            eng.score_random_window(11, 5, count, ids, g.num_nodes, init=init),  # nothing to add
            eng.score_window(assign, first_node, init=init))]

    from_table = all_scores()
    monkeypatch.setattr(engine_mod, "_SCORE_SMALL_FROM_TABLE", False)
    from_arrays = all_scores()
    monkeypatch.setattr(engine_mod, "_SCORE_LANES_FROM", 1)  # one lane per assignment, from records
    monkeypatch.setattr(engine_mod, "_SCORE_FROM_TABLE", False)
    want = all_scores()
    for a, b, c in zip(from_table, from_arrays, want):
        assert (a == c).all() and (b == c).all()


def test_the_table_stands_for_the_arrays_only_while_it_does(engines):
    """Clamped and unclamped builds; and where the arrays were edited, the arrays decide."""
    eng = engines[0][0]
    for clamp in (False, True):
        eng.build(clamp_inf=clamp)
        got = _bits(eng.score_random(3, 0, 70))
        eng.mark_results_edited()  # from here on the arrays are read
        assert (got == _bits(eng.score_random(3, 0, 70))).all()
    for array in (eng.cost, eng.comm):  # an edit in place is noticed without being told
        eng.build()
        got = _bits(eng.score_random(3, 0, 70))
        array.mul_(2.0)
        assert not (got == _bits(eng.score_random(3, 0, 70))).all()
    eng.build()

"""The layout of a feasible draw in steps (apc_sample_steps, host) and the draw over it: every
node once, behind its producers, its choices found where they are; the same draws as by the walk
with one lane per assignment."""
import ctypes as C

import numpy as np
import pytest
import torch

from autoparallel_amd import _lib, graphgen
from autoparallel_amd import engine as engine_mod

REC = np.dtype([("node", "<i4"), ("nstrat", "<i4"), ("n_arg", "<i4"), ("reserved", "<i4"),
                ("arg", [("from", "<u4"), ("col", "<u4")], 6)])
RING = 128


def _layout(edge_off, src, nstrat, col_off, first_node, n_waves):
    n = len(nstrat) - first_node
    max_step = n + 128 * int((np.diff(edge_off) > 6).sum())
    recs = np.zeros(max_step * 16, REC)
    n_step, waves = C.c_int32(), C.c_int32()
    a = [np.ascontiguousarray(x, t) for x, t in ((edge_off, np.int32), (src, np.int32), (nstrat, np.int32),
                                                 (col_off, np.int64))]
    rc = _lib.load().apc_sample_steps(len(nstrat), len(src), *[x.ctypes.data for x in a], first_node, n_waves,
                                      recs.ctypes.data, max_step, C.byref(n_step), C.byref(waves))
    _lib.check(rc, "apc_sample_steps")
    return recs[:n_step.value * waves.value].reshape(n_step.value, waves.value), waves.value


@pytest.mark.parametrize("n_waves", [0, 2, 16])
@pytest.mark.parametrize("first_node", [0, 7])
@pytest.mark.parametrize("reach", [2, 40, 400])  # how far back the producers lie: chains to wide graphs
def test_layout(n_waves, first_node, reach):
    rng = np.random.default_rng(reach)
    n = 400
    n_arg = rng.choice([0, 1, 1, 2, 3, 6, 7, 9], n)
    edge_off = np.concatenate([[0], np.cumsum(n_arg)])
    src = np.concatenate([[int(rng.integers(max(0, v - reach), v)) if v and rng.random() < 0.9 else -1
                           for _ in range(n_arg[v])] for v in range(n)]).astype(np.int32)
    nstrat = rng.integers(1, 300, n)
    col_off = 2 * rng.integers(0, 1 << 31, len(src))
    recs, waves = _layout(edge_off, src, nstrat, col_off, first_node, n_waves)
    assert recs.dtype.itemsize == _lib.SAMPLE_REC_BYTES and waves in (2, 16) and n_waves in (0, waves)
    place = np.full(n, -1)
    flat = recs.reshape(-1)
    at = np.nonzero(flat["node"] >= 0)[0]
    place[flat["node"][at]] = at
    assert len(at) == n - first_node and (np.sort(flat["node"][at]) == np.arange(first_node, n)).all()
    settled = RING // waves  # steps behind which a choice has left the ring and is in the matrix
    for q in at:
        r, step = flat[q], q // waves
        v = int(r["node"])
        assert r["nstrat"] == nstrat[v] and r["n_arg"] == n_arg[v]
        for i in range(n_arg[v]):
            u = int(src[edge_off[v] + i])
            inside = u >= first_node
            assert not inside or place[u] // waves < step
            if i >= 6:
                assert not inside or place[u] // waves <= step - settled
                continue
            assert r["arg"][i]["col"] == col_off[edge_off[v] + i] // 2
            slot, named = int(r["arg"][i]["from"]) >> 24, int(r["arg"][i]["from"]) & 0xFFFFFF
            if u < 0:
                assert (slot, named) == (RING, 0)
            elif slot == 255:
                assert named == u and (not inside or place[u] // waves <= step - settled)
            else:
                assert named == u and slot == place[u] % RING and place[u] + RING >= (step + 1) * waves


def test_layout_refuses():
    off, src, one = [0, 0, 1], [1], [1, 1]
    with pytest.raises(_lib.ApcError):  # a producer that is not in front of its consumer
        _layout(off, src, one, [0], 0, 2)
    with pytest.raises(_lib.ApcError):  # an odd column offset
        _layout(off, [0], one, [3], 0, 2)
    with pytest.raises(_lib.ApcError):
        _layout(off, [0], one, [0], 0, 3)


def test_layout_says_when_there_are_more_steps_than_room():
    """A chain of nodes with seven argument rows: each waits until its producer has left the ring."""
    n = 40
    src = np.repeat(np.arange(-1, n - 1), 7).astype(np.int32)
    recs, n_step, waves = np.zeros(129 * n * 16, REC), C.c_int32(), C.c_int32()
    a = [np.ascontiguousarray(x, t) for x, t in ((7 * np.arange(n + 1), np.int32), (src, np.int32),
                                                 (np.full(n, 5), np.int32), (np.zeros(7 * n), np.int64))]

    def steps(room):
        rc = _lib.load().apc_sample_steps(n, 7 * n, *[x.ctypes.data for x in a], 0, 2, recs.ctypes.data, room,
                                          C.byref(n_step), C.byref(waves))
        return rc, n_step.value

    rc, most = steps(129 * n)
    assert rc == 0 and most > 60 * (n - 1)
    assert steps(most) == (0, most)
    for room in (most - 1, n):
        assert steps(room) == (_lib.ERR_UNSUPPORTED, 0)


def _long_rows(chain):
    """Nodes with eight argument rows, one after the other or among many of one row."""
    import itertools

    from autoparallel_amd import packed
    from autoparallel_amd.packed import GraphBuilder, NodeDesc

    b = GraphBuilder((2, 2), 4)
    m = b.meta((8, 16, 32), (512, 32, 1), 4, packed.DT_F32)
    tuples = list(itertools.product([0x00, 0x40, 0x41, 0x42, 0x80], repeat=2))
    rng = np.random.default_rng(1)

    def specs(n):
        return [b.spec(m, tuples[i]) for i in rng.choice(len(tuples), n, replace=False)]

    first = specs(6)
    at = [b.add_node(NodeDesc("first", in_specs=[[x] for x in first], out_specs=[[x] for x in first], inputs=[],
                              default_rows=[[[0.0]] for _ in first]))]
    for v in range(1, 20 if chain else 400):
        s, rows = specs(int(rng.integers(2, 12))), 8 if chain or v % 100 == 0 else 1
        inputs = [at[-1]] * 8 if chain else [int(x) for x in rng.integers(max(0, v - 300), v, rows)]
        at.append(b.add_node(NodeDesc(f"n{v}", in_specs=[[x] * rows for x in s], out_specs=[[x] for x in s],
                                      inputs=inputs)))
    return b.pack(), None, 0


GRAPHS = {
    "long_rows": lambda: _long_rows(False),
    "gpt2": lambda: (graphgen.gpt2_graph((2, 3), 2, vocab=4096, seq=512, batch=64), None, 0),
    "llama_8x8": lambda: (graphgen.llama_graph((8, 8), 1, 1024, 8, 4, 2048, 8192, 512, 16), None, 0),
    "stress_512": lambda: (graphgen.stress_graph(60, (2, 2, 4), seed=4, s_min=2, s_max=700), None, 0),
    "window": lambda: graphgen.stress_dag_window(2000, 600, 700, (2, 2), seed=0),
}


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 63, 65, 1000])
@pytest.mark.parametrize("n_waves", [2, 16])
@pytest.mark.parametrize("name", list(GRAPHS))
def test_draws_equal_the_lane_walks(name, n_waves, count, monkeypatch):
    g, gid, first_node = GRAPHS[name]()
    eng = engine_mod.CostEngine(g).build()
    rng = np.random.default_rng(count)
    filters = {v: rng.random(int(g.node_nstrat[v])) < 0.7 for v in range(first_node, g.num_nodes, 3)}
    given = (rng.integers(0, 1 << 20, (g.num_nodes, count)) % g.node_nstrat[:, None]).astype(np.int16)

    def draws():
        out = []
        for row_filter in (None, filters):
            assign = torch.from_numpy(given).cuda().view(torch.uint16)
            a, f = eng.sample_feasible(3, 17, count, node_gid=gid, first_node=first_node, assign=assign,
                                       row_filter=row_filter) if first_node else \
                eng.sample_feasible(3, 17, count, row_filter=row_filter)
            out += [a.view(torch.int16).cpu().numpy(), f.cpu().numpy()]
        return out

    monkeypatch.setattr(engine_mod, "_SAMPLE_WAVES", n_waves)
    got = draws()
    assert eng._sample_steps(first_node)[2] == n_waves
    monkeypatch.setattr(engine_mod, "_SAMPLE_LANES_FROM", {2: 0, 16: 0})
    for a, b in zip(got, draws()):
        assert (a == b).all()


@pytest.mark.gpu
def test_a_chain_of_long_argument_rows_is_drawn_by_lanes():
    eng = engine_mod.CostEngine(_long_rows(True)[0]).build()
    eng.sample_feasible(3, 17, 64)
    assert eng._sample_steps(0) is None

"""The walk that keeps the schedule in LDS, by the streams it tells apart (up to four, up to eight): memory and timeline
on wavefronts of their own, against the oracle."""
import dataclasses

import numpy as np
import pytest

from autoparallel_amd import schedule_metrics as SM
from oracle import schedule_oracle as SO


@pytest.mark.gpu
@pytest.mark.parametrize("n_stream", [1, 2, 4, 5, 8])
@pytest.mark.parametrize("n_layers,copies", [(4, 1), (20, 1), (4, 300)])  # 64 walks over one, two and four wavefronts
def test_streams_against_the_oracle(n_stream, n_layers, copies):
    ps = SM.synthetic_schedule(n_layers, seed=2)
    rng = np.random.default_rng(n_stream)
    own = (ps.stream != 0) & (n_stream > 1)
    # collectives on any stream but the first, computations on some, and collectives that are waited for at once
    stream = np.where(own, rng.integers(1, max(n_stream, 2), ps.n_node), 0)
    plain = (ps.flags & SM.SCHED_COMM) == 0
    stream = np.where(plain & (rng.random(ps.n_node) < 0.2), rng.integers(0, n_stream, ps.n_node), stream)
    flags = ps.flags | np.where((stream != 0) & (rng.random(ps.n_node) < 0.3), SM.SCHED_SYNC, 0)
    ps = dataclasses.replace(ps, stream=stream.astype(ps.stream.dtype), flags=flags.astype(ps.flags.dtype), n_stream=n_stream)
    ps.validate()
    orders = ps.random_orders(67, seed=3)
    want = [SO.schedule_metrics(ps, order) for order in orders]
    times, peak = SM.ScheduleEstimator(ps).evaluate(np.tile(orders, (copies, 1)))
    for b in range(len(orders)):
        assert tuple(times[b]) == want[b][:4] and int(peak[b]) == want[b][4], (b, times[b], peak[b], want[b])
    assert (times.reshape(copies, len(orders), 4) == times[:len(orders)]).all()
    assert (peak.reshape(copies, len(orders)) == peak[:len(orders)]).all()
    own_order, own_peak = SM.ScheduleEstimator(ps).evaluate()
    assert tuple(own_order[0]) == want[0][:4] and int(own_peak[0]) == want[0][4]

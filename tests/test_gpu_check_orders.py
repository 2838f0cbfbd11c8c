"""apc_check_orders: a batch of orders passes where every row names each node once."""
import ctypes as C

import numpy as np
import pytest
import torch

from autoparallel_amd import _lib

pytestmark = pytest.mark.gpu


def _bad(orders):
    d = torch.from_numpy(np.ascontiguousarray(orders, np.int32)).cuda()
    bad = torch.zeros(1, dtype=torch.int32, device="cuda")
    _lib.check(_lib.load().apc_check_orders(d.data_ptr(), d.shape[0], d.shape[1], bad.data_ptr(),
                                            C.c_void_p(torch.cuda.current_stream().cuda_stream)), "apc_check_orders")
    return int(bad.item()) != 0


@pytest.mark.parametrize("n_sched", [1, 5, 9000])  # more rows than the launch has wavefronts
@pytest.mark.parametrize("n_node", [1, 31, 32, 33, 64, 65, 700])
def test_check_orders(n_node, n_sched):
    rng = np.random.default_rng(n_node)
    orders = rng.permuted(np.tile(np.arange(n_node), (n_sched, 1)), axis=1)
    assert not _bad(orders)
    for row, col, value in ((n_sched - 1, n_node - 1, n_node), (0, 0, -1), (n_sched // 2, n_node // 2, 2**31 - 1)):
        wrong = orders.copy()
        wrong[row, col] = value
        assert _bad(wrong)
    if n_node > 1:  # one node twice
        wrong = orders.copy()
        wrong[n_sched - 1, 0] = wrong[n_sched - 1, n_node - 1]
        assert _bad(wrong)


def test_check_orders_at_the_limit():
    """131 072 nodes: four bitmaps fill the 64 KB of LDS a launch may ask for."""
    limit = _lib.CHECK_MAX_NODES
    rng = np.random.default_rng(0)
    orders = np.stack([rng.permutation(limit) for _ in range(6)])
    assert not _bad(orders)
    for row, col, value in ((5, limit - 1, limit), (0, 0, -1)):
        wrong = orders.copy()
        wrong[row, col] = value
        assert _bad(wrong)
    for row in (0, 3, 5):  # one node twice, in the bitmap of the first and the last wavefront too
        wrong = orders.copy()
        wrong[row, 17] = wrong[row, limit - 1]
        assert _bad(wrong)
    d = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert _lib.load().apc_check_orders(d.data_ptr(), 1, limit + 1, d.data_ptr(), None) != 0  # refused by the host

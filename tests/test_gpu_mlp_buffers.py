"""Inference through the buffers kept with a network (pinned rows for small
calls, device rows for larger ones, a call's own above and beside another
call): every size gives the rows' values of any other size bit for bit, in any
order of sizes and from two threads at once."""
import threading

import numpy as np
import pytest

from peridem_amd import capi

pytestmark = pytest.mark.gpu

SIZES = (1, 17, 256, 257, 5000, 16384, 16385, 100, 262144, 262145, 3)


def _net():
    net = capi.Mlp(3)
    x = np.random.default_rng(1).normal(size=(max(SIZES), 16)).astype(np.float32)
    return net, x


def test_sizes_agree():
    net, x = _net()
    ref = net.forward(x)
    assert np.isfinite(ref).all() and np.ptp(ref) > 0
    for n in SIZES:
        print(f"[mlp buffers] rows={n}", flush=True)
        np.testing.assert_array_equal(net.forward(x[-n:]), ref[-n:])
    net.close()


@pytest.mark.parametrize("sizes", [(17, 400), (20000, 64), (20000, 30000)])
def test_two_threads_share_a_network(sizes):
    net, x = _net()
    ref = net.forward(x[:31000])
    bad = []

    def work(n):
        for k in range(50):
            if not np.array_equal(net.forward(x[k:k + n]), ref[k:k + n]):
                bad.append((n, k))

    ts = [threading.Thread(target=work, args=(n,)) for n in sizes]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    net.close()

"""The row pointers of pdem_mlp_forward: host or device memory, in any
combination and at every size class of the kept buffers; null is refused."""
import ctypes as C

import numpy as np
import pytest
import torch

from peridem_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 17, 16384, 16385, 300000])
def test_device_rows(rows):
    print(f"[mlp pointers] rows={rows}", flush=True)
    net = capi.Mlp(3)
    x = np.random.default_rng(2).normal(size=(rows, 16)).astype(np.float32)
    ref = net.forward(x)
    xd = torch.from_numpy(x).cuda()
    for x_dev in (False, True):
        for y_dev in (False, True):
            y = np.zeros((rows, 4), np.float32)
            yd = torch.zeros(rows, 4, device="cuda")
            torch.cuda.synchronize()
            rc = net.lib.pdem_mlp_forward(
                net.h, C.cast(xd.data_ptr() if x_dev else x.ctypes.data, C.POINTER(C.c_float)), rows,
                C.cast(yd.data_ptr() if y_dev else y.ctypes.data, C.POINTER(C.c_float)))
            assert rc == 0, net.lib.pdem_mlp_last_error(net.h)
            np.testing.assert_array_equal(yd.cpu().numpy() if y_dev else y, ref)
    net.close()


@pytest.mark.parametrize("rows", [1, 20000])
def test_null_rows_are_refused(rows):
    net = capi.Mlp(3)
    x = np.zeros((rows, 16), np.float32)
    y = np.zeros((rows, 4), np.float32)
    f = C.POINTER(C.c_float)
    assert net.lib.pdem_mlp_forward(net.h, None, rows, y.ctypes.data_as(f)) != 0
    assert net.lib.pdem_mlp_forward(net.h, x.ctypes.data_as(f), rows, None) != 0
    assert net.forward(x).shape == (rows, 4)  # the network goes on
    net.close()

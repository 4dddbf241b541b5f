"""mlp_forward with its result over its input (shifted both ways, row for row in its
place, directly after it): the same bits as into a buffer of its own."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(13, 64, 180), (70, 128, 9), (33, 64, 33)])
def test_result_over_the_input(dims):
    from mpifdtd_amd import surrogate as S
    from mpifdtd_amd._native import check, lib
    B = 700
    rng = np.random.default_rng(3)
    x = rng.random((B, dims[0])).astype(np.float32)
    net = S.MLP(list(dims), batch_max=B, seed=2)
    want = net.forward(x)
    nx, ny = x.size, want.size
    # element offsets of x and y in one buffer
    for ox, oy in ((0, 0), (5, 0), (0, 40), (ny - 3, 0), (0, nx), (ny, 0)):
        print(dims, ox, oy, flush=True)
        host = np.zeros(nx + ny, np.float32)
        host[ox:ox + nx] = x.ravel()
        buf = S.DeviceArray(host)
        at = lambda o: ctypes.c_void_p(buf.ptr.value + 4 * o)
        check(lib().mlp_forward(net._h, at(ox), B, at(oy)), "mlp_forward")
        got = buf.numpy()[oy:oy + ny].reshape(want.shape)
        assert np.array_equal(got, want), (ox, oy)

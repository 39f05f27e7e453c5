"""A training pass whose activations do not fit the GPU is refused before any
launch, and the network goes on as before."""
import ctypes as ct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_network_after_a_refused_allocation():
    from primaldualtoolbox import _capi as C
    from primaldualtoolbox import warmstart as ws
    net = ws.WarmStartCNN(depth=5, seed=3)
    rng = np.random.default_rng(0)
    n, h, w = 1, 24, 40
    x = C.DeviceArray.from_numpy(rng.standard_normal(n * h * w * 2).astype(np.float32))
    t = C.DeviceArray.from_numpy(rng.standard_normal(n * h * w * 6).astype(np.float32))

    def gradient(vx, vt, n, h, w):
        g, loss = np.empty(net.n_params, np.float32), ct.c_double()
        C.check(C.lib().pdt_cnn_loss_grad(net._h, vx.h, vt.h, n, h, w, ct.byref(loss),
                                          g.ctypes.data_as(ct.POINTER(ct.c_float)), g.size))
        return loss.value, g

    before = gradient(x, t, n, h, w)
    # 2^36 pixels, 4 TB a layer (the arrays only claim the size: nothing of them is read)
    big = (65536, 1024, 1024)
    px = big[0] * big[1] * big[2]
    vx = C.DeviceArray.wrap(C.PDT_F32, [2 * px], x.device_ptr(), owner=x)
    vt = C.DeviceArray.wrap(C.PDT_F32, [6 * px], t.device_ptr(), owner=t)
    with pytest.raises(C.PdtError, match="memory"):
        gradient(vx, vt, *big)
    after = gradient(x, t, n, h, w)
    assert after[0] == before[0]
    np.testing.assert_array_equal(after[1], before[1])

"""Non-finite pixels in the network's input: they change the outputs whose
receptive field (depth pixels each way) holds them, in the one-launch inference
with the same bits as in the per-layer kernels, and no others.  A NaN that
reaches a hidden layer is zero behind its ReLU, max(NaN, 0) = 0: a NaN pixel
makes no output NaN, and an infinity need not make any infinite (the next layer
adds infinities of both signs, which is NaN again)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _per_layer(C, net, x):
    """(an output array that covers the input takes the per-layer kernels)"""
    n, h, w, _ = x.shape
    px = n * h * w
    buf = C.DeviceArray.from_numpy(np.concatenate([x.reshape(-1), np.zeros(4 * px, np.float32)]))
    vx = C.DeviceArray.wrap(C.PDT_F32, [2 * px], buf.device_ptr(), owner=buf)
    C.check(C.lib().pdt_cnn_forward(net._h, vx.h, buf.h, n, h, w))
    return buf.numpy().reshape(n, h, w, 6)


@pytest.mark.parametrize("depth", [2, 5, 8])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("y,x", [(30, 23), (0, 0), (59, 69)])
def test_neighbourhood_of_a_non_finite_pixel(depth, value, y, x):
    from primaldualtoolbox import _capi as C
    from primaldualtoolbox import warmstart as ws
    net = ws.WarmStartCNN(depth=depth, seed=9)
    img = np.random.default_rng(2).standard_normal((1, 60, 70, 2)).astype(np.float32)
    want = net.forward(img)
    img[0, y, x, 0] = value
    got = net.forward(img)
    np.testing.assert_array_equal(got, _per_layer(C, net, img))
    near = np.zeros((60, 70), bool)
    near[max(y - depth, 0):y + depth + 1, max(x - depth, 0):x + depth + 1] = True
    np.testing.assert_array_equal(got[0][~near], want[0][~near])
    assert (got[0, y, x] != want[0, y, x]).any()
    if np.isnan(value):
        assert np.isfinite(got).all()

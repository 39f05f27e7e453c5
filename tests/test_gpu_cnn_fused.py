"""Inference in one launch (a wave per layer, rows handed on through LDS) at
the edges of its strips (32 - 2 (depth - 1) output columns) and row chunks,
from the shallowest to the deepest network that takes it, and in several
rounds of workgroups.

The products are added in the order of the per-layer kernels, so the outputs
are compared bit for bit with theirs: a call whose output array covers its
input takes the per-layer kernels.  Against the oracle that rounds to bf16 at
the same points, rel. L2 2e-3 as in the other network tests.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _per_layer(ws, C, net, x):
    n, h, w, _ = x.shape
    px = n * h * w
    buf = C.DeviceArray.from_numpy(np.concatenate([x.reshape(-1), np.zeros(4 * px, np.float32)]))
    vx = C.DeviceArray.wrap(C.PDT_F32, [2 * px], buf.device_ptr(), owner=buf)
    C.check(C.lib().pdt_cnn_forward(net._h, vx.h, buf.h, n, h, w))
    return buf.numpy().reshape(n, h, w, 6)


@pytest.mark.parametrize("depth,shapes", [
    (2, [(1, 1, 1), (2, 7, 30), (1, 9, 31), (3, 64, 61)]),
    (3, [(1, 5, 28), (2, 8, 29)]),
    (5, [(1, 1, 23), (1, 2, 24), (2, 3, 25), (1, 100, 48), (1, 37, 49), (3, 111, 73), (2, 320, 97)]),
    (6, [(1, 40, 22), (1, 3, 45)]),
    (8, [(1, 4, 18), (1, 50, 19), (2, 33, 37), (1, 1, 200)]),
    (9, [(1, 12, 20)]),  # one more than the launch takes
])
def test_one_launch_equals_per_layer_launches(oracle, depth, shapes):
    from primaldualtoolbox import _capi as C
    from primaldualtoolbox import warmstart as ws
    net = ws.WarmStartCNN(depth=depth, seed=6)
    rng = np.random.default_rng(depth)
    p = net.get_params()
    o = 0
    for a, b in zip(net.channels[:-1], net.channels[1:]):  # biases: outside the image must stay zero
        o += 9 * a * b
        p[o:o + b] = 0.3 * rng.standard_normal(b)
        o += b
    net.set_params(p)
    for n, h, w in shapes:
        print(f"cnn depth {depth} n={n} h={h} w={w}", flush=True)
        x = rng.standard_normal((n, h, w, 2)).astype(np.float32)
        y = net.forward(x)
        np.testing.assert_array_equal(y, _per_layer(ws, C, net, x))
        assert rel_l2(y, oracle.cnn_forward(net.channels, p.astype(np.float64), x, bf16=True)) < 2e-3


def test_one_launch_in_rounds():
    """More strips than stay resident, images that end inside a chunk."""
    from primaldualtoolbox import _capi as C
    from primaldualtoolbox import warmstart as ws
    net = ws.WarmStartCNN(depth=5, seed=8)
    x = np.random.default_rng(1).standard_normal((9, 331, 805, 2)).astype(np.float32)
    np.testing.assert_array_equal(net.forward(x), _per_layer(ws, C, net, x))


def test_non_finite_pixels_stay_local():
    """A NaN and an infinity reach the outputs whose receptive field (depth
    pixels each way) holds them, and no others."""
    from primaldualtoolbox import warmstart as ws
    net = ws.WarmStartCNN(depth=5, seed=9)
    x = np.random.default_rng(2).standard_normal((1, 60, 70, 2)).astype(np.float32)
    want = net.forward(x)
    x[0, 30, 23, 0], x[0, 30, 24, 1] = np.nan, np.inf
    got = net.forward(x)
    far = np.ones((60, 70), bool)
    far[25:36, 18:30] = False
    np.testing.assert_array_equal(got[0][far], want[0][far])

"""The network kernels where their tiling can go wrong: widths around the 16-
and 32-pixel strips, images of one to a few rows, shares of rows that cross
strips and images, arrays at 4-byte alignment, and networks deeper than one
launch's layer table.

Tolerances as for the other network tests: outputs within rel. L2 2e-3 and
gradients within 2e-2 per layer of the oracle that rounds to bf16 at the same
points (a bf16 rounding flips now and then between fp32 and fp64 sums).
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 2, 15), (2, 1, 17), (1, 3, 16), (3, 3, 50), (1, 4, 31), (2, 5, 33), (1, 37, 32), (1, 70, 18)]


def _data(n, h, w, seed=0):
    rng = np.random.default_rng(seed + 1000 * n + 31 * h + w)
    return (rng.standard_normal((n, h, w, 2)).astype(np.float32),
            (0.3 * rng.standard_normal((n, h, w, 6))).astype(np.float32))


@pytest.mark.parametrize("n,h,w", SHAPES)
def test_forward_and_gradient_tiles(oracle, n, h, w):
    from primaldualtoolbox import warmstart as ws
    net = ws.WarmStartCNN(seed=3)
    p, ch = net.get_params().astype(np.float64), net.channels
    x, t = _data(n, h, w)
    print(f"cnn tiles n={n} h={h} w={w}", flush=True)
    assert rel_l2(net.forward(x), oracle.cnn_forward(ch, p, x, bf16=True)) < 2e-3
    loss, g = net.loss_grad(x, t)
    ref_loss, ref = oracle.cnn_loss_grad(ch, p, x, t, bf16=True)
    assert abs(loss - ref_loss) <= 1e-3 * ref_loss
    o = 0
    for a, b in zip(ch[:-1], ch[1:]):
        nw = 9 * a * b
        assert rel_l2(g[o:o + nw], ref[o:o + nw]) < 2e-2
        assert rel_l2(g[o + nw:o + nw + b], ref[o + nw:o + nw + b]) < 2e-2
        o += nw + b


def test_arrays_at_four_byte_alignment():
    from primaldualtoolbox import _capi as C
    from primaldualtoolbox import warmstart as ws
    net = ws.WarmStartCNN(seed=4)
    n, h, w = 1, 9, 21
    x, _ = _data(n, h, w)
    want = net.forward(x)
    px = n * h * w
    dx = C.DeviceArray.from_numpy(np.concatenate([np.zeros(1, np.float32), x.reshape(-1)]))
    dy = C.DeviceArray.from_numpy(np.zeros(6 * px + 1, np.float32))
    vx = C.DeviceArray.wrap(C.PDT_F32, [2 * px], dx.device_ptr() + 4, owner=dx)
    vy = C.DeviceArray.wrap(C.PDT_F32, [6 * px], dy.device_ptr() + 4, owner=dy)
    C.check(C.lib().pdt_cnn_forward(net._h, vx.h, vy.h, n, h, w))
    got = dy.numpy()
    assert got[0] == 0
    np.testing.assert_array_equal(got[1:].reshape(n, h, w, 6), want)


@pytest.mark.parametrize("depth", [2, 10])
def test_depths(oracle, depth):
    """Two layers (no hidden one) and more than the eight of a layer table."""
    from primaldualtoolbox import warmstart as ws
    net = ws.WarmStartCNN(depth=depth, seed=5)
    p, ch = net.get_params().astype(np.float64), net.channels
    x, t = _data(1, 6, 20)
    assert rel_l2(net.forward(x), oracle.cnn_forward(ch, p, x, bf16=True)) < 2e-3
    _, g = net.loss_grad(x, t)
    _, ref = oracle.cnn_loss_grad(ch, p, x, t, bf16=True)
    assert rel_l2(g, ref) < 2e-2
    before = net.get_params()
    net.adam_step(lr=1e-3)
    assert not np.array_equal(before, net.get_params())
    after = net.get_params().astype(np.float64)
    assert rel_l2(net.forward(x), oracle.cnn_forward(ch, after, x, bf16=True)) < 2e-3

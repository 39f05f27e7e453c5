"""Blocked denoising launches (tiles in registers) where their tiling can go
wrong, against the one-iteration kernels, bit for bit: images narrower than a
wave or lower than a wave's rows, one row or column, sizes around the regions'
edges, halos up to the widest, the default tile, iteration counts that are not
a multiple of a launch's, and images with NaN and infinite pixels at the
borders."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _image(shape, dtype, seed=0):
    rng = np.random.default_rng(seed + 1000 * shape[0] + shape[1])
    f = rng.standard_normal(shape)
    if np.dtype(dtype).kind == "c":
        f = f + 1j * rng.standard_normal(shape)
    return f.astype(dtype)


def _solve(solver, f, tile, iters, fp16=False):
    """tile: (x, y, iterations), None for the one-iteration kernels."""
    import primaldualtoolbox as pdt
    cls = {"tv": pdt.denoising.TvOptimizer_2f, "tgv": pdt.denoising.TgvOptimizer_2f}[solver]
    opt = cls(dtype=f.dtype)
    opt.setNoisyData(f)
    p = opt.getParameters()
    p.Lambda, p.max_iter = 9.0, iters - 1
    if solver == "tgv":
        p.alpha0, p.alpha1, p.dual_fp16 = 0.5, 0.3, int(fp16)
    pdt.denoising.set_tiles([opt], rpi=1, tv_block=tile, dual_px=1)
    opt.solve()
    assert opt.getStats()["iters"] == iters
    return [opt.getResult().copy()] + ([opt.getV().copy()] if solver == "tgv" else [])


def _check(solver, f, tile, iters, fp16=False):
    for a, b in zip(_solve(solver, f, None, iters, fp16), _solve(solver, f, tile, iters, fp16)):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("solver", ["tv", "tgv"])
@pytest.mark.parametrize("shape", [(1, 1), (1, 70), (70, 1), (2, 2), (3, 64), (4, 65), (5, 63), (33, 66), (64, 128),
                                   (65, 129)])
def test_sizes(solver, shape):
    for tile in ((52, 4, 6), (56, 24, 4)):
        _check(solver, _image(shape, np.float32), tile, 25)


@pytest.mark.parametrize("solver", ["tv", "tgv"])
@pytest.mark.parametrize("dtype", [np.float32, np.complex64, np.float64, np.complex128])
@pytest.mark.parametrize("tile", [(62, 2, 1), (24, 24, 20), (1, 1, 15), (200, 200, 7), (3, 100, 13)])
def test_halos(solver, dtype, tile):
    for iters in (1, 2, 3, 41):
        _check(solver, _image((75, 131), dtype), tile, iters)


@pytest.mark.parametrize("fp16", [False, True])
def test_non_finite_pixels(fp16):
    f = _image((70, 100), np.float32)
    f[0, 0], f[69, 99], f[35, 99], f[69, 50], f[20, 0] = np.nan, np.inf, np.nan, -np.inf, np.inf
    _check("tgv", f, (52, 20, 6), 12, fp16)
    if not fp16:
        _check("tv", f, (40, 8, 12), 24)


@pytest.mark.parametrize("solver,dtype,shape", [("tv", np.float32, (61, 47)), ("tv", np.complex64, (300, 210)),
                                                ("tgv", np.float32, (150, 333)), ("tgv", np.complex128, (90, 81))])
def test_default_tile(solver, dtype, shape):
    """A fresh shape takes the blocked launches by default."""
    import primaldualtoolbox as pdt
    f = _image(shape, dtype)
    cls = {"tv": pdt.denoising.TvOptimizer_2f, "tgv": pdt.denoising.TgvOptimizer_2f}[solver]
    opt = cls(dtype=dtype)
    opt.setNoisyData(f)
    p = opt.getParameters()
    p.Lambda, p.max_iter = 9.0, 52
    if solver == "tgv":
        p.alpha0, p.alpha1 = 0.5, 0.3
    opt.solve()
    assert opt.profileKernels(1)[0]["name"] == {"tv": "k_tv_block", "tgv": "k_tgv_block"}[solver]
    got = opt.getResult().copy()
    np.testing.assert_array_equal(_solve(solver, f, None, 53)[0], got)

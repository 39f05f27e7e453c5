"""Projections of the dual steps in single precision where |b|^2 is subnormal
(|b| < 1.1e-19, with a radius below it), against the FP64 oracle: blocked and
one-iteration TGV denoising, and the MRI iterations in pairs and in three
passes.  The oracle's result with the projection is 90 % away from the one
without.

Tolerance 2e-3: at the radius, 1e-20, |b|^2 = 1e-40 is known to some three
steps of 2^-149, 2e-5 of the projection factor, over 30 iterations.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL, RADIUS = 2e-3, 1e-20


@pytest.mark.parametrize("dtype", [np.float32, np.complex64])
@pytest.mark.parametrize("tile", [None, (52, 20, 6)])
def test_denoising_at_a_tiny_radius(oracle, dtype, tile):
    import primaldualtoolbox as pdt
    rng = np.random.default_rng(1)
    f = rng.standard_normal((40, 50))
    if dtype is np.complex64:
        f = f + 1j * rng.standard_normal((40, 50))
    f = (6e-20 * f).astype(dtype)
    opt = pdt.denoising.TgvOptimizer_2f(dtype=dtype)
    opt.setNoisyData(f)
    p = opt.getParameters()
    p.Lambda, p.alpha0, p.alpha1, p.max_iter = 5, 2 * RADIUS, RADIUS, 29
    pdt.denoising.set_tiles([opt], rpi=1, tv_block=tile)
    opt.solve()
    wide = np.complex128 if dtype is np.complex64 else np.float64
    want = oracle.solve(oracle.TGV, f.astype(wide), lambda_=5, alpha0=2 * RADIUS, alpha1=RADIUS, max_iter=29)[0]
    assert rel_l2(opt.getResult().astype(wide) * 1e20, want * 1e20) < TOL


@pytest.mark.parametrize("n,n_pe,coils", [(16, 256, 8), (32, 32, 4)])
def test_reconstruction_at_a_tiny_radius(oracle, n, n_pe, coils):
    import primaldualtoolbox as pdt
    from primaldualtoolbox import synthetic as syn
    case = syn.mri_case(seed=0, n=n, n_pe=n_pe, coils=coils, center=4)
    k = (1e-18 * case["kspace"]).astype(np.complex64)
    op = pdt.mri.MriCartesianRemoveROOSOperator()
    op.setCoilSens(case["sens"])
    op.setMask(case["mask"])
    o = pdt.mri.TgvMriOptimizer_2c3c()
    o.setOperator(op)
    o.setNoisyData(k)
    p = o.getParameters()
    p.alpha0, p.alpha1, p.max_iter = 2 * RADIUS, RADIUS, 29
    o.solve()
    oop = oracle.Op(oracle.OP_CARTESIAN_ROOS, case["sens"].astype(np.complex128), case["mask"].astype(np.float64))
    prm = dict(op=oop, max_iter=29)
    want = oracle.solve(oracle.TGV_MRI, k.astype(np.complex128), alpha0=2 * RADIUS, alpha1=RADIUS, **prm)[0]
    free = oracle.solve(oracle.TGV_MRI, k.astype(np.complex128), alpha0=1.0, alpha1=1.0, **prm)[0]
    assert rel_l2(free * 1e20, want * 1e20) > 10 * TOL
    assert rel_l2(o.getResult().astype(np.complex128) * 1e20, want * 1e20) < TOL


@pytest.mark.parametrize("tile", [None, (52, 20, 6)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_negative_zero_projects_nothing(dtype, tile):
    """max(1, |b| / alpha) is 1 for every alpha below zero, -0.0 among them."""
    import primaldualtoolbox as pdt
    f = np.random.default_rng(2).standard_normal((40, 50)).astype(dtype)
    out = []
    for radius in (-0.0, -1.0):
        opt = pdt.denoising.TgvOptimizer_2f(dtype=dtype)
        opt.setNoisyData(f)
        p = opt.getParameters()
        p.Lambda, p.alpha0, p.alpha1, p.max_iter = 5, radius, radius, 9
        pdt.denoising.set_tiles([opt], rpi=1, tv_block=tile)
        opt.solve()
        out.append(opt.getResult().copy())
    np.testing.assert_array_equal(*out)

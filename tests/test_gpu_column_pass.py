"""The column pass of the lengths 8 M 8 (256 to 768 points): operators against
the FP64 oracle for every length, both precisions, full and cropped images,
and numbers of sampled columns and coils that leave the last group partial;
and solves whose iterates must not depend on the columns per group.

Tolerances as for the other operator tests: 2e-5 relative L2 in single
precision; 1e-13 in double (three stages of about 10 roundings of 1.1e-16 in
each direction, with a factor above 10 to spare).
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

LENGTHS = [256, 320, 384, 512, 640, 768]


def _mask(rng, Hk, W, nc):
    m = np.zeros(W)
    m[rng.permutation(W)[:nc]] = 1.0
    return np.repeat(m[None, :], Hk, axis=0) * (0.5 + rng.random((Hk, 1)))  # weights, not only 0 and 1


@pytest.mark.parametrize("dtype,tol", [(np.complex64, 2e-5), (np.complex128, 1e-13)])
@pytest.mark.parametrize("Hk", LENGTHS)
@pytest.mark.parametrize("roos", [False, True])
def test_operator_matches_oracle(oracle, dtype, tol, Hk, roos):
    import primaldualtoolbox as pdt
    rng = np.random.default_rng(Hk)
    W, C, nc = 22, 3, {256: 1, 320: 9, 384: 7, 512: 5, 640: 3, 768: 11}[Hk]
    S = (rng.standard_normal((C, Hk, W)) + 1j * rng.standard_normal((C, Hk, W))).astype(dtype)
    mask = _mask(rng, Hk, W, nc).astype(np.float64)
    kind = oracle.OP_CARTESIAN_ROOS if roos else oracle.OP_CARTESIAN
    cls = pdt.mri.MriCartesianRemoveROOSOperator if roos else pdt.mri.MriCartesianOperator
    oop = oracle.Op(kind, S.astype(np.complex128), mask)
    op = cls(dtype=dtype)
    op.setCoilSens(S)
    op.setMask(mask)
    y = (rng.standard_normal((C, Hk, W)) + 1j * rng.standard_normal((C, Hk, W))).astype(dtype)
    print(f"columns of {Hk} roos={roos} {np.dtype(dtype).name}", flush=True)
    u = op.adjoint(y)
    assert rel_l2(u, oop.adjoint(y.astype(np.complex128))) < tol
    assert rel_l2(op.forward(u), oop.forward(u.astype(np.complex128))) < tol


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("Hk", LENGTHS)
def test_iterates_do_not_depend_on_columns_per_group(dtype, Hk):
    import primaldualtoolbox as pdt
    rng = np.random.default_rng(Hk + 1)
    W, C, nc = 24, 2, 11
    S = (rng.standard_normal((C, Hk, W)) + 1j * rng.standard_normal((C, Hk, W))).astype(dtype) / 2
    mask = (_mask(rng, Hk, W, nc) > 0).astype(np.float64)
    f = ((rng.standard_normal((C, Hk, W)) + 1j * rng.standard_normal((C, Hk, W))) * mask).astype(dtype)
    res = []
    for cg in (0, 1, 2, 3, 5, 16):
        op = pdt.mri.MriCartesianRemoveROOSOperator(dtype=dtype)
        op.setCoilSens(S)
        op.setMask(mask)
        opt = pdt.mri.TgvMriOptimizer_2c3c(dtype=dtype)
        opt.setOperator(op)
        opt.setNoisyData(f)
        p = opt.getParameters()
        p.alpha0, p.alpha1, p.max_iter, p.gap_every = 0.02, 0.01, 24, 10
        pdt.denoising.set_tiles([opt], cg=cg)
        opt.solve()
        res.append((opt.getResult().copy(), opt.getStats()["rel_gap"]))
    for u, gap in res[1:]:
        np.testing.assert_array_equal(u, res[0][0])
        # the gap's FP64 partial sums are grouped by column item
        assert abs(gap - res[0][1]) <= 1e-12 * abs(res[0][1])

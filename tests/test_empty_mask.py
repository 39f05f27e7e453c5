"""Masks without a sampled line: A and A^* are zero, so a solve only smooths
its start.  The adjoint row pass that holds every coil of a row reads its
sampled entries branch-free and must not be chosen for such a slice (host rule,
CPU); solves through every other route against the FP64 oracle (GPU).

Tolerance 2e-5 relative L2: 20 iterations of some 20 single precision steps
(6e-8 each) on values of one magnitude.
"""
import ctypes as ct

import numpy as np
import pytest

from conftest import rel_l2

TOL = 2e-5


@pytest.mark.parametrize("W", [256, 320, 368, 384, 512])
def test_no_straight_line_rows_without_listed_columns(W):
    from primaldualtoolbox import _capi as C
    ok = C.lib()._ZN3pdt17rows_adj_fused_okEiiii  # pdt::rows_adj_fused_ok(dtype, W, C, nc)
    ok.restype, ok.argtypes = ct.c_bool, [ct.c_int] * 4
    coils = 10
    assert ok(C.PDT_C64, W, coils, 1) and ok(C.PDT_C64, W, coils, 64)
    for c in range(1, 21):
        assert not ok(C.PDT_C64, W, c, 0)


def _case(n, n_pe, coils):
    from primaldualtoolbox import synthetic as syn
    case = syn.mri_case(seed=5, n=n, n_pe=n_pe, coils=coils, center=4)
    case["mask"] = np.zeros_like(case["mask"])
    return case


def _solver(case, dtype, u0, tv=False):
    import primaldualtoolbox as pdt
    op = pdt.mri.MriCartesianRemoveROOSOperator(dtype=dtype)
    op.setCoilSens(case["sens"])
    op.setMask(case["mask"])
    o = (pdt.mri.TvOptimizerWithOp_2c3c if tv else pdt.mri.TgvMriOptimizer_2c3c)(dtype=dtype)
    o.setOperator(op)
    o.setNoisyData(case["kspace"])
    o.setInput0(u0)
    p = o.getParameters()
    p.max_iter, p.gap_every = 19, 7
    if not tv:
        p.alpha1, p.alpha0 = 0.05, 0.1
    return o


def _want(oracle, case, u0, tv=False):
    op = oracle.Op(oracle.OP_CARTESIAN_ROOS, case["sens"].astype(np.complex128), case["mask"].astype(np.float64))
    prm = {} if tv else dict(alpha1=0.05, alpha0=0.1)
    return oracle.solve(oracle.TV_OP if tv else oracle.TGV_MRI, case["kspace"].astype(np.complex128), op=op, u0=u0,
                        max_iter=19, **prm)[0]


def _start(n, n_pe):
    rng = np.random.default_rng(n_pe)
    return (rng.standard_normal((n, n_pe)) + 1j * rng.standard_normal((n, n_pe))).astype(np.complex64)


@pytest.mark.gpu
@pytest.mark.parametrize("tiles", [None, "all coils", "all coils, three passes"])
@pytest.mark.parametrize("n_pe,coils", [(256, 2), (256, 15), (320, 2), (320, 15), (512, 10), (96, 3)])
def test_solve_with_an_empty_mask_matches_oracle(oracle, n_pe, coils, tiles):
    import primaldualtoolbox as pdt
    n, tv = 24, coils == 10
    case, u0 = _case(n, n_pe, coils), _start(n, n_pe)
    o = _solver(case, np.complex64, u0, tv)
    print(f"empty mask, PE {n_pe}, {coils} coils, {tiles}", flush=True)
    if tiles:
        pdt.mri.set_tiles([o], cb=4, cg=1, cb_a=coils, unpaired=int("three" in tiles))
    try:
        o.solve()
    finally:
        if tiles:
            pdt.mri.set_tiles([o])
    assert o.getStats()["iters"] == 20
    assert rel_l2(o.getResult(), _want(oracle, case, u0, tv)) < TOL


@pytest.mark.gpu
def test_double_precision_and_a_batch_with_an_empty_mask(oracle):
    import primaldualtoolbox as pdt
    case, u0 = _case(24, 256, 4), _start(24, 256)
    o = _solver(case, np.complex128, u0)
    o.solve()
    assert rel_l2(o.getResult(), _want(oracle, case, u0)) < 1e-12
    batch = [_solver(_case(24, w, 3), np.complex64, _start(24, w)) for w in (256, 40)]
    pdt.mri.set_tiles(batch, cb=3, cg=1, cb_a=3)  # work lists over the batch
    pdt.mri.batch_solve(batch)
    for w, b in zip((256, 40), batch):
        assert rel_l2(b.getResult(), _want(oracle, _case(24, w, 3), _start(24, w))) < TOL


@pytest.mark.gpu
def test_operator_with_an_empty_mask_is_zero():
    case = _case(24, 256, 3)
    op = _solver(case, np.complex64, _start(24, 256))._op
    assert not np.any(op.forward(_start(24, 256)))
    assert not np.any(op.adjoint(case["kspace"]))

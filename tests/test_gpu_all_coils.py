"""Which single slices hold every coil of a row in one adjoint workgroup by
default, and that the iterates stay those of the other groupings: bit for bit
on planned rows (two launches per iteration against three passes, from one
coil on), within the rounding of a reordered coil sum on rows with a runtime
plan (256 and 1024 threads, on both sides of the LDS and size limits, single
and double precision; 2e-5 relative L2, 1e-12 in double, after 31 iterations
that do not amplify it)."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_more import _mri_solver, _pdt

pytestmark = pytest.mark.gpu


def _solve(pdt, case, coils, dtype, kind, **tiles):
    a1 = 1e-5 * float(np.linalg.norm(case["kspace"]))
    case = dict(case, sens=case["sens"].astype(dtype), kspace=case["kspace"].astype(dtype))
    cls = pdt.mri.TvOptimizerWithOp_2c3c if kind == "tvop" else pdt.mri.TgvMriOptimizer_2c3c
    prm = dict(gap_every=10, gap_tol=0.0)
    if kind == "tvop":
        prm["Lambda"] = 0.5
    _, opt = _mri_solver(pdt, case, cls=cls, dtype=dtype, a1=None if kind == "tvop" else a1, max_iter=30, **prm)
    try:
        if tiles:
            pdt.mri.set_tiles([opt], **tiles)
        names = [k["name"] for k in opt.profileKernels(2)]
        opt.solve()
    finally:
        pdt.mri.set_tiles([opt])
    return names, opt.getResult().copy(), opt.getStats()["rel_gap"]


@pytest.mark.parametrize("kind", ["tgvmri", "tvop"])
@pytest.mark.parametrize("coils,n,n_pe", [(1, 30, 256), (2, 48, 256), (7, 32, 256), (1, 40, 320), (3, 40, 320),
                                          (2, 30, 384), (1, 96, 512)])
def test_planned_rows_equal_three_passes(kind, coils, n, n_pe):
    pdt = _pdt()
    from primaldualtoolbox import synthetic as syn
    case = syn.mri_case(seed=51, n=n, n_pe=n_pe, coils=coils)
    n2, u2, g2 = _solve(pdt, case, coils, np.complex64, kind)
    n3, u3, g3 = _solve(pdt, case, coils, np.complex64, kind, cb_a=coils, unpaired=1)
    print(f"  {kind} {coils} coils, rows of {n_pe}: {n2} / {n3}", flush=True)
    assert n2 == ["k_cols_dual", "k_rows_adj_next"]
    assert n3 == ["k_rows_fwd", "k_cols", "k_rows_adj"]
    assert np.array_equal(u2, u3) and g2 == g3


@pytest.mark.parametrize("dtype,tol", [(np.complex64, 2e-5), (np.complex128, 1e-12)])
@pytest.mark.parametrize("coils,n,n_pe", [(1, 20, 60), (3, 24, 66), (7, 30, 147), (8, 30, 128), (9, 26, 230),
                                          (25, 20, 200), (50, 16, 200)])
def test_runtime_rows_equal_coil_groups(dtype, tol, coils, n, n_pe):
    pdt = _pdt()
    from primaldualtoolbox import synthetic as syn
    case = syn.mri_case(seed=53, n=n, n_pe=n_pe, coils=coils)
    names, u, gap = _solve(pdt, case, coils, dtype, "tgvmri")
    print(f"  {coils} coils, rows of {n_pe}, {np.dtype(dtype).name}: {names}", flush=True)
    for tiles in (dict(cb=4, cb_a=min(4, coils)), dict(cb=1, cb_a=1), dict(cb=3, cb_a=coils)):
        _, v, g = _solve(pdt, case, coils, dtype, "tgvmri", **tiles)
        assert rel_l2(u, v) < tol
        assert abs(gap - g) <= 1e-3 * abs(g)

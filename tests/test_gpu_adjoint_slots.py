"""The adjoint row pass with every coil of a row in one workgroup, on rows of
384 and 512 (two groups of threads): 10 coils are the most that the kernel
with five sensitivity slots per thread takes, 11 to 16 go to the one with
eight, 17 to the general passes.  The two-launch iterations against the three
passes per iteration, bit for bit, gaps included."""
import numpy as np
import pytest

from test_gpu_more import _mri_solver, _pdt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coils,n,n_pe,paired", [(10, 48, 384, True), (11, 48, 384, True), (15, 384, 384, True),
                                                 (16, 48, 384, True), (17, 48, 384, False), (11, 40, 512, True),
                                                 (16, 40, 512, True), (17, 40, 512, False)])
def test_two_thread_groups_equal_three_passes(coils, n, n_pe, paired):
    pdt = _pdt()
    from primaldualtoolbox import synthetic as syn
    case = syn.mri_case(seed=41, n=n, n_pe=n_pe, coils=coils)
    a1 = 1e-5 * float(np.linalg.norm(case["kspace"]))
    prm = dict(gap_every=10, use_graph=1, gap_tol=0.0)
    _, two = _mri_solver(pdt, case, a1=a1, max_iter=30, **prm)
    _, three = _mri_solver(pdt, case, a1=a1, max_iter=30, **prm)
    try:
        names = [k["name"] for k in two.profileKernels(2)]
        two.solve()
        pdt.mri.set_tiles([three], cb_a=coils, unpaired=1)
        three.solve()
    finally:
        pdt.mri.set_tiles([two])
    print(f"  {coils} coils, rows of {n_pe}: {names}", flush=True)
    assert (names == ["k_cols_dual", "k_rows_adj_next"]) == paired
    s2, s3 = two.getStats(), three.getStats()
    assert s2["iters"] == s3["iters"] == 31
    if paired:
        assert s2["rel_gap"] == s3["rel_gap"]
        assert np.array_equal(two.getResult(), three.getResult())
        assert np.array_equal(two.getV(), three.getV())
    else:  # sums over the coils in other groups
        from conftest import rel_l2
        assert rel_l2(two.getResult(), three.getResult()) < 2e-5

"""The two ways a batch of operator solvers is run (concurrent single solves,
or work-list launches over the batch) give the same iterates, stops and
statistics (bit for bit those of single solves on the first way): mixed and equal sizes, few and many slices, single and double
precision, stops at the gap; tuned or set tiles and direct launches keep the
work-list launches."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL_ORDER = 2e-5


def _solvers(shapes, dtype=np.complex64, max_iter=120, gap_tol=0.0, graph=1):
    import primaldualtoolbox as pdt
    from primaldualtoolbox import synthetic as syn
    out = []
    for k, (n, n_pe, coils) in enumerate(shapes):
        case = syn.mri_case(seed=70 + k, n=n, n_pe=n_pe, coils=coils, center=8)
        op = pdt.mri.MriCartesianRemoveROOSOperator(dtype=dtype)
        op.setCoilSens(case["sens"])
        op.setMask(case["mask"])
        o = pdt.mri.TgvMriOptimizer_2c3c(dtype=dtype)
        o.setOperator(op)
        o.setNoisyData(case["kspace"])
        p = o.getParameters()
        a1 = 1e-5 * float(np.linalg.norm(case["kspace"]))
        p.alpha1, p.alpha0, p.max_iter, p.gap_every, p.gap_tol = a1, 2 * a1, max_iter - 1, 40, gap_tol
        p.use_graph = graph
        out.append(o)
    return out


@pytest.mark.parametrize("shapes,dtype", [
    ([(64, 64, 4), (48, 80, 6)], np.complex64),                                   # two groups of one
    ([(32, 32, 2)] * 9 + [(40, 32, 3)], np.complex64),                            # many small slices
    ([(128, 256, 8), (128, 256, 5), (96, 320, 9), (64, 368, 4)], np.complex64),   # paired and three-pass singles
    ([(64, 64, 4), (64, 96, 3), (80, 64, 5)], np.complex128),
])
def test_routes_agree(shapes, dtype):
    import primaldualtoolbox as pdt
    many = len(shapes) > 8
    auto, lists, alone = (_solvers(shapes, dtype, gap_tol=4e-3, graph=g) for g in (1, 0, 1))
    pdt.mri.batch_solve(auto)
    pdt.mri.batch_solve(lists)  # direct launches: the work lists
    for o in alone:
        o.solve()
    for a, b, c in zip(auto, lists, alone):
        if not many:  # (many small slices take the work lists)
            np.testing.assert_array_equal(a.getResult(), c.getResult())
        # the work lists add the coils of a row in groups of four, a wide single
        # slice in one group: FP32 sums in another order (6e-8 each, TOL for 120
        # iterations as for one operator application)
        assert rel_l2(b.getResult(), c.getResult()) < TOL_ORDER
        sa, sb, sc = a.getStats(), b.getStats(), c.getStats()
        assert sa["iters"] == sb["iters"] == sc["iters"] and sa["converged"] == sc["converged"]
        assert abs(sb["rel_gap"] - sc["rel_gap"]) <= 1e-3 * abs(sc["rel_gap"])
        assert abs(sa["rel_gap"] - sc["rel_gap"]) <= 1e-3 * abs(sc["rel_gap"])
        assert sa["ms_to_stop"] > 0 and sa["ms"] > 0  # (host and device clocks: not compared)
    # a second batch on the same solvers continues from their state
    pdt.mri.batch_solve(auto)
    for o in alone:
        o.solve()
    for a, c in zip(auto, alone):
        assert rel_l2(a.getResult(), c.getResult()) < TOL_ORDER
        if not many:
            np.testing.assert_array_equal(a.getResult(), c.getResult())


def test_set_tiles_keep_the_work_lists():
    """Tiles set for a batch are those of its launches (and of no other batch)."""
    import primaldualtoolbox as pdt
    shapes = [(72, 72, 5), (72, 88, 4), (56, 72, 6)]
    a, b = _solvers(shapes, max_iter=50), _solvers(shapes, max_iter=50)
    pdt.mri.set_tiles(a, cb=2, cg=1, cb_a=3)
    pdt.mri.batch_solve(a)
    assert len({o.getStats()["ms_to_stop"] for o in a}) == 1  # one loop over the whole batch
    for o in b:
        o.solve()
    for x, y in zip(a, b):
        assert rel_l2(x.getResult(), y.getResult()) < TOL_ORDER


def test_a_failing_member_stops_the_batch_before_any_solve():
    import primaldualtoolbox as pdt
    from primaldualtoolbox import _capi as C
    good = _solvers([(64, 64, 4), (48, 64, 3)])
    bad = pdt.mri.TgvMriOptimizer_2c3c()
    bad.getParameters().gap_every = 40
    with pytest.raises(C.PdtError):
        pdt.mri.batch_solve(good + [bad])
    assert good[0].getStats()["iters"] == 0

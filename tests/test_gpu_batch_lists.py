"""Batches on the work lists (one set of launches over all slices), with
graphs: slices that stop at different iterations leave the lists, which are
compacted and captured again; mixed lengths with and without a compile-time
plan.  Every slice's result equals that of its own solve bit for bit, its gap
to 1e-12 (a single solve sums the dual step's FP64 gap terms over other
workgroups).

That a batch took the lists shows in two slices of equal iteration limit: they
leave in the same chunk of the one loop, so their times to stop are one number.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(n, n_pe, coils, seed, max_iter, tol):
    import primaldualtoolbox as pdt
    from primaldualtoolbox import synthetic as syn
    case = syn.mri_case(seed=seed, n=n, n_pe=n_pe, coils=coils, center=4)
    op = pdt.mri.MriCartesianRemoveROOSOperator()
    op.setCoilSens(case["sens"])
    op.setMask(case["mask"])
    o = pdt.mri.TgvMriOptimizer_2c3c()
    o.setOperator(op)
    o.setNoisyData(case["kspace"])
    p = o.getParameters()
    a1 = 1e-3 * float(np.linalg.norm(case["kspace"]))
    p.alpha1, p.alpha0, p.max_iter, p.gap_every, p.gap_tol = a1, 2 * a1, max_iter, 25, tol
    return o


def _check(specs, tiles):
    import primaldualtoolbox as pdt
    alone, batch = ([_solver(*s) for s in specs] for _ in range(2))
    if tiles:
        pdt.mri.set_tiles(batch, **tiles)
        for o in alone:
            pdt.mri.set_tiles([o], **tiles)
    try:
        for o in alone:
            o.solve()
        pdt.mri.batch_solve(batch)
    finally:
        if tiles:
            for o in alone:
                pdt.mri.set_tiles([o])
    stats = [o.getStats() for o in batch]
    assert stats[0]["ms_to_stop"] == stats[1]["ms_to_stop"]  # the twins: one loop
    for a, b, sb in zip(alone, batch, stats):
        sa = a.getStats()
        print(f"  iterations alone {sa['iters']} batch {sb['iters']}", flush=True)
        assert sa["iters"] == sb["iters"] and sa["converged"] == sb["converged"]
        assert abs(sa["rel_gap"] - sb["rel_gap"]) <= 1e-12 * abs(sb["rel_gap"])
        np.testing.assert_array_equal(a.getResult(), b.getResult())
        np.testing.assert_array_equal(a.getV(), b.getV())
    return stats


TILES = dict(cb=4, cg=2, cb_a=4)


def test_ragged_stops_with_set_tiles():
    stats = _check([(36, 36, 3, 1, 49, 0.0), (36, 28, 2, 2, 49, 0.0), (28, 28, 2, 3, 299, 0.0), (36, 36, 4, 4, 999, 1e-2),
                    (20, 28, 2, 5, 149, 0.0), (36, 36, 3, 6, 999, 3e-3), (28, 28, 2, 7, 99, 0.0)], TILES)
    iters = [s["iters"] for s in stats]
    # two of seven leave at 50, the next at 100 and 150: each time more than a
    # sixth of the items that are left, so the lists are compacted
    assert iters[0] == iters[1] == 50 and iters[6] == 100 and iters[4] == 150 and iters[2] == 300
    assert stats[3]["converged"] and stats[5]["converged"] and len(set(iters)) >= 5
    order = sorted(range(7), key=lambda i: iters[i])
    times = [stats[i]["ms_to_stop"] for i in order]
    assert times == sorted(times)


def test_mixed_compiled_and_runtime_lengths():
    _check([(256, 256, 2, 7, 29, 0.0), (48, 44, 3, 8, 29, 0.0), (256, 256, 3, 9, 29, 0.0), (48, 320, 3, 9, 39, 0.0)], TILES)


def test_many_small_slices_by_default():
    """Twelve slices of two sizes: the lists without any tiles set."""
    stats = _check([(30, 30, 2 + i % 3, 20 + i, 49 if i < 2 else 29 + 20 * i, 0.0) if i % 2 else
                    (26, 34, 2 + i % 3, 20 + i, 49 if i < 2 else 29 + 20 * i, 0.0) for i in range(12)], None)
    assert len({s["iters"] for s in stats}) == 11

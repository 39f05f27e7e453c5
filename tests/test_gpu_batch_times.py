"""Times that a batch run as concurrent single solves reports: ms is device
time of the iteration loop, from the start of the first slice's to the end of
the last one's; ms_to_stop counts on the host from the same start to the chunk
in which a slice stopped."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solvers(shapes, max_iter):
    import primaldualtoolbox as pdt
    from primaldualtoolbox import synthetic as syn
    out = []
    for k, (n, n_pe, coils) in enumerate(shapes):
        case = syn.mri_case(seed=20 + k, n=n, n_pe=n_pe, coils=coils, center=8)
        op = pdt.mri.MriCartesianRemoveROOSOperator()
        op.setCoilSens(case["sens"])
        op.setMask(case["mask"])
        o = pdt.mri.TgvMriOptimizer_2c3c()
        o.setOperator(op)
        o.setNoisyData(case["kspace"])
        p = o.getParameters()
        a1 = 1e-5 * float(np.linalg.norm(case["kspace"]))
        p.alpha1, p.alpha0, p.max_iter = a1, 2 * a1, max_iter - 1
        out.append(o)
    return out


def test_ms_is_device_time():
    """HIP events give single precision milliseconds, a host clock does not."""
    import primaldualtoolbox as pdt
    opts = _solvers([(64, 64, 6), (48, 80, 6), (64, 96, 4)], 60)
    for _ in range(3):
        t0 = time.perf_counter()
        pdt.mri.batch_solve(opts)
        wall = 1e3 * (time.perf_counter() - t0)
        ms = {o.getStats()["ms"] for o in opts}
        assert len(ms) == 1
        ms = ms.pop()
        assert 0 < ms < wall and ms == float(np.float32(ms))


def test_time_to_stop_counts_from_the_loops_start():
    """A slice that stops after 20 of 20 iterations beside one that takes 2000."""
    import primaldualtoolbox as pdt
    opts = _solvers([(64, 64, 6), (128, 128, 8)], 2000)
    opts[0].getParameters().max_iter = 19
    for _ in range(2):
        t0 = time.perf_counter()
        pdt.mri.batch_solve(opts)
        wall = 1e3 * (time.perf_counter() - t0)
        short, long = (o.getStats() for o in opts)
        assert short["iters"] == 20 and long["iters"] == 2000
        assert 0 < short["ms_to_stop"] < 0.5 * long["ms_to_stop"]
        assert long["ms_to_stop"] < wall and long["ms"] < wall

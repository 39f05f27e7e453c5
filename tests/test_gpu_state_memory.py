"""Device memory of a denoising solver: the data, the state (ROF: u, ubar and
two planes of p; TGV: u, ubar, v and vbar of two planes each, p of two and q of
three, and two planes of scratch) and a second copy of what the blocked
launches hand on (ROF: u, ubar, p; TGV: u, v, p, q), and no more."""
import ctypes as ct
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 2048  # planes of 32 MB in complex64: far above the granule of allocations


def _free():
    from primaldualtoolbox import _capi as C
    hip = C.lib()  # (its own HIP runtime)
    free, total = ct.c_size_t(), ct.c_size_t()
    assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(ct.byref(free), ct.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("solver,planes", [("tv", 1 + 4 + 4), ("tgv", 1 + 11 + 2 + 8)])
def test_planes_of_a_solver(solver, planes):
    import primaldualtoolbox as pdt
    from primaldualtoolbox import _capi as C
    warm = pdt.denoising.TgvOptimizer_2f(dtype=np.complex64)  # the runtime's own memory: code, queues
    warm.setNoisyData(np.ones((64, 64), np.complex64))
    warm.solve()
    data = C.DeviceArray.from_numpy(np.ones((N, N), np.complex64))
    opt = {"tv": pdt.denoising.TvOptimizer_2f, "tgv": pdt.denoising.TgvOptimizer_2f}[solver](dtype=np.complex64)
    gc.collect()
    free = _free()
    C.check(C.lib().pdt_solver_set_noisy_data(opt._h, data.h))
    C.check(C.lib().pdt_solver_set_input0(opt._h, data.h, None))
    used = free - _free()
    print(f"{solver}: {used / (8 * N * N):.2f} planes", flush=True)
    assert used <= (planes + 0.5) * 8 * N * N
    opt.getParameters().max_iter = 20
    opt.solve()
    assert np.isfinite(opt.getResult()).all()

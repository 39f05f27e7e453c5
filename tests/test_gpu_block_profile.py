"""What the profile reports of a blocked denoising launch: the planes that the
kernel reads and writes, each once (ROF: u, ubar, p and f in, u, ubar and p
out; TGV: u, v, p, q and f in, u, v, p and q out; p and q in their storage
type)."""
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver,dtype,fp16,per_pixel", [
    ("tv", np.float32, False, 9 * 4), ("tv", np.complex128, False, 9 * 16), ("tgv", np.float32, False, 17 * 4),
    ("tgv", np.complex64, False, 17 * 8), ("tgv", np.complex64, True, 7 * 8 + 10 * 4)])
def test_bytes_of_a_launch(solver, dtype, fp16, per_pixel):
    import primaldualtoolbox as pdt
    f = np.random.default_rng(0).standard_normal((90, 130)).astype(dtype)
    opt = {"tv": pdt.denoising.TvOptimizer_2f, "tgv": pdt.denoising.TgvOptimizer_2f}[solver](dtype=dtype)
    opt.setNoisyData(f)
    if fp16:
        opt.getParameters().dual_fp16 = True
        opt._push_params()
    opt.solve()
    (k,) = opt.profileKernels(1)
    assert k["bytes"] == per_pixel * f.size


@pytest.mark.parametrize("solver", ["tv", "tgv"])
def test_the_reported_name_is_that_of_a_kernel(solver):
    """(to be found in a kernel trace)"""
    import primaldualtoolbox as pdt
    from primaldualtoolbox import _capi as C
    opt = {"tv": pdt.denoising.TvOptimizer_2f, "tgv": pdt.denoising.TgvOptimizer_2f}[solver]()
    opt.setNoisyData(np.random.default_rng(0).standard_normal((90, 130)).astype(np.float32))
    opt.solve()
    (k,) = opt.profileKernels(1)
    names = subprocess.run(["nm", "-C", C.LIB_PATH], capture_output=True, text=True, check=True).stdout
    assert f"__device_stub__{k['name']}<float" in names

"""A forward application whose output overlaps its input: the output is zeroed
before the row transforms read the input, so what the output covers counts as
zero (an in-place application gives zero), in every repetition; arrays that
only touch are not affected.  Single precision against the FP64 oracle, 2e-5
relative L2; zeros exactly."""
import ctypes as ct

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("C,W,Hk", [(1, 256, 96), (3, 320, 64), (2, 48, 40)])
def test_forward_onto_its_input(oracle, C, W, Hk, noalloc):
    import primaldualtoolbox as pdt
    from primaldualtoolbox import _capi as capi
    lib = capi.lib()
    rng = np.random.default_rng(C)
    S = (rng.standard_normal((C, Hk, W)) + 1j * rng.standard_normal((C, Hk, W))).astype(np.complex64)
    mask = np.repeat((rng.random(W) < 0.5)[None, :], Hk, axis=0).astype(np.float32)
    op = pdt.mri.MriCartesianOperator()
    op.setCoilSens(S)
    op.setMask(mask)
    x = (rng.standard_normal((Hk, W)) + 1j * rng.standard_normal((Hk, W))).astype(np.complex64)
    want = oracle.Op(oracle.OP_CARTESIAN, S.astype(np.complex128), mask.astype(np.float64)).forward(x.astype(np.complex128))
    assert rel_l2(op.forward(x), want) < 2e-5  # prepares the operator
    px = W * Hk
    for at in (0, (C - 1) * px, C * px):  # x at this element of y's array; the last: behind y
        for _ in range(5):
            buf = capi.DeviceArray.from_numpy(np.concatenate([np.full(at, np.nan, np.complex64), x.reshape(-1),
                                                              np.full(C * px, np.nan, np.complex64)]))
            ptr = buf.device_ptr()
            vx = capi.DeviceArray.wrap(capi.PDT_C64, [W, Hk], ptr + 8 * at, owner=buf)
            vy = capi.DeviceArray.wrap(capi.PDT_C64, [W, Hk, C], ptr, owner=buf)
            if noalloc:
                capi.check(lib.pdt_op_apply_noalloc(op._h, 1, vx.h, vy.h, ct.c_void_p()))
            else:
                capi.check(lib.pdt_op_forward(op._h, vx.h, vy.h))
            y = buf.numpy().reshape(-1)[:C * px].reshape(C, Hk, W)
            if at < C * px:
                assert not y.any()
            else:
                assert rel_l2(y, want) < 2e-5

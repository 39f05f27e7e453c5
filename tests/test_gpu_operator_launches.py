"""One operator application: the output of A is zeroed beside the row
transforms (every element outside the listed columns, whatever it held), and
A^* of many coils in one workgroup per row (2048 or more coil pixels a row,
256-point and other planned rows) or in coil groups.  Against the FP64 oracle,
2e-5 relative L2 in single and 1e-13 in double precision as in the other
operator tests; the zeros exactly.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(np.complex64, 2e-5), (np.complex128, 1e-13)])
@pytest.mark.parametrize("W,Hk,C,nc", [(256, 6, 7, 5), (256, 6, 8, 64), (256, 10, 20, 100), (320, 8, 6, 320),
                                       (368, 5, 9, 40), (512, 7, 4, 1), (512, 64, 5, 90), (300, 9, 8, 30),
                                       (31, 259, 2, 3)])
def test_application_matches_oracle(oracle, dtype, tol, W, Hk, C, nc):
    import primaldualtoolbox as pdt
    from primaldualtoolbox import _capi as C_
    rng = np.random.default_rng(W + Hk + C)
    S = (rng.standard_normal((C, Hk, W)) + 1j * rng.standard_normal((C, Hk, W))).astype(dtype)
    line = np.zeros(W)
    line[rng.permutation(W)[:nc]] = 1.0
    mask = np.repeat(line[None, :], Hk, axis=0)
    oop = oracle.Op(oracle.OP_CARTESIAN, S.astype(np.complex128), mask)
    op = pdt.mri.MriCartesianOperator(dtype=dtype)
    op.setCoilSens(S)
    op.setMask(mask)
    x = (rng.standard_normal((Hk, W)) + 1j * rng.standard_normal((Hk, W))).astype(dtype)
    print(f"application W={W} Hk={Hk} C={C} nc={nc} {np.dtype(dtype).name}", flush=True)
    y = op.forward(x)  # prepares the operator
    ref = oop.forward(x.astype(np.complex128))
    assert rel_l2(y, ref) < tol
    dx = C_.DeviceArray.from_numpy(x)
    dy = C_.DeviceArray.from_numpy(np.full((C, Hk, W), np.nan, dtype))
    for _ in range(2):
        C_.check(C_.lib().pdt_op_forward(op._h, dx.h, dy.h))
        got = dy.numpy().reshape(C, Hk, W)
        assert not got[:, :, line == 0].any()
        np.testing.assert_array_equal(got, y.reshape(C, Hk, W))
    assert rel_l2(op.adjoint(y), oop.adjoint(ref)) < 2 * tol  # (of a rounded y)

"""Transform lengths of the row and column passes against the FP64 oracle:
prime factors without a register codelet (7 to 61, alone, repeated and mixed
with the codelet radices), in single and double precision.

Tolerances as for the other operator tests: 2e-5 relative L2 for an FP32
transform; 1e-13 for FP64 (about 10 rounding steps of 1.1e-16 per stage and
a sum of at most 61 terms, with a factor of 10 to spare).
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(np.complex64, 2e-5), (np.complex128, 1e-13)])
@pytest.mark.parametrize("W,Hk,C", [(7, 61, 2), (49, 53, 3), (121, 74, 5), (230, 217, 2), (13, 11, 1), (2, 59, 1)])
def test_operator_lengths_match_oracle(oracle, dtype, tol, W, Hk, C):
    import primaldualtoolbox as pdt
    rng = np.random.default_rng(W * 1000 + Hk)
    S = rng.standard_normal((C, Hk, W)) + 1j * rng.standard_normal((C, Hk, W))
    mask = np.repeat((rng.random(W) < 0.6)[None, :], Hk, axis=0).astype(np.float64)
    mask[:, 0] = 1.0
    S = S.astype(dtype)
    oop = oracle.Op(oracle.OP_CARTESIAN, S.astype(np.complex128), mask)
    op = pdt.mri.MriCartesianOperator(dtype=dtype)
    op.setCoilSens(S)
    op.setMask(mask)
    x = (rng.standard_normal((Hk, W)) + 1j * rng.standard_normal((Hk, W))).astype(dtype)
    y = (rng.standard_normal((C, Hk, W)) + 1j * rng.standard_normal((C, Hk, W))).astype(dtype)
    print(f"operator W={W} Hk={Hk} C={C} {np.dtype(dtype).name}", flush=True)
    assert rel_l2(op.forward(x), oop.forward(x.astype(np.complex128))) < tol
    assert rel_l2(op.adjoint(y), oop.adjoint(y.astype(np.complex128))) < tol

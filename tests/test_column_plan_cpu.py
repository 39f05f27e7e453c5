"""Columns per group of the MRI column pass (host rule): the lengths with the
kernel that holds the first and last stages in registers take as many columns
as it has threads for; every other length, and 256 points in single precision,
take the general kernel's two by default and at most what fits the LDS."""
import ctypes as ct

import pytest

# length, columns per group of the register kernel
DIRECT = [(320, 4), (384, 3), (512, 2), (640, 2), (768, 2)]


def _rules():
    from primaldualtoolbox import _capi as C
    most, default = C.lib()._ZN3pdt6max_cgEiii, C.lib()._ZN3pdt10default_cgEii
    for f, n in ((most, 3), (default, 2)):
        f.restype, f.argtypes = ct.c_int, [ct.c_int] * n
    return C, most, default


@pytest.mark.parametrize("n,columns", DIRECT)
def test_register_kernel_lengths(n, columns):
    C, most, default = _rules()
    for dtype in (C.PDT_C64, C.PDT_C128):
        assert default(dtype, n) == columns
        assert most(dtype, n, 1) == 1
    assert most(C.PDT_C64, n, 100) == columns


@pytest.mark.parametrize("n", [16, 200, 256, 368, 434, 736])
def test_general_kernel_lengths(n):
    C, most, default = _rules()
    assert default(C.PDT_C64, n) == 2
    assert most(C.PDT_C64, n, 0) == 1


def test_256_points_in_single_precision():
    C, most, default = _rules()
    assert most(C.PDT_C64, 256, 12) == 12  # bounded by LDS alone, not by threads


def test_256_points_in_double_precision():
    C, most, default = _rules()
    assert default(C.PDT_C128, 256) == 5 and most(C.PDT_C128, 256, 100) == 5

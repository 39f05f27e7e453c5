"""Coils per row item of the MRI passes of a single slice on rows without a
compile-time plan (host rule), where one item of the adjoint row pass holds
every coil and where it holds the same number: us per iteration with two and with four, measured on one MI355X.
The rule's choice is at most 5 % slower than the other one."""
import ctypes as ct

import pytest

# H, W, coils, precision, one item with every coil, us with 2, us with 4
MEASURED = [
    (320, 64, 12, "c64", True, 20.79, 18.47),
    (320, 64, 24, "c64", True, 25.85, 22.85),
    (384, 128, 20, "c64", True, 32.23, 29.55),
    (256, 64, 15, "c64", True, 19.99, 17.63),
    (256, 200, 24, "c64", True, 31.21, 28.32),
    (320, 200, 20, "c64", True, 35.65, 32.71),
    (192, 200, 20, "c64", True, 27.76, 25.54),
    (192, 64, 20, "c64", True, 20.31, 17.92),
    (128, 200, 12, "c64", True, 20.43, 20.95),
    (128, 64, 12, "c64", True, 16.53, 16.55),
    (128, 230, 20, "c64", True, 36.18, 37.91),
    (320, 64, 16, "c128", True, 30.07, 27.11),
    (320, 100, 12, "c128", True, 30.55, 27.84),
    (256, 64, 12, "c128", True, 22.36, 20.07),
    (128, 64, 20, "c128", True, 23.42, 21.32),
    (400, 230, 5, "c64", True, 38.12, 41.61),
    (200, 300, 20, "c64", False, 46.06, 41.67),
    (256, 300, 20, "c64", False, 44.23, 36.79),
    (128, 300, 20, "c64", False, 32.05, 31.95),
    (200, 500, 20, "c64", False, 57.44, 54.39),
    (256, 500, 16, "c64", False, 51.73, 48.96),
    (300, 500, 10, "c64", False, 49.39, 52.8),
    (225, 500, 20, "c64", False, 63.58, 72.8),
    (400, 400, 12, "c64", False, 64.56, 72.52),
    (256, 390, 20, "c64", False, 65.08, 60.73),
    (256, 390, 24, "c64", False, 72.23, 79.14),
]


@pytest.mark.parametrize("H,W,coils,dtype,one,two,four", MEASURED)
def test_the_faster_items(H, W, coils, dtype, one, two, four):
    from primaldualtoolbox import _capi as C
    rule = C.lib()._ZN3pdt10default_cbEiiiiib
    rule.restype, rule.argtypes = ct.c_int, [ct.c_int] * 5 + [ct.c_bool]
    cb = rule(C.PDT_C128 if dtype == "c128" else C.PDT_C64, W, H, coils, W // 4, one)
    assert cb in (2, 4)
    assert (two if cb == 2 else four) <= 1.05 * min(two, four)


@pytest.mark.parametrize("dtype,W,one,cb", [("c64", 320, True, 4), ("c128", 230, False, 4), ("c128", 320, False, 4)])
def test_other_rows(dtype, W, one, cb):
    from primaldualtoolbox import _capi as C
    rule = C.lib()._ZN3pdt10default_cbEiiiiib
    rule.restype, rule.argtypes = ct.c_int, [ct.c_int] * 5 + [ct.c_bool]
    for H, coils in ((1, 1), (320, 15), (1000, 20)):
        assert rule(C.PDT_C128 if dtype == "c128" else C.PDT_C64, W, H, coils, W // 4, one) == cb

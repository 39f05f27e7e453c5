"""The rule that runs a batch of operator solvers as concurrent single solves
or on the work lists (host function), at measured batches: ms per 100
iterations each way on one MI355X.  The way it takes is at most 5 % slower than
the other one."""
import ctypes as ct

import pytest


class _Slice(ct.Structure):
    _fields_ = [("W", ct.c_int), ("Hk", ct.c_int), ("x", ct.c_double), ("paired", ct.c_bool)]


# slices, (W, Hk) in turn, coils, operator, precision, work lists, single solves
MEASURED = [
    (4, [(128, 256)], 15, "roos", "c64", 4.27, 4.96),
    (3, [(128, 256)], 15, "roos", "c64", 3.80, 4.52),
    (4, [(128, 256)], 8, "roos", "c64", 3.41, 4.43),
    (6, [(368, 736)], 4, "roos", "c64", 9.67, 11.18),
    (4, [(160, 320)], 8, "roos", "c64", 3.93, 4.81),
    (4, [(128, 128)], 8, "cart", "c64", 3.37, 4.51),
    (3, [(128, 256)], 4, "roos", "c64", 2.69, 3.89),
    (4, [(256, 256)], 1, "samp", "c64", 3.09, 3.97),
    (2, [(384, 768)], 8, "roos", "c64", 5.70, 3.62),
    (2, [(96, 192)], 8, "roos", "c128", 3.19, 2.49),
    (16, [(256, 512), (320, 640), (320, 768), (368, 736)], 6, "roos", "c64", 35.02, 25.29),
    (2, [(128, 128)], 8, "cart", "c64", 2.97, 2.26),
    (2, [(48, 96), (64, 128)], 6, "roos", "c64", 5.34, 2.15),
    (8, [(320, 640)], 15, "roos", "c64", 21.30, 14.73),
    (4, [(256, 512), (320, 640)], 12, "roos", "c64", 10.35, 6.16),
    (6, [(64, 128), (96, 192), (128, 256), (160, 320)], 12, "roos", "c64", 12.21, 7.20),
    (2, [(368, 736)], 4, "roos", "c64", 4.74, 3.66),
    (16, [(256, 512)], 15, "roos", "c64", 26.37, 19.59),
    (8, [(256, 512)], 8, "roos", "c128", 19.74, 15.60),
    (6, [(128, 128)], 1, "samp", "c64", 3.15, 6.43),
    (8, [(64, 128)], 15, "roos", "c64", 4.37, 7.51),
    (8, [(96, 192)], 8, "roos", "c128", 4.17, 7.75),
    (32, [(192, 384)], 4, "roos", "c64", 13.45, 24.92),
    (16, [(180, 400), (230, 434)], 6, "roos", "c64", 21.53, 25.87),
    (8, [(128, 128)], 8, "cart", "c64", 4.28, 7.32),
]


@pytest.mark.parametrize("n,sizes,coils,op,dtype,lists,singles", MEASURED)
def test_the_faster_way(n, sizes, coils, op, dtype, lists, singles):
    from primaldualtoolbox import _capi as C
    rule = C.lib()._ZN3pdt20batch_singles_fasterEPKNS_10BatchSliceEi
    rule.restype, rule.argtypes = ct.c_bool, [ct.POINTER(_Slice), ct.c_int]
    fused = C.lib()._ZN3pdt17rows_adj_fused_okEiiii
    fused.restype, fused.argtypes = ct.c_bool, [ct.c_int] * 4
    s = []
    for i in range(n):
        W, Hk = sizes[i % len(sizes)]
        paired = dtype == "c64" and op != "samp" and W % 64 == 0 and fused(C.PDT_C64, W, coils, W // 4)
        s.append(_Slice(W, Hk, 0.5e-6 * (4 if dtype == "c128" else 1) * coils * W * Hk, paired))
    taken = singles if rule((_Slice * n)(*s), n) else lists
    assert taken <= 1.05 * min(lists, singles)

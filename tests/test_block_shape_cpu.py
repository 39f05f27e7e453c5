"""Workgroups of the blocked denoising launches (host rule): a tile narrower
than a region's 64 columns is widened to them, so a narrow tile (one chosen for
another kernel, from a saved file or a program) takes no more workgroups than
the widest of its rows and iterations."""
import ctypes as ct

import pytest


class _Shape(ct.Structure):
    _fields_ = [("ry", ct.c_int), ("waves", ct.c_int), ("grid", ct.c_int), ("nbx", ct.c_int)]


@pytest.mark.parametrize("kind,dtype,rows", [(0, 0, 64), (0, 1, 64), (0, 2, 64), (0, 3, 32), (1, 0, 64), (1, 1, 32),
                                             (1, 2, 32), (1, 3, 32)])
def test_narrow_tiles_are_widened(kind, dtype, rows):
    from primaldualtoolbox import _capi as C
    f = C.lib()._ZN3pdt11block_shapeEiiiiiii  # pdt::block_shape(kind, dtype, W, H, tx, ty, k)
    f.restype, f.argtypes = _Shape, [ct.c_int] * 7
    for W, H in ((47, 61), (64, 64), (65, 200), (512, 512), (1100, 961)):
        for k in (1, 4, 6, 12, 20, 31):
            for ty in (1, 8, 16, 32, 64):
                wide = f(kind, dtype, W, H, 64 - 2 * k, ty, k)
                # whole waves of four rows around tile and halo, as many as the image has
                waves = min((min(ty, rows) + 2 * min(k, rows) + 3) // 4, rows // 4, (H + 3) // 4)
                if H > 4 * waves and 4 * waves <= 2 * k:
                    assert wide.grid == 0
                else:
                    assert (wide.waves, wide.ry) == (waves, 4 * waves)
                    nx = 1 if W <= 64 else -(-(W - 2 * k) // (64 - 2 * k))
                    ny = 1 if H <= wide.ry else -(-(H - 2 * k) // (wide.ry - 2 * k))
                    assert (wide.grid, wide.nbx) == (nx * ny, nx)
                for tx in (1, 2, 16, 31, 32, 48, 64, 200):
                    s = f(kind, dtype, W, H, tx, ty, k)
                    assert (s.ry, s.waves, s.grid) == (wide.ry, wide.waves, wide.grid)
        assert f(kind, dtype, 65, 200, 8, 8, 32).grid == 0

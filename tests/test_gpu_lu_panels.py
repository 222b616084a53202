"""The blocked LU's panels at the sizes and places where they can go wrong, through sfh_debug_lu_solve
against LAPACK (numpy): last blocks of every remainder class (one 16-wide step, a part of one, several
panels with a short last block), more trailing tiles than workgroups, and the interchange check with
a single multiplier above 1 placed in each part that checks it.

Tolerance: an LU solution without growth has a relative error of at most about n eps cond(A); the systems
are near 0.5 I (cond < 1.1), the bound used is 2 n eps."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _solve(n, A, b):
    import cusuperhelium as c
    x, flag = np.empty(n), ctypes.c_int(-1)
    dp = ctypes.POINTER(ctypes.c_double)
    A = np.ascontiguousarray(A)
    assert c.lib().sfh_debug_lu_solve(n, A.ctypes.data_as(dp), b.ctypes.data_as(dp), x.ctypes.data_as(dp),
                                      ctypes.byref(flag)) == 0
    return x, flag.value


@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 33, 48, 63, 64, 65, 80, 96, 128, 129, 144, 192, 250, 320, 960, 1000])
def test_lu_sizes(n):
    print(f"lu panels n={n}", flush=True)
    rng = np.random.default_rng(n)
    A = rng.uniform(-1, 1, (n, n)) * (0.02 / n) + 0.5 * np.eye(n)
    b = rng.uniform(-1, 1, n)
    x, flag = _solve(n, A, b)
    xr = np.linalg.solve(A, b)
    assert flag == 0
    assert np.abs(x - xr).max() <= 2 * n * EPS * np.abs(xr).max()


# (row, column) of the one entry that forces an interchange: inside a 16 x 16 tile, between the tiles of
# a diagonal block (next to it, further down), in a block below it, in a later panel's tile and block
@pytest.mark.parametrize("row,col", [(5, 2), (20, 3), (63, 14), (64, 0), (130, 40), (70, 66), (140, 100), (143, 130)])
def test_lu_interchange_found(row, col):
    n = 144
    print(f"lu interchange at {row} {col}", flush=True)
    rng = np.random.default_rng(row)
    A = rng.uniform(-1, 1, (n, n)) * (0.02 / n) + 0.5 * np.eye(n)
    A[row, col] = 1.0
    b = rng.uniform(-1, 1, n)
    x, flag = _solve(n, A, b)
    xr = np.linalg.solve(A, b)
    assert flag == 1
    assert np.abs(x - xr).max() <= 2 * n * EPS * np.linalg.cond(A) * np.abs(xr).max()

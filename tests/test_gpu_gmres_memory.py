"""GMRES handles that form their products from cotangent sums keep no matrix: 4 water surfaces of 4096 nodes, 134 MB of
matrix each, take a few vectors per Krylov step (33 of 32 KB, sums and basis: less than 8 MB a handle).

The free memory is asked of the HIP runtime that the library is bound to, opened by its SONAME."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def test_gmres_handles_without_a_matrix_allocate_none():
    import cusuperhelium as c
    with c.Ensemble([4096], c.Props(), solver=c.GMRES):   # whatever a first handle loads
        pass
    hip = ctypes.CDLL("libamdhip64.so.7")

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value
    before = free()
    handles = [c.Ensemble([4096], c.Props(), solver=c.GMRES) for _ in range(4)]
    used = before - free()
    for h in handles:
        h.close()
    print(f"4 handles of 4096 nodes: {used / 1e6:.0f} MB", flush=True)
    assert 0 < used < 134e6

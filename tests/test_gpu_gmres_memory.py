"""GMRES handles that form their products from cotangent sums keep no matrix: 4 water surfaces of 4096 nodes, 134 MB of
matrix each, take a few vectors per Krylov step (33 of 32 KB, sums and basis: less than 8 MB a handle)."""
import pytest

pytestmark = pytest.mark.gpu


def test_gmres_handles_without_a_matrix_allocate_none():
    import cusuperhelium as c
    import torch
    with c.Ensemble([4096], c.Props(), solver=c.GMRES):   # whatever a first handle loads
        pass
    free = torch.cuda.mem_get_info()[0]
    handles = [c.Ensemble([4096], c.Props(), solver=c.GMRES) for _ in range(4)]
    used = free - torch.cuda.mem_get_info()[0]
    for h in handles:
        h.close()
    print(f"4 handles of 4096 nodes: {used / 1e6:.0f} MB", flush=True)
    assert used < 134e6

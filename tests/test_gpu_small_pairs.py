"""The pair kernels of surfaces of up to 256 nodes (LU), whose waves own 4 whole rows each, against the oracle: sizes below
a wave's rows and columns, at and beside multiples of 16 and 64, the largest, and mixed sizes in one launch, also beside a
surface of 384 nodes (which takes the whole handle to the general kernels); water with and without the rho quirk, film.

Tolerance: 1e-12 (1 + max), as the parity tests of the general kernels use."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _surface(n, seed):
    rng = np.random.default_rng(seed)
    x = 2 * np.pi * np.arange(n) / n
    y = sum(rng.uniform(0, 0.05 / k) * np.cos(k * x + rng.uniform(0, 2 * np.pi)) for k in range(1, 4))
    return x + 1j * y, 0.01 * np.sin(x + 0.3)


@pytest.mark.parametrize("kw", [{}, dict(rho=0.3), dict(kind=1, depth=1.0), dict(kind=1, depth=0.8, kappa=0.01)], ids=str)
@pytest.mark.parametrize("sizes", [[1, 2, 3], [4, 6, 12, 16], [24, 48, 64], [96, 192], [256, 32], [256, 384]], ids=str)
def test_small_surfaces_match_oracle(oracle, sizes, kw):
    import cusuperhelium as c
    print(f"small surfaces {sizes} {kw}", flush=True)
    parts = [_surface(n, 5 + n) for n in sizes]
    Z, P = (np.concatenate(v) for v in zip(*parts))
    with c.Ensemble(sizes, c.Props(**kw)) as e:
        e.set_state(Z, P)
        q, dp, d = e.rhs(diagnostics=True)
    o = 0
    for n, (z, p) in zip(sizes, parts):
        qo, dpo, do = oracle.rhs(oracle.Props(**kw), z, p, diagnostics=True)
        for a, b in ((d["mu"], do["mu"]), (q, qo), (dp, dpo)):
            assert np.abs(a[o:o + n] - b).max() <= 1e-12 * (1 + np.abs(b).max()), n
        o += n

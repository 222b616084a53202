"""Surfaces of the batched stage that are shared by several workgroups: a right-hand side and steps against the
direct (LU) solver, and against runs in which fewer workgroups join than the work has parts (force_trim, the test
hook, launches at most that many), which have to give the same bits.  Sizes: no multiple of 64, one to sixteen blocks
of 64, alone and beside surfaces that are not shared; water and film, FP64 and mixed.

Tolerance against LU: both solutions satisfy |b - M mu| <= tol |b| with tol = 1e-13 (rounding for the LU) and M's
smallest singular value is about 1/2, so 1e-12 (1 + max), as the other solves' tests use."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(n, seed):
    rng = np.random.default_rng(seed)
    x = 2 * np.pi * np.arange(n) / n
    y = sum(rng.uniform(0, 0.05 / k) * np.cos(k * x + rng.uniform(0, 2 * np.pi)) for k in range(1, 9))
    return x + 1j * y, 0.01 * np.sin(x + 0.3) + 0.004 * np.cos(3 * x)


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
@pytest.mark.parametrize("film", [False, True], ids=["water", "film"])
@pytest.mark.parametrize("sizes", [[192], [256], [384], [512, 96], [768, 1, 48], [1024], [1024, 768, 384, 24]], ids=str)
def test_shared_surfaces(sizes, film, mixed):
    import cusuperhelium as c
    print(f"shared surfaces {sizes} film {film} mixed {mixed}", flush=True)
    parts = [_state(n, 7 + n) for n in sizes]
    Z, P = (np.concatenate(v) for v in zip(*parts))
    props = c.Props(kind=c.HELIUM, depth=1.0, g=0.15) if film else c.Props()
    with c.Ensemble(sizes, props) as e:
        e.set_state(Z, P)
        q0, d0 = e.rhs()
    out = []
    for wgs in (0, 1, 3):
        with c.Ensemble(sizes, props, solver=c.BATCHED, tol=1e-13, precision=c.MIXED if mixed else c.FP64, force_trim=wgs) as e:
            e.set_state(Z, P)
            q1, d1 = e.rhs()
            e.step(0.002, 2)
            out.append((q1, d1) + tuple(e.get_state()))
            assert e.stats()["unconverged"] == 0
    for a, b in zip(out[0], (q0, d0)):
        assert np.abs(a - b).max() <= 1e-12 * (1 + np.abs(b).max())
    for o in out[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(o, out[0]))

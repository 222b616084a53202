"""Films of the fewest nodes, GMRES and BATCHED against the direct (LU) solve: the preconditioner's Fourier modes have
to stay below n / 2.  The depths are those at which the projections with aliased modes add up to a singular matrix
(found by bisection for n = 2, 3, 4), and two beside them.

Tolerance: as in the other film solves, both end at |b - M mu| <= 1e-13 |b| and M's smallest singular value is about
1/2 or more, so 1e-12 (1 + max) holds for mu, q and dPhi/dt."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", ["gmres", "batched"])
@pytest.mark.parametrize("depth", [0.08, 0.1071283190426088, 0.11076935424690315, 0.1231377483995334, 0.15])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 6, 8])
def test_smallest_films_match_lu(n, depth, solver):
    import cusuperhelium as c
    print(f"film n {n} depth {depth} {solver}", flush=True)
    x = 2 * np.pi * np.arange(n) / n
    P = 0.01 * np.sin(x + 0.3)
    props = c.Props(kind=c.HELIUM, depth=depth, g=0.15)
    for amp in (0.0, 0.2 * depth):
        Z = x + 1j * amp * np.sin(x + 0.7)
        with c.Ensemble([n], props) as e:
            e.set_state(Z, P)
            q0, d0, g0 = e.rhs(diagnostics=True)
        with c.Ensemble([n], props, solver={"gmres": c.GMRES, "batched": c.BATCHED}[solver], tol=1e-13) as e:
            e.set_state(Z, P)
            q1, d1, g1 = e.rhs(diagnostics=True)
            assert e.stats()["unconverged"] == 0
        for a, b in ((g1["mu"], g0["mu"]), (q1, q0), (d1, d0)):
            assert np.abs(a - b).max() <= 1e-12 * (1 + np.abs(b).max())

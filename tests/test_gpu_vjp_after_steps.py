"""sfh_rhs_vjp on a GMRES handle that has stepped past the calibration of its launch sequence, and after a
trajectory's backward pass: the forward solve at the current state is a standalone one and gets the full sequence,
whatever length the calls before it left behind.

Tolerance: against a fresh handle at the same state.  Both forward solves end at |b - M mu| <= 1e-13 |b| and both
transposed ones at their 1e-13, with M's smallest singular value about 1/2, so mu and gb differ by less than 4e-13
relative; the reverse pass is linear in each with coefficients of order n / 2 at most (two derivatives).  With n = 192
that is 1e-10 of the largest entry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N = 192


def _state(amp):
    x = 2 * np.pi * np.arange(N) / N
    return x + 1j * amp * (np.cos(x) + 0.5 * np.sin(2 * x + 0.4)), 0.01 * np.sin(x + 0.3) + 0.004 * np.cos(3 * x)


def _cotangent():
    x = 2 * np.pi * np.arange(N) / N
    return np.cos(3 * x) + 1j * np.sin(2 * x), np.cos(x)


@pytest.mark.parametrize("before", ["steps", "backward"])
@pytest.mark.parametrize("kw", [dict(), dict(rho=0.3), dict(kind=1, depth=1.0, g=0.15)], ids=["water", "rho", "film"])
def test_gmres_rhs_vjp_after_other_calls_matches_a_fresh_handle(kw, before):
    import cusuperhelium as c
    print(f"rhs_vjp after {before} {kw}", flush=True)
    Z, P = _state(0.1)
    gq, gp = _cotangent()
    with c.Ensemble([N], c.Props(**kw), solver=c.GMRES, tol=1e-13) as e:
        e.set_state(Z, P)
        if before == "steps":
            e.step(0.005, 12)
        else:
            rec = e.traj_forward(0.005, 12, 6)
            e.traj_backward(rec, gq, gp)
            e.traj_release(rec)
        Zs, Ps = e.get_state()
        gZ, gP = e.rhs_vjp(gq, gp)
        unconverged = e.stats()["unconverged"]
    with c.Ensemble([N], c.Props(**kw), solver=c.GMRES, tol=1e-13) as e:
        e.set_state(Zs, Ps)
        gZ0, gP0 = e.rhs_vjp(gq, gp)
    assert unconverged == 0
    for a, b in ((gZ, gZ0), (gP, gP0)):
        assert np.abs(a - b).max() <= 1e-10 * np.abs(b).max()

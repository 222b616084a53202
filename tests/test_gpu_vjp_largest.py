"""Reverse mode of the largest surfaces that LU handles take (above the 4096 nodes of the GMRES solver): <g, J v> by
central differences of the right-hand side against <J^T g, v>.

Tolerance: with the step h = 1e-4 along a direction v of a few low modes, the truncation is h^2 / 6 times a third
derivative of order 10, about 2e-8, and the rounding of the right-hand sides, about 1e-12 of their size, becomes 1e-8
divided by 2 h; both relative to sum |g| |J v|.  1e-6 of that sum is used."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kw", [(192, dict()), (6144, dict()), (8192, dict(kind=1, depth=1.0, g=0.15))],
                         ids=["water192", "water6144", "film8192"])
def test_rhs_vjp_of_the_largest_lu_surfaces(n, kw):
    import cusuperhelium as c
    print(f"rhs_vjp LU n {n} {kw}", flush=True)
    x = 2 * np.pi * np.arange(n) / n
    Z, P = x + 0.05j * (np.cos(x) + 0.4 * np.sin(2 * x + 0.4)), 0.05 * np.sin(x + 0.3)
    vZ, vP = 0.3 * np.sin(x) + 1j * np.cos(2 * x), np.cos(x + 1.0)
    gq, gp = np.cos(3 * x) + 1j * np.sin(2 * x), np.cos(x)
    h = 1e-4
    with c.Ensemble([n], c.Props(**kw)) as e:
        e.set_state(Z + h * vZ, P + h * vP)
        qp, dp = e.rhs()
        e.set_state(Z - h * vZ, P - h * vP)
        qm, dm = e.rhs()
        e.set_state(Z, P)
        gZ, gP = e.rhs_vjp(gq, gp)
    jq, jd = (qp - qm) / (2 * h), (dp - dm) / (2 * h)
    terms = np.concatenate([(np.conj(gq) * jq).real, gp * jd])
    back = (np.conj(gZ) * vZ).real.sum() + (gP * vP).sum()
    assert abs(terms.sum() - back) <= 1e-6 * np.abs(terms).sum()

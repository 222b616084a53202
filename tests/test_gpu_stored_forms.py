"""The pair kernels with 1, 2 and 4 rows per workgroup and the stored matrices of GMRES (FP64, FP32 with a refinement
solve), on sizes and physics that launch them: LU above 256 nodes and with the rho quirk, GMRES with the rho quirk, up
to 2048 nodes in all (4 matrix rows per workgroup) and above (16), one surface and uneven ones.

Tolerances as for the other forms: right-hand sides 1e-12 relative to 1 + max|reference| (mixed precision 1e-9, the
bound of its refinement at tol 1e-13), trajectories of 10 steps 1e-11 and 1e-9."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _surface(n, seed, amp=0.03):
    rng = np.random.default_rng(seed)
    x = 2 * np.pi * np.arange(n) / n
    a = rng.uniform(0, amp / np.arange(1, 9))
    th = rng.uniform(0, 2 * np.pi, 8)
    return x + 1j * sum(a[k] * np.cos((k + 1) * x + th[k]) for k in range(8)), 0.01 * np.cos(x + 0.2 * seed)


def _close(a, b, tol):
    assert np.abs(a - b).max() <= tol * (1.0 + np.abs(b).max())


@pytest.mark.parametrize("rows", [1, 2, 4])
@pytest.mark.parametrize("n,kw", [(384, dict()), (384, dict(kind=1, depth=1.0)), (192, dict(rho=0.3)), (384, dict(rho=0.3))],
                         ids=["water384", "film384", "rho192", "rho384"])
def test_lu_rows_match_oracle(oracle, n, kw, rows):
    import cusuperhelium as c
    print(f"lu rows {rows} n {n} {kw}", flush=True)
    Z, P = _surface(n, 31 + rows)
    q0, d0 = oracle.rhs(oracle.Props(**kw), Z, P)
    Zo, Po = oracle.rk4(oracle.Props(**kw), Z, P, 0.002, 4)
    with c.Ensemble([n], c.Props(**kw), pair_rows=rows) as e:
        e.set_state(Z, P)
        e.kernel_timing(True)
        q, d = e.rhs()
        assert e.kernel_report("mu_deriv")["launches"] == 1   # not the small-surface velocity
        e.kernel_timing(False)
        e.step(0.002, 4)
        Zg, Pg = e.get_state()
    for a, b, tol in ((q, q0, 1e-12), (d, d0, 1e-12), (Zg, Zo, 1e-11), (Pg, Po, 1e-11)):
        _close(a, b, tol)


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
@pytest.mark.parametrize("sizes,rows", [([192], 1), ([192], 2), ([192], 4), ([512, 96, 1024], 4), ([1536, 96, 12, 768], 2),
                                        ([3072], 4)], ids=str)
def test_stored_matrix_gmres_matches_lu(sizes, rows, mixed):
    import cusuperhelium as c
    print(f"stored gmres {sizes} rows {rows} mixed {mixed}", flush=True)
    Z, P = (np.concatenate(v) for v in zip(*[_surface(n, 50 + i) for i, n in enumerate(sizes)]))
    props = c.Props(rho=0.3)
    with c.Ensemble(sizes, props) as e:
        e.set_state(Z, P)
        q0, d0 = e.rhs()
        e.step(0.002, 10)
        Z0, P0 = e.get_state()
    with c.Ensemble(sizes, props, solver=c.GMRES, tol=1e-13, pair_rows=rows, precision=c.MIXED if mixed else c.FP64) as e:
        e.set_state(Z, P)
        e.kernel_timing(True)
        q, d = e.rhs()
        assert e.kernel_report("assemble")["launches"] == 1
        assert e.kernel_report("residual")["launches"] == (1 if mixed else 0)
        e.kernel_timing(False)
        e.step(0.002, 10)
        Zg, Pg = e.get_state()
        assert e.stats()["unconverged"] == 0
    rtol, ttol = (1e-9, 1e-9) if mixed else (1e-12, 1e-11)
    for a, b, tol in ((q, q0, rtol), (d, d0, rtol), (Zg, Z0, ttol), (Pg, P0, ttol)):
        _close(a, b, tol)

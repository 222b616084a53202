"""GMRES on films too thin for the preconditioner of the image term.

They take the stored matrix, in both row splits (up to 2048 nodes in all and above) and in uneven handles, deeper ones
and the thinnest of up to 2048 nodes the cotangent sums; and a solve that ends at its step limit still has to be a
solution up to a residual."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(n, seed, amp):
    rng = np.random.default_rng(seed)
    x = 2 * np.pi * np.arange(n) / n
    y = sum(rng.uniform(0, amp / k) * np.cos(k * x + rng.uniform(0, 2 * np.pi)) for k in range(1, 9))
    return x + 1j * y, 0.01 * np.sin(x + 0.3) + 0.004 * np.cos(3 * x)


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
@pytest.mark.parametrize("sizes,depth,stored", [([768], 0.2, True), ([3072], 0.25, True), ([512, 64, 2048], 0.2, True),
                                                ([256], 0.05, True), ([128], 0.1, False), ([512], 0.02, False),
                                                ([768], 0.4, False)], ids=str)
def test_thin_films_match_lu(sizes, depth, stored, mixed):
    # both solutions end at |b - M mu| <= 1e-11 |b| (LU at rounding), M's smallest singular value is about 1/2: mu differs
    # by at most 4e-11 |b|; mu' and with it the velocity by n / 2 times that, and 8 steps of dt = 1e-3 add up to less
    import cusuperhelium as c
    print(f"thin film {sizes} depth {depth} mixed {mixed}", flush=True)
    parts = [_state(n, 7 + n, 0.05 * depth) for n in sizes]
    Z, P = (np.concatenate(v) for v in zip(*parts))
    props = c.Props(kind=c.HELIUM, depth=depth, g=0.15)
    out = []
    for solver in (c.LU, c.GMRES):
        with c.Ensemble(sizes, props, solver=solver, tol=1e-11, precision=c.MIXED if mixed and solver == c.GMRES else c.FP64) as e:
            e.set_state(Z, P)
            e.kernel_timing(True)
            q, d, diag = e.rhs(diagnostics=True)
            if solver == c.GMRES:
                assert (e.kernel_report("assemble")["launches"] > 0) == stored
            e.kernel_timing(False)
            e.step(1e-3, 8)
            out.append((diag["mu"], q, d, *e.get_state()))
            assert e.stats()["unconverged"] == 0
    bnorm = 0.02 * np.sqrt(sum(sizes))   # |b| <= 0.01 + 0.012 per node
    n = max(sizes)
    for u, v, bound in zip(out[1], out[0], (4e-11 * bnorm,) + 4 * (2e-11 * n * bnorm,)):
        assert np.abs(u - v).max() <= bound


# residual allowed at 1e-13 within the step limit: None where the solve has to converge (then 2e-13, with the rounding of
# the check's own product), else ten times what the solver without a preconditioner has always reached there
@pytest.mark.parametrize("n,depth,solver,mixed,bound", [
    (256, 0.05, "gmres", False, 1e-10), (256, 0.05, "gmres", True, 1e-10), (256, 0.05, "batched", False, 1e-9),
    (256, 0.05, "batched", True, 2e-11), (512, 0.02, "gmres", False, None), (512, 0.02, "gmres", True, None),
    (512, 0.02, "batched", False, None), (512, 0.02, "batched", True, 3e-11), (256, 0.15, "gmres", False, 2e-12),
    (256, 0.15, "gmres", True, 2e-12), (256, 0.15, "batched", False, 2e-6), (256, 0.15, "batched", True, 2e-8),
    (128, 0.15, "gmres", False, None), (128, 0.15, "gmres", True, None), (128, 0.15, "batched", False, 1e-7),
    (128, 0.15, "batched", True, 1e-10)])
def test_thin_film_residuals(oracle, n, depth, solver, mixed, bound):
    import cusuperhelium as c
    print(f"residual n {n} depth {depth} {solver} mixed {mixed}", flush=True)
    Z, P = _state(n, 7 + n, min(0.05, 0.3 * depth))
    kw = dict(kind=1, depth=depth, g=0.15)
    Zp, Zpp, Pp = oracle.zphi_derivative(oracle.Props(**kw), Z, P)
    M, b = oracle.assemble(oracle.Props(**kw), Z, Zp, Zpp), Pp.real
    with c.Ensemble([n], c.Props(**kw), solver={"gmres": c.GMRES, "batched": c.BATCHED}[solver], tol=1e-13,
                    precision=c.MIXED if mixed else c.FP64) as e:
        e.set_state(Z, P)
        q, d, diag = e.rhs(diagnostics=True)
        unconverged = e.stats()["unconverged"]
    assert all(np.all(np.isfinite(v)) for v in (q, d, diag["mu"]))
    residual = np.linalg.norm(b - M @ diag["mu"]) / np.linalg.norm(b)
    print(f"  unconverged {unconverged} residual {residual:.2e}", flush=True)
    if bound is None:
        assert unconverged == 0 and residual <= 2e-13
    else:
        assert residual <= bound

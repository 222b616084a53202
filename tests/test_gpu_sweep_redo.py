"""The reverse sweep over thin films, whose transposed solves keep needing more steps than the sequence that the step
before suggests: what ran out of launches while the warm-start rings fill is run again step by step, not the segment
with it.  Six reverse steps in one segment: the first has the full sequence, the other five are the ones that can be
run again, so fewer than six are."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(n, depth):
    x = 2 * np.pi * np.arange(n) / n
    rng = np.random.default_rng(1)
    amp = 0.05 * depth
    y = sum(rng.uniform(0.5 * amp / k, amp / k) * np.cos(k * x + rng.uniform(0, 2 * np.pi)) for k in range(1, 5)) / 2
    k = np.arange(1, 40)[:, None]
    rough = np.cos(k * x + rng.uniform(0, 2 * np.pi, (39, 1))) / np.sqrt(k)
    return (x + 1j * y, 0.01 * np.sin(x + 0.3) + 0.004 * np.cos(3 * x), rough.sum(0) + 1j * rough[::-1].sum(0),
            np.roll(rough.sum(0), 7))


def _gradient(n, depth, solver, steps, every):
    import cusuperhelium as c
    print(f"sweep n {n} depth {depth} {solver} steps {steps}", flush=True)
    Z, P, gZ, gP = _case(n, depth)
    sv = {"lu": c.LU, "gmres": c.GMRES, "batched": c.BATCHED}[solver]
    with c.Ensemble([n], c.Props(kind=c.HELIUM, depth=depth, g=0.15), solver=sv, tol=1e-13,
                    max_iter=48 if solver == "batched" else 32) as e:
        e.set_state(Z, P)
        rec = e.traj_forward(0.001, steps, every)
        before = e.stats()["redone_steps"]
        out = e.traj_backward(rec, gZ, gP)
        st = e.stats()
        e.traj_release(rec)
    return out, st["redone_steps"] - before, st["unconverged"]


@pytest.mark.parametrize("solver", ["lu", "gmres"])
@pytest.mark.parametrize("n,depth", [(128, 0.1), (512, 0.1)])
def test_steps_of_a_segment_are_run_again_alone(n, depth, solver):
    _, redone, _ = _gradient(n, depth, solver, 6, 6)
    assert redone < 6


@pytest.mark.parametrize("solver", ["lu", "gmres"])
def test_gradient_with_steps_run_again_matches_the_batched_solver(solver):
    # both solve to 1e-13 (the restarted solver of the one-workgroup reverse pass needs no sequence): a solution's error
    # of 4e-13 is multiplied by at most n / 2 = 256 (two derivatives), and 160 stages add up to 1.6e-8 of the largest
    # entry; 1e-7 is used
    a, redone, unconverged = _gradient(512, 0.3, solver, 40, 20)
    print(f"  redone {redone} unconverged {unconverged}", flush=True)
    b, _, _ = _gradient(512, 0.3, "batched", 40, 20)
    assert unconverged == 0
    for u, v in zip(a, b):
        assert np.abs(u - v).max() <= 1e-7 * np.abs(v).max()

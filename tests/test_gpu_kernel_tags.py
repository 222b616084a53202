"""What a kernel report's tags stand for on GMRES handles: without a stored matrix the closing launch forms the velocity
and is reported as that, whatever the sequence's length (also the full one of the first step); with one the closing
launch and the velocity are two."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw,stored", [(dict(), False), (dict(kind=1, depth=1.0, g=0.15), False), (dict(rho=0.3), True)],
                         ids=["water", "film", "rho"])
def test_closing_launches_of_a_step(kw, stored):
    import cusuperhelium as c
    print(f"tags {kw}", flush=True)
    n = 192
    x = 2 * np.pi * np.arange(n) / n
    with c.Ensemble([n], c.Props(**kw), solver=c.GMRES) as e:
        e.set_state(x + 0.02j * np.cos(x), 0.01 * np.sin(x))
        e.kernel_timing(True)
        e.step(0.002, 1)
        e.sync()
        count = {t: e.kernel_report(t)["launches"] for t in ("velocity", "gm_close_mu", "gm_start", "assemble")}
    assert count == ({"velocity": 4, "gm_close_mu": 4, "gm_start": 0, "assemble": 4} if stored else
                     {"velocity": 4, "gm_close_mu": 0, "gm_start": 4, "assemble": 0})

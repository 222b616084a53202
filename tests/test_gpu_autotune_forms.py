"""The tuner times what differs: where the rows per workgroup and the precision change no launch it reports the
defaults, and a ranking of rho = 0 (or of a deep film) is not applied where GMRES takes its other route."""
import os

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture()
def cache(tmp_path):
    # entries of this process stay in memory, so every test uses sizes of its own
    os.environ["SFH_TUNE_CACHE"] = str(tmp_path / "tuning.txt")
    yield tmp_path / "tuning.txt"
    del os.environ["SFH_TUNE_CACHE"]


def test_equal_forms_are_not_ranked(cache):
    import cusuperhelium as c
    for n in (16, 24, 32, 48, 64, 96, 128, 192):
        t = c.autotune(n, allow_mixed=True, steps=2)
        print(n, t, flush=True)
        assert t["pair_rows"] == 4
        assert t["precision"] == c.FP64 or t["solver"] == c.BATCHED


@pytest.mark.parametrize("a,b", [(dict(), dict(rho=0.3)), (dict(kind=1, depth=1.0, g=0.15), dict(kind=1, depth=0.1, g=0.15))],
                         ids=["rho", "thin"])
def test_rankings_are_kept_per_gmres_route(cache, a, b):
    import cusuperhelium as c
    n = 384
    c.autotune(n, c.Props(**a), steps=2)
    assert c.tuned(n, c.Props(**a))["from_cache"]
    assert not c.tuned(n, c.Props(**b))["from_cache"]
    assert c.tuned(n, c.Props(**b))["from_cache"] and c.tuned(n, c.Props(**a))["from_cache"]
    keys = [ln.split()[:5] for ln in cache.read_text().splitlines() if not ln.startswith("#")]
    assert len({tuple(k) for k in keys}) == len(keys)

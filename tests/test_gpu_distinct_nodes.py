"""set_state refuses two nodes at one point (x mod 2 pi, y).  Surfaces listed in order of x take a check without a
sort; what it accepts and refuses is compared with all pairs' comparison: in order, with one wrap at any node, from
negative and from far-away x, in reverse and shuffled, overturning, with coincident nodes next to each other, across
the wrap, and where a tiny negative x rounds to the node at 0."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TWO_PI = 2.0 * np.pi


def _reduced(x):
    r = np.fmod(x, TWO_PI)
    r = np.where(r < 0, r + TWO_PI, r)
    return np.where(r >= TWO_PI, 0.0, r)


def _cases(n):
    rng = np.random.default_rng(n)
    x, y = TWO_PI * np.arange(n) / n, 0.1 * rng.standard_normal(n)
    yield "ordered", x, y
    yield "wrapped", np.roll(x, n // 3), y
    yield "beyond one period", x + 1.0, y
    yield "negative", x - np.pi, y
    yield "far away", x - 20 * np.pi + 0.3, y
    yield "reversed", x[::-1].copy(), y
    yield "shuffled", rng.permutation(x), y
    yield "overturning", x + 1.5 * np.sin(3 * x), y
    if n < 3:
        return
    two = x.copy()
    two[n // 2] = two[n // 2 - 1]
    yield "same x, other y", two, y
    same = y.copy()
    same[n // 2] = same[n // 2 - 1]
    yield "coincident neighbours", two, same
    ends = y.copy()
    ends[-1] = ends[0]
    last = x.copy()
    last[-1] = TWO_PI
    yield "coincident across the period", last, ends
    tiny = np.roll(x, 1)
    tiny[0] = -1e-20
    ends = y.copy()
    ends[0] = ends[1]
    yield "rounds to the node at 0", tiny, ends
    twice = x.copy()
    twice[n // 2:] = twice[:n - n // 2]
    yield "two sweeps, other y", twice, y
    yield "two sweeps, coincident", twice, np.concatenate([y[:n // 2], y[:n - n // 2]])


@pytest.mark.parametrize("n", [1, 2, 3, 8, 96])
def test_coincident_nodes_as_all_pairs(n):
    import cusuperhelium as c
    with c.Ensemble([4, n]) as e:
        z0 = TWO_PI * np.arange(4) / 4 + 0j
        for name, x, y in _cases(n):
            r = _reduced(x)
            refused = any(r[i] == r[j] and y[i] == y[j] for i in range(n) for j in range(i))
            print(f"distinct nodes n={n}: {name}, refused {refused}", flush=True)
            Z, P = np.concatenate([z0, x + 1j * y]), np.zeros(4 + n)
            if refused:
                with pytest.raises(Exception, match="coincident nodes .* of surface 1"):
                    e.set_state(Z, P)
            else:
                e.set_state(Z, P)
                assert np.array_equal(e.get_state()[0], Z)

"""The circulant derivative kernels against the oracle's FFT derivatives: every launch shape (up to 256, 1024 and
2048 nodes and above, where the columns come in several chunks), sizes below a wave, 3 * 2^k sizes that leave a
part of a chunk empty, surfaces of different sizes in one launch; with LU (mu' by its own kernel) and with GMRES
(mu' in the closing launch).

Tolerance: a row is a dot product of n terms, of which a thread adds at most 16 per chunk in sequence (4 columns
of at most 4 chunks) before a tree of sums; its rounding error is at most 40 eps / 2 times sum_j |c_j| |v_j|, and
the oracle's FFT stays well below that.  The bound used is 40 eps S max |v|, S the kernel's absolute row sum.  mu'
shows in the velocity: the two solvers' agree within 1e-12 (1 + max), as their solutions do in the other tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _surface(n, seed):
    rng = np.random.default_rng(seed)
    x = 2 * np.pi * np.arange(n) / n
    y = sum(rng.uniform(0, 0.05 / k) * np.cos(k * x + rng.uniform(0, 2 * np.pi)) for k in range(1, 9))
    return x + 0.01 * np.sin(x + 1.0) + 1j * y, 0.01 * np.sin(x + 0.3)


def _row_sum(O, n, second):
    e = np.zeros(n, np.complex128)
    e[0] = 1.0
    return np.abs(O.fft_derivative(e, second=second)).sum()


@pytest.mark.parametrize("sizes", [[1, 2, 3, 24, 48], [64, 192, 256], [384], [1024, 96], [1536, 12], [2048], [3072, 256], [4096]], ids=str)
def test_circulant_derivatives_match_fft(oracle, sizes):
    import cusuperhelium as c
    print(f"circulant derivatives {sizes}", flush=True)
    parts = [_surface(n, 3 + n) for n in sizes]
    Z, P = (np.concatenate(v) for v in zip(*parts))
    eps, q = np.finfo(float).eps, []
    for solver in (c.LU, c.GMRES):
        with c.Ensemble(sizes, c.Props(), solver=solver, tol=1e-13) as e:
            e.set_state(Z, P)
            u, dp, d = e.rhs(diagnostics=True)
        q.append(u)
        o = 0
        for n, (z, p) in zip(sizes, parts):
            zp, zpp, _ = oracle.zphi_derivative(oracle.Props(), z, p.astype(complex))
            s1, s2 = _row_sum(oracle, n, False) * 2 * np.pi / n, _row_sum(oracle, n, True) * 4 * np.pi ** 2 / n ** 2
            v = np.abs(z - 2 * np.pi * np.arange(n) / n).max()
            for name, ref, bound in (("Zp", zp, s1 * v + 1), ("Zpp", zpp, s2 * v)):
                err = np.abs(d[name][o:o + n] - ref).max()
                assert err <= 40 * eps * bound, (n, name, err, 40 * eps * bound)
            o += n
    assert np.abs(q[1] - q[0]).max() <= 1e-12 * (1 + np.abs(q[0]).max())

"""dc2_whiten on metrics whose spectrum is so dense at its low end that Lanczos does not separate
the smallest eigenvalue in its 256 steps: the metric is of whole rank all the same, and its factor
and its smallest eigenvalue (from the eigensolver then) are returned."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [200, 256, 700, 1100])
def test_dense_low_end(n):
    from dirac_caspt2_amd.api import Caspt2Context, whiten
    from gpu_helpers import say
    say("whiten, dense low end", n)
    rng = np.random.default_rng(n)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)))
    # 1 / w with the density of Chebyshev nodes: gaps of 1 / n^2 at both ends
    w = 1.0 / (0.75 + 0.25 * np.cos(np.pi * (np.arange(n) + 0.5) / n))
    S = (Q * w) @ Q.conj().T
    S = 0.5 * (S + S.conj().T)
    with Caspt2Context(0) as c:
        got = whiten(c, S, np.eye(n, dtype=complex), 0.5)
        assert got is not None, "a metric of whole rank was reported as rank-deficient"
        assert whiten(c, S, np.eye(n, dtype=complex), 1.5) is None
    linv, _, lam = got
    tol = 3 * n * 2.2e-16 * w.max()   # n eps |S| for the eigenvalue, |L^-1|^2 = 1 / low more for the factor
    assert abs(lam - w.min()) < tol
    assert np.abs(linv @ S @ linv.conj().T - np.eye(n)).max() < tol / w.min()

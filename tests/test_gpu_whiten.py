"""Metrics of whole rank by their Cholesky factor (dc2_whiten) against numpy, at sizes on both
sides of the 64-row blocks and of every merge of the inverse (odd block counts included).

Tolerances: the eigenvalues of S lie in [low, 3], so |L^-1|^2 <= 1 / low; the factorisation and
the products leave errors of n eps |S| |L^-1|^2 at most (n eps = 3e-13 at n = 1281)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from dirac_caspt2_amd.api import Caspt2Context
    with Caspt2Context(0) as c:
        yield c


def _problem(n, low, seed=0):
    rng = np.random.default_rng(seed + n)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)))
    w = np.geomspace(low, 3.0, n) if n > 1 else np.array([low])
    S = (Q * w) @ Q.conj().T
    B = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    return 0.5 * (S + S.conj().T), 0.5 * (B + B.conj().T) / np.sqrt(n)


@pytest.mark.parametrize("low", [1e-2, 1e-6])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 191, 200, 321, 449, 705, 1281])
def test_whiten(ctx, n, low):
    from dirac_caspt2_amd.api import whiten
    from gpu_helpers import say
    say("whiten", n, low)
    S, B = _problem(n, low)
    Li, bt, lam = whiten(ctx, S, B)
    assert np.abs(np.triu(Li, 1)).max() == 0.0
    tol = 3 * n * 2.2e-16 * 3.0 / low + 1e-14
    assert np.abs(Li @ S @ Li.conj().T - np.eye(n)).max() < tol
    assert np.abs(bt - Li @ B @ Li.conj().T).max() < tol
    assert np.abs(bt - bt.conj().T).max() == 0.0
    assert abs(lam - low) < 1e-9 * low + 3 * n * 2.2e-16 * 3.0


def test_thresholds(ctx):
    """An eigenvalue below sigma, a singular and a non-finite S are refused."""
    from dirac_caspt2_amd.api import whiten
    S, B = _problem(130, 1e-6)
    assert whiten(ctx, S, B, 0.999e-6) is not None
    assert whiten(ctx, S, B, 1.001e-6) is None
    X = S[:, :100]
    assert whiten(ctx, X @ X.conj().T, B) is None
    S[5, 5] = np.nan
    assert whiten(ctx, S, B) is None


def test_clustered_low_end(ctx):
    """The smallest eigenvalue of a metric whose lowest ones are close together and paired."""
    from dirac_caspt2_amd.api import whiten
    rng = np.random.default_rng(3)
    n = 640
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)))
    w = np.concatenate([np.repeat(np.linspace(7.3e-7, 9e-7, 20), 2), np.geomspace(1e-6, 2.0, n - 40)])
    S = (Q * w) @ Q.conj().T
    _, _, lam = whiten(ctx, 0.5 * (S + S.conj().T), np.eye(n, dtype=complex))
    assert abs(lam - 7.3e-7) < 1e-8 * 7.3e-7 + 3 * n * 2.2e-16 * 2.0

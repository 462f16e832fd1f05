"""Deflation in the tridiagonal divide and conquer by parallel tests and serial chains of rotations, and the
back-transformation with 16 lanes per eigenvector: spectra whose merges deflate every entry, none, single pairs and
long chains, at the sizes where the kernels change (leaves of 16, rows of 64, 128 and 256, chunks of 256 entries).

A backward-stable eigensolver leaves a residual and a loss of orthogonality of a modest multiple of n eps |A|; 20 n
eps is allowed, eps = 2^-53."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


@pytest.fixture(scope="module")
def ctx():
    from dirac_caspt2_amd.api import Caspt2Context
    c = Caspt2Context(0)
    yield c
    c.close()


def _matrix(kind, n, rng):
    if kind == "glued":       # Wilkinson blocks of 21, weakly coupled: chains of close pairs
        d = np.abs((np.arange(n) % 21) - 10.0)
        e = np.where(np.arange(1, n) % 21 == 0, 1e-13, 1.0)
        return (np.diag(d) + np.diag(e, 1) + np.diag(e, -1)).astype(complex)
    Q = np.linalg.qr(rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n)))[0]
    if kind == "clusters":    # a few values, each many times up to 1e-14
        w = rng.integers(1, 5, n) + 1e-14 * rng.normal(size=n)
    elif kind == "graded":
        w = 10.0 ** rng.uniform(-14, 0, n)
    else:                     # "identity": every entry deflates
        w = np.ones(n)
    A = (Q * w) @ Q.conj().T
    return (A + A.conj().T) / 2


@pytest.mark.parametrize("kind", ["glued", "clusters", "graded", "identity"])
@pytest.mark.parametrize("n", [17, 33, 64, 65, 128, 129, 255, 256, 257, 513, 1100])
def test_chains(ctx, n, kind):
    from dirac_caspt2_amd import api
    A = _matrix(kind, n, np.random.default_rng(n))
    w, V, _ = api.cdiag(ctx, A.copy(), 0.0)
    norm = np.linalg.norm(A, 2)
    assert np.all(np.diff(w) >= 0)
    assert np.linalg.norm(A @ V - V * w, 2) <= 20 * n * EPS * norm
    assert np.linalg.norm(V.conj().T @ V - np.eye(n), 2) <= 20 * n * EPS

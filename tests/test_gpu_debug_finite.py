"""DC2_DEBUG=1 stops at the first device array that holds a non-finite value: B~ of a metric that
goes by its Cholesky factor is one of them, as B~ of the eigenvector route is."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_b_tilde_of_the_cholesky_route(monkeypatch):
    from dirac_caspt2_amd.api import Caspt2Context, whiten
    monkeypatch.setenv("DC2_DEBUG", "1")
    S, B = np.diag(np.linspace(1.0, 2.0, 70)).astype(complex), np.eye(70, dtype=complex)
    with Caspt2Context(0) as c:
        assert whiten(c, S, B) is not None
        B[3, 5] = B[5, 3] = np.nan
        with pytest.raises(RuntimeError, match="non-finite value in B~"):
            whiten(c, S, B)

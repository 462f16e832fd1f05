"""Metrics of at most 256 rows (the one-workgroup Lanczos of dc2_whiten) while another context's
products of NaN operands run on the same compute units: what those leave in LDS must not reach a
result.  Sizes away from 256 rows, whose last rows meet the unrolled loop's tail."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [66, 91, 144, 196, 229])
def test_whiten_beside_nan(n):
    from dirac_caspt2_amd.api import Caspt2Context, DeviceArray, whiten, zgemm
    from gpu_helpers import say
    say("whiten beside NaN products", n)
    rng = np.random.default_rng(n)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)))
    S = (Q * np.geomspace(1e-3, 2.0, n)) @ Q.conj().T
    S = 0.5 * (S + S.conj().T)
    stop = threading.Event()
    M, N, K = 8192, 256, 64

    def poison():
        with Caspt2Context(0) as c:
            A, B, C = (DeviceArray(c, host=np.full(x, np.nan + 1j * np.nan)) for x in (M * K, N * K, M * N))
            while not stop.is_set():
                for _ in range(8):
                    zgemm(c, "N", "N", M, N, K, 1.0, A, M, 0, B, K, 0, 0.0, C, M, 0)
                c.synchronize()

    t = threading.Thread(target=poison)
    t.start()
    try:
        with Caspt2Context(0) as c:
            got = [whiten(c, S, np.eye(n, dtype=complex)) for _ in range(40)]
    finally:
        stop.set()
        t.join()
    refused = sum(g is None for g in got)
    assert refused == 0, f"{refused} of {len(got)} metrics of whole rank refused"
    # the eigenvalue's error: n eps |S|, and the square of a residual below 1e-7
    for g in got:
        assert abs(g[2] - 1e-3) < 1e-9 * 1e-3 + 3 * n * 2.2e-16 * 2.0

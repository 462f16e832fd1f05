"""The split-precision product at the edges of its tiles: 16-row blocks, 128 x 32 (up to 6 digits) and 64 x 32
workgroup tiles, K' chunks of 32 complex k, and the rows held in registers up to K = 128 and 384.

The digits and their INT32 sums are exact, so the product is known to the last bits of FP64: numpy forms the same
digits in int64 and recombines them, and both round S - 1 additions of FP64 (5e-16 of the largest level's value)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _split(Z, S):
    """Rows of complex Z: digits of re and im (S, rows, K) and the row exponents."""
    big = np.maximum(np.abs(Z.real), np.abs(Z.imag)).max(axis=1)
    e = np.where(big > 0, np.frexp(np.where(big > 0, big, 1.0))[1], 0)
    out = []
    for X in (Z.real, Z.imag):
        m = np.floor(np.ldexp(np.abs(X), (7 * S - e)[:, None])).astype(np.int64)
        out.append(np.stack([np.sign(X).astype(np.int64) * ((m >> (7 * (S - 1 - p))) & 127) for p in range(S)]))
    return out[0], out[1], e


@pytest.mark.parametrize("slices", [3, 6, 8])
@pytest.mark.parametrize("shape", [(1, 1, 1), (15, 31, 31), (17, 33, 33), (63, 5, 128), (65, 32, 129), (127, 64, 384),
                                   (129, 65, 385), (300, 17, 700)])
def test_digits_to_the_last_bits(slices, shape):
    from dirac_caspt2_amd.api import Caspt2Context, DeviceArray, zgemm_split
    M, N, K = shape
    S = slices
    rng = np.random.default_rng(M + 7 * N + 13 * K)
    A = (rng.normal(size=(M, K)) + 1j * rng.normal(size=(M, K))) * 10.0 ** rng.uniform(-3, 3, (M, 1))
    B = (rng.normal(size=(N, K)) + 1j * rng.normal(size=(N, K))) * 10.0 ** rng.uniform(-3, 3, (N, 1))
    A[M // 2] = 0.0
    Ar, Ai, ea = _split(A, S)
    for op in "NR":
        Br, Bi, eb = _split(np.conj(B) if op == "R" else B, S)
        re, im = np.zeros((M, N)), np.zeros((M, N))
        for L in range(S - 1, -1, -1):
            lr = sum(Ar[p] @ Br[L - p].T - Ai[p] @ Bi[L - p].T for p in range(L + 1))
            li = sum(Ar[p] @ Bi[L - p].T + Ai[p] @ Br[L - p].T for p in range(L + 1))
            re, im = re + np.ldexp(lr.astype(float), -7 * (L + 2)), im + np.ldexp(li.astype(float), -7 * (L + 2))
        ref = np.ldexp(re, ea[:, None] + eb) + 1j * np.ldexp(im, ea[:, None] + eb)
        with Caspt2Context(0) as ctx:
            dA = DeviceArray(ctx, np.ascontiguousarray(A))
            dB = DeviceArray(ctx, np.ascontiguousarray(B))
            dC = DeviceArray(ctx, np.zeros(M * N, dtype=np.complex128))
            zgemm_split(ctx, S, op, M, N, K, dA, K, dB, K, dC, M)
            out = dC.to_host().reshape((M, N), order="F")
        scale = 2.0 * K * np.ldexp(1.0, ea[:, None] + eb)    # the largest level is below K 2^(ea + eb) in each part
        assert np.all(np.abs(out - ref) <= S * 1.2e-16 * scale)

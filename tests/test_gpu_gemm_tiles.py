"""The matrix-core product at the edges of its tiles: rows around 64, columns around every
fragment count of 16 up to 64 and past it, K around the tiles of 8 and 16 and their groups of
four, every pair of operations, leading dimensions larger than the matrices, alpha and beta,
batches and split K, NaN and infinity outside the operands.

Tolerance: FP64 accumulation of K terms in any order, |error| <= 8 K eps max|a| max|b|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(64, 16, 16), (65, 17, 5), (63, 15, 4), (1, 1, 1), (130, 33, 9), (200, 48, 8), (64, 64, 17), (17, 65, 40),
          (300, 100, 23), (129, 31, 33), (70, 129, 300), (257, 7, 3), (16500, 33, 12), (16500, 70, 31), (66000, 65, 10),
          (2100, 2050, 20)]


@pytest.fixture(scope="module")
def ctx():
    from dirac_caspt2_amd.api import Caspt2Context
    with Caspt2Context(0) as c:
        yield c


def _run(ctx, oa, ob, M, N, K, pad, alpha, beta, rng, batch=1):
    from dirac_caspt2_amd.api import DeviceArray, zgemm

    def rand(*shape):
        return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)

    ra, ca = (M, K) if oa == "N" else (K, M)
    rb, cb = (K, N) if ob in "NR" else (N, K)
    A, B, C = (np.full((batch, c, r + pad), np.nan + 1j * np.inf) for r, c in ((ra, ca), (rb, cb), (M, N)))
    A[:, :, :ra], B[:, :, :rb], C[:, :, :M] = rand(batch, ca, ra), rand(batch, cb, rb), rand(batch, N, M)
    dA, dB, dC = (DeviceArray(ctx, host=x) for x in (A, B, C))
    zgemm(ctx, oa, ob, M, N, K, alpha, dA, ra + pad, ca * (ra + pad), dB, rb + pad, cb * (rb + pad), beta, dC, M + pad,
          N * (M + pad), batch)
    ctx.synchronize()
    got = dC.to_host().reshape(C.shape)
    a, b = A[:, :, :ra].transpose(0, 2, 1), B[:, :, :rb].transpose(0, 2, 1)
    a = {"N": a, "T": a.transpose(0, 2, 1), "C": a.transpose(0, 2, 1).conj()}[oa]
    b = {"N": b, "R": b.conj(), "T": b.transpose(0, 2, 1), "C": b.transpose(0, 2, 1).conj()}[ob]
    want = alpha * (a @ b) + beta * C[:, :, :M].transpose(0, 2, 1)
    tol = 8 * (K + 2) * 1.2e-16 * (np.abs(a).max() * np.abs(b).max() + 4.0) * max(1.0, abs(alpha))
    assert np.abs(got[:, :, :M].transpose(0, 2, 1) - want).max() < tol
    if pad:
        assert np.isnan(got[:, :, M:].real).all()   # nothing is written past the rows


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("ops", ["NN", "NR", "NT", "NC", "TN", "TR", "TT", "TC", "CN", "CR", "CT", "CC"])
def test_tiles(ctx, ops, shape):
    from gpu_helpers import say
    if shape[0] * shape[1] > 3e6 and ops not in ("TR", "NC"):
        pytest.skip("the largest shapes with one pair of each kind")
    say("gemm tiles", ops, shape)
    rng = np.random.default_rng(sum(shape))
    _run(ctx, ops[0], ops[1], *shape, 3, 0.7 - 0.2j, 0.3 + 0.1j, rng)
    _run(ctx, ops[0], ops[1], *shape, 0, 1.0 + 0.0j, 0.0j, rng, batch=2)

"""Products whose operands have leading dimensions around 2^22, from where the matrix-core kernel
takes 64-bit offsets within a tile (63 columns of 2^22 complex numbers are 4.2e9 bytes): the last
size below it, itself and one past it, for every variant and each operand, and the Hermitian product.

Tolerance: FP64 accumulation of K terms in any order, |error| <= 8 K eps max|a| max|b|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _far(ctx, a, ld):
    """The matrix a with leading dimension ld on the device; nothing but a itself is written."""
    from dirac_caspt2_amd.api import DeviceArray, check
    buf = DeviceArray(ctx, nbytes=16 * (ld * (a.shape[1] - 1) + a.shape[0]))
    for j in range(a.shape[1]):
        col = np.ascontiguousarray(a[:, j])
        check("dc2_memcpy", ctx.lib.dc2_memcpy(ctx.h, buf.ptr + 16 * ld * j, col.ctypes.data, col.nbytes, 1))
    return buf


@pytest.fixture(scope="module")
def ctx():
    from dirac_caspt2_amd.api import Caspt2Context
    with Caspt2Context(0) as c:
        yield c


def _rand(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def _op(a, op):
    return {"N": a, "R": a.conj(), "T": a.T, "C": a.conj().T}[op]


@pytest.mark.parametrize("ld", [(1 << 22) - 1, 1 << 22, (1 << 22) + 1])
@pytest.mark.parametrize("ops,far", [("TN", "A"), ("CR", "A"), ("NT", "A"), ("NN", "B"), ("TR", "B"), ("NC", "B")])
def test_far_operand(ctx, ops, far, ld):
    from dirac_caspt2_amd.api import DeviceArray, gemm_clear_choices, gemm_set_choice, zgemm
    from gpu_helpers import say
    say("far operand", ops, far, ld)
    rng = np.random.default_rng(ld + ord(ops[0]) + ord(ops[1]))
    M, N, K = 65, 66, 21
    A = _rand(rng, M, K) if ops[0] == "N" else _rand(rng, K, M)
    B = _rand(rng, K, N) if ops[1] in "NR" else _rand(rng, N, K)
    want = _op(A, ops[0]) @ _op(B, ops[1])
    lda, ldb = (ld, B.shape[0]) if far == "A" else (A.shape[0], ld)
    dA = _far(ctx, A, ld) if far == "A" else DeviceArray(ctx, host=A.T)
    dB = _far(ctx, B, ld) if far == "B" else DeviceArray(ctx, host=B.T)
    dC = DeviceArray(ctx, nbytes=16 * M * N)
    try:
        for variant in (1, 2, 3, 4):
            gemm_set_choice(ops[0], ops[1], M, N, K, 1, variant, 1)
            zgemm(ctx, ops[0], ops[1], M, N, K, 1.0, dA, lda, 0, dB, ldb, 0, 0.0, dC, M, 0)
            ctx.synchronize()
            got = dC.to_host().reshape(N, M).T
            assert np.abs(got - want).max() < 8 * K * 1.2e-16 * np.abs(A).max() * np.abs(B).max(), variant
    finally:
        gemm_clear_choices()


@pytest.mark.parametrize("ld", [(1 << 22) - 1, 1 << 22])
@pytest.mark.parametrize("split", [0, 2])
def test_far_hermitian(ctx, ld, split):
    from dirac_caspt2_amd.api import DeviceArray, zherk
    from gpu_helpers import say
    say("far Hermitian product", ld, split)
    rng = np.random.default_rng(ld)
    m, k = 130, 37
    A = _rand(rng, m, k)
    dA, dC = _far(ctx, A, ld), DeviceArray(ctx, nbytes=16 * m * m)
    zherk(ctx, m, k, dA, ld, dC, m, split)
    ctx.synchronize()
    got = dC.to_host().reshape(m, m).T
    assert np.abs(got - A @ A.conj().T).max() < 8 * k * 1.2e-16 * np.abs(A).max() ** 2

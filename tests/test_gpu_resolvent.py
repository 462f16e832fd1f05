"""The A and C resolvents by conjugate gradients (dc2_resolvent_energy and the CASPT2 route
that uses it) against dense solves and against the eigendecomposition route.

Tolerance: a column stops at a relative residual of 1e-14, and the condition number of the
matrices here is at most 60, so u_k is within 60 * 1e-14 of the exact one plus the rounding of
its n-term sums: 1e-11 of the value holds with room.  The two routes of a whole energy differ
by the rounding of their own S^-1/2 V, which is common to both: 1e-11 Eh."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from dirac_caspt2_amd.api import Caspt2Context
    with Caspt2Context(0) as c:
        yield c


def _problem(n, npert, low, seed=0):
    rng = np.random.default_rng(seed + 7 * n + npert)
    X = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    Q, _ = np.linalg.qr(X)
    w = np.linspace(low, 6.0, n) if n > 1 else np.array([low])
    B = (Q * w) @ Q.conj().T
    y = rng.standard_normal((n, npert)) + 1j * rng.standard_normal((n, npert))
    alpha = np.sort(rng.uniform(0.1, 20.0, npert))
    return 0.5 * (B + B.conj().T), y, alpha


@pytest.mark.parametrize("n,npert", [(1, 1), (33, 3), (255, 40), (256, 1), (257, 17), (512, 5), (513, 64), (1024, 2),
                                     (1025, 9), (1280, 30), (1281, 70), (2048, 3)])
def test_resolvent_energy(ctx, n, npert):
    from dirac_caspt2_amd.api import resolvent_energy
    from gpu_helpers import say
    say("resolvent", n, npert)
    B, y, alpha = _problem(n, npert, 0.0)
    u = np.stack([np.linalg.solve(B + a * np.eye(n), y[:, k]) for k, a in enumerate(alpha)], axis=1)
    e, s, it = resolvent_energy(ctx, B, y, alpha)
    assert abs(e + np.vdot(y, u).real) < 1e-11 * abs(np.vdot(y, u))
    assert abs(s - np.vdot(u, u).real) < 1e-11 * np.vdot(u, u).real


def test_zero_columns_and_refusals(ctx):
    """Zero columns cost nothing; an indefinite matrix and non-finite inputs are refused."""
    from dirac_caspt2_amd.api import resolvent_energy
    B, y, alpha = _problem(70, 5, 0.0)
    y[:, 1:4] = 0.0
    u = np.stack([np.linalg.solve(B + a * np.eye(70), y[:, k]) for k, a in enumerate(alpha)], axis=1)
    e, s, _ = resolvent_energy(ctx, B, y, alpha)
    assert abs(e + np.vdot(y, u).real) < 1e-11 * abs(np.vdot(y, u))
    assert resolvent_energy(ctx, B, y * 0.0, alpha)[:2] == (0.0, 0.0)
    assert resolvent_energy(ctx, B - 3.0 * np.eye(70), y, np.zeros(5)) is None
    y[3, 0] = np.inf
    assert resolvent_energy(ctx, B, y, alpha) is None
    y[3, 0] = np.nan
    assert resolvent_energy(ctx, B, y, alpha) is None


@pytest.mark.parametrize("metric", ["formula", "antisymmetric_det"])
@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("eshift", [0.0, 0.3, -1.0])
def test_energy_against_eigenvectors(metric, lanes, eshift):
    """eshift -1.0 makes resolvents indefinite: the route falls back to the eigenvectors."""
    from dirac_caspt2_amd import synth
    from gpu_helpers import context_from_synth, say
    say("resolvent route", metric, lanes, eshift)
    sp = synth.generate(synth.CONFIG_SMALL)
    with context_from_synth(sp) as c:
        c.set_option("ac_metric", metric)
        c.set_option("lanes", lanes)
        c.set_option("schur", "off")
        c.casci(1)
        a = c.caspt2(1, eshift)
        c.set_option("eigensolver", "native")
        b = c.caspt2(1, eshift)
    for X in "ABCDEFGH":
        scale = max(1.0, abs(b.e2[X]), abs(b.sumc2[X]))
        assert abs(a.e2[X] - b.e2[X]) < 1e-11 * scale, X
        assert abs(a.sumc2[X] - b.sumc2[X]) < 1e-11 * scale, X
    assert a.info == b.info


def test_thin_c_with_more_strings_than_rows():
    """14 spinors with 7 electrons: C(14, 6) = 3003 strings against 14^3 = 2744 formula rows and
    1274 of the thin factor.  The two metrics weight the weakest directions differently by
    rounding (eps / 1e-8 of them): the 1e-9 Eh of the oracle comparisons."""
    from dirac_caspt2_amd import synth
    from gpu_helpers import context_from_synth, say
    say("thin C, 14 spinors with 7 electrons")
    sp = synth.generate(synth.SynthSpec(ninact=4, nact=14, nsec=20, nelec=7, seed=20300))
    out = []
    for metric in ("auto", "formula"):
        with context_from_synth(sp) as c:
            c.set_option("ac_metric", metric)
            c.casci(2)
            out.append(c.caspt2(1, 0.0))
    a, b = out
    for X in "ABCDEFGH":
        assert abs(a.e2[X] - b.e2[X]) < 1e-9, X
        assert abs(a.sumc2[X] - b.sumc2[X]) < 1e-9, X
    assert a.info == b.info

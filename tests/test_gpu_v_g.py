"""The right-hand side of subspace G in 16 x 16 tiles of secondary pairs, 8 or 16 active spinors at a time, against the
oracle's G energy: secondary counts at and beside multiples of 16, one and several passes over the active spinors.

Both sides take the same CASCI root, converged to a residual of 1e-11; 1e-9 Eh is the bound of every energy
comparison of this suite."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nact,nelec,nsec", [(6, 2, 2), (6, 2, 14), (8, 4, 16), (8, 4, 18), (10, 4, 34), (16, 2, 30),
                                             (18, 2, 40)])
def test_g_energy(nact, nelec, nsec):
    from dirac_caspt2_amd import synth
    from gpu_helpers import context_from_synth, oracle_problem
    from oracle import caspt2_ref as R
    sp = synth.generate(synth.SynthSpec(4, nact, nsec, nelec, seed=7 * nact + nsec))
    ref = R.run_caspt2(oracle_problem(sp), subspaces=["G"])
    with context_from_synth(sp) as ctx:
        ctx.casci(sp.spec.selectroot)
        out = ctx.caspt2(sp.spec.selectroot, sp.spec.eshift)
    assert abs(out.e2["G"] - ref.e2["G"]) < 1e-9
    assert abs(out.sumc2["G"] - ref.sumc2["G"]) < 1e-9

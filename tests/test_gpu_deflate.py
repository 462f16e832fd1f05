"""The determinant-space metrics of A and C without their eigendecomposition (whole rank by the
Cholesky factor, a few cut directions by subspace iteration) against the eigendecomposition
route: 8, 10 and 12 active spinors (56, 210 and 792 strings; the last has eigenvalues on both
sides of the threshold), ground and excited roots, level shifts, one lane and four.

Tolerance: the two routes weight directions of eigenvalue w by rounding eps |G| / w relative to
their own size, at most 1e-16 * 5 / 1e-8 = 5e-8 for the weakest retained one, which carries
about one part in 1e3 of E2: the 1e-9 Eh of the oracle comparisons (sumc2 relative to its own
size, which an excited root can take above 1)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [1, 2])
@pytest.mark.parametrize("dims", [(4, 8, 20, 4), (4, 10, 22, 5), (6, 12, 26, 6)])
def test_against_eigenvectors(dims, seed):
    from dirac_caspt2_amd import synth
    from gpu_helpers import context_from_synth, say
    say("deflated metrics", dims, seed)
    sp = synth.generate(synth.SynthSpec(*dims, seed=seed))
    with context_from_synth(sp) as c:
        for lanes, root, eshift in ((4, 1, 0.0), (1, 1, 0.0), (4, 3, 0.4)):
            c.set_option("lanes", lanes)
            c.casci(4)
            c.set_option("eigensolver", "auto")
            a = c.caspt2(root, eshift)
            c.set_option("eigensolver", "native")
            b = c.caspt2(root, eshift)
            for X in "ABCDEFGH":
                assert abs(a.e2[X] - b.e2[X]) < 1e-9 * max(1.0, abs(b.e2[X])), (X, lanes, root)
                assert abs(a.sumc2[X] - b.sumc2[X]) < 1e-9 * max(1.0, abs(b.sumc2[X])), (X, lanes, root)
            assert a.info == b.info
            for X in "AC":   # the distance to the threshold, to the rounding of the eigenvalues
                assert abs(a.margin[X] - b.margin[X]) < 1e-13, (X, lanes, root)

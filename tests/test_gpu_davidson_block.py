"""The block Davidson's step for a block of four: subspaces from the smallest (a restart in every
step) past the largest that one workgroup's coefficients take (60 vectors), sizes that are and are
not multiples of the kernels' 64 and 256 rows, and a space so small that blocks shrink.

Against the dense solver of the same context.  A residual of 1e-11 leaves an error of its square
over the gap in the energy and of itself over the gap in the vector: with gaps above 0.01 Eh here,
1e-10 Eh is a safe bound for the energies and 1e-9 for what is linear in the vector."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nact,nelec", [(6, 2), (8, 4), (10, 4), (10, 5), (12, 6)])
@pytest.mark.parametrize("maxsub", [0, 8, 11, 60, 64])
def test_block_of_four(nact, nelec, maxsub):
    from dirac_caspt2_amd import synth
    from dirac_caspt2_amd.api import Caspt2Context
    from dirac_caspt2_amd.problem import load_factors
    spec = synth.SynthSpec(4, nact, 10, nelec, seed=100 + nact)
    sp = synth.generate(spec)
    got = {}
    with Caspt2Context(0) as ctx:
        load_factors(ctx, (spec.ninact, spec.nact, spec.nsec, spec.nelec), sp.h, sp.B, sp.ecore, on_device=True)
        ctx.set_option("davidson_maxsub", maxsub)
        for solver in ("dense", "davidson", "davidson"):
            ctx.set_option("casci_solver", solver)
            e = ctx.casci(1)[0]
            assert (ctx.casci_info()[2] > 0) == (solver == "davidson")
            # an odd count's lowest state is one of a pair, refused with one root
            r = ctx.caspt2(1, 0.0) if nelec % 2 == 0 else None
            if solver == "davidson":
                assert abs(e - got["dense"][0]) < 1e-10
                for name in r.e2 if r else ():
                    assert abs(r.e2[name] - got["dense"][1].e2[name]) < 1e-9, name
                    assert abs(r.sumc2[name] - got["dense"][1].sumc2[name]) < 1e-9, name
            got[solver] = (e, r)

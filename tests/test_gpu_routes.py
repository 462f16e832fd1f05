"""Which way each subspace goes (dc2_get_routes), so that a comparison of two routes compares two:
metrics of whole rank, metrics with a few and with many cut directions, resolvents that are not
positive definite, a chosen eigensolver.  Energies against the eigenvector routes of the same
context.

Tolerance: as in the comparisons of these routes (1e-9, weak directions weighted by rounding
1e-16 |G| / 1e-8); 1e-11 relative for an energy whose metrics both routes treat alike."""
import pytest

pytestmark = pytest.mark.gpu


def _both(dims, seed, amplitude=0.25, eshift=0.0, options=()):
    from dirac_caspt2_amd import synth
    from gpu_helpers import context_from_synth, say
    say("routes", dims, seed, amplitude, eshift, options)
    sp = synth.generate(synth.SynthSpec(*dims, seed=seed), amplitude=amplitude)
    with context_from_synth(sp) as c:
        for k, v in options:
            c.set_option(k, v)
        c.casci(1 + dims[3] % 2)
        a = c.caspt2(1, eshift)
        routes = c.routes()
        c.set_option("eigensolver", "native")
        b = c.caspt2(1, eshift)
        for X in "ABCDEFG":
            assert not c.routes()[X] & {"whole_rank", "deflated", "cg", "refused"}, X
    assert a.info == b.info
    for X in "ABCDEFGH":
        assert abs(a.e2[X] - b.e2[X]) < 1e-9 * max(1.0, abs(b.e2[X])), X
        assert abs(a.sumc2[X] - b.sumc2[X]) < 1e-9 * max(1.0, abs(b.sumc2[X])), X
    return routes, a.info


@pytest.mark.parametrize("lanes", [1, 4])
def test_whole_rank(lanes):
    routes, info = _both((4, 10, 22, 4), 3, options=(("lanes", lanes),))
    assert info["C"][1] == 120 and routes["C"] == {"whole_rank", "compressed"}
    for X in "BF":
        assert routes[X] == {"whole_rank", "b_vectors"}, X
    assert routes["D"] == {"whole_rank", "b_vectors"}
    assert routes["E"] == routes["G"] == {"vectors", "b_vectors"} and routes["H"] == set()


@pytest.mark.parametrize("lanes", [1, 2, 4])
def test_a_few_directions_cut(lanes):
    routes, info = _both((6, 12, 26, 6), 1, options=(("lanes", lanes),))
    for X in "AC":
        assert 0 < 792 - info[X][1] <= 32
        assert routes[X] == {"deflated", "compressed"}, X


@pytest.mark.parametrize("lanes", [1, 2, 4])
@pytest.mark.parametrize("dims,amplitude", [((6, 12, 26, 6), 0.04), ((4, 10, 22, 5), 0.04), ((4, 8, 20, 4), 0.04)])
def test_many_directions_cut(dims, amplitude, lanes):
    """A weakly correlated state: the factor routes are tried and the metrics diagonalised."""
    routes, info = _both(dims, 1, amplitude, options=(("lanes", lanes),))
    for X in "AC":
        assert {"vectors", "refused"} <= routes[X] and not routes[X] & {"whole_rank", "deflated"}, X
        assert routes[X] & {"cg", "compressed"}, X


def test_thin_factor_and_antisymmetric_reduction():
    routes, info = _both((4, 14, 20, 6), 2)
    assert info["A"][1] == info["C"][1] == 1274
    assert routes["A"] == routes["C"] == {"whole_rank", "cg"}
    routes, info = _both((4, 14, 20, 6), 2, 0.04)
    assert info["A"][1] < 1274 and info["C"][1] < 1274
    assert routes["A"] == routes["C"] == {"vectors", "cg", "refused"}


@pytest.mark.parametrize("metric", ["formula", "antisymmetric_det"])
def test_indefinite_resolvents(metric):
    """A shift that makes some B~ + alpha indefinite: conjugate gradients are refused."""
    options = (("ac_metric", metric), ("schur", "off"))
    routes, _ = _both((4, 8, 40, 4), 20240, options=options)
    assert "cg" in routes["A"] and "cg" in routes["C"]
    routes, _ = _both((4, 8, 40, 4), 20240, eshift=-1.0, options=options)
    assert any({"refused", "b_vectors"} <= routes[X] for X in "AC")

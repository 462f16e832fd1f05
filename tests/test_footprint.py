"""The admission estimate of a request (dc2_request_footprint): budgets that admitted a request go
on admitting it, and a slot holds no more than its request's estimate."""
import ctypes

import pytest

ADMITTED = {(4, 8, 40, 4): 212147584, (18, 10, 210, 5): 2107652096, (12, 12, 132, 6): 2046920192,
            (16, 12, 164, 6): 2581845504, (10, 14, 100, 4): 4101295200, (30, 14, 280, 6): 15309354336,
            (10, 14, 100, 7): 8766360576, (2, 16, 20, 4): 10790872576}


@pytest.mark.parametrize("dims", sorted(ADMITTED))
def test_budgets_keep_admitting(dims):
    from dirac_caspt2_amd.api import request_footprint
    assert request_footprint(*dims) <= ADMITTED[dims]


@pytest.mark.gpu
@pytest.mark.parametrize("amplitude", [0.25, 0.04])
@pytest.mark.parametrize("dims", [(12, 12, 20, 6), (4, 14, 20, 6), (18, 10, 60, 4)])
def test_slot_holds_no_more(dims, amplitude):
    """amplitude 0.04: the metrics of A and C are factorised first and diagonalised then."""
    from dirac_caspt2_amd import synth
    from dirac_caspt2_amd.api import Server, request_footprint
    from gpu_helpers import say
    sp = synth.generate(synth.SynthSpec(*dims, seed=4), amplitude=amplitude)
    with Server(0, nslots=1, lanes_per_slot=1) as srv:
        mol = srv.add_molecule(dims, sp.B)
        with open("/proc/self/maps") as f:   # the HIP runtime that the library runs on
            hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))

        def free():
            a, b = ctypes.c_size_t(), ctypes.c_size_t()
            assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
            return a.value

        before = free()
        srv.submit(mol, sp.h, sp.ecore)
        r = srv.wait(60.0)
        assert r is not None and r.status == 0
        held = before - free()
    say("slot", dims, amplitude, "held", held, "footprint", request_footprint(*dims))
    assert held < request_footprint(*dims)

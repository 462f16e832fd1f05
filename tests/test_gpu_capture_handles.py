"""Graph captures of the Davidson beside other threads' work on the null stream, which HIP refuses
while any thread captures and which breaks the capture: contexts being made and closed (a rocBLAS
handle each; the library keeps those and its captures apart, so neither side may fail), and a
program's own synchronisations (a broken capture must only cost the context its graphs).  Every
energy must come out, the same one."""
import threading

import pytest

pytestmark = pytest.mark.gpu


def _energies(rounds, work):
    """The CASCI energies and the graphs' states of fresh contexts while a thread repeats work()."""
    from dirac_caspt2_amd import synth
    from dirac_caspt2_amd.api import Caspt2Context
    from dirac_caspt2_amd.problem import load_factors
    sp = synth.generate(synth.SynthSpec(4, 10, 10, 4, seed=5))
    stop, out = threading.Event(), []

    def loop():
        while not stop.is_set():
            work()

    t = threading.Thread(target=loop)
    t.start()
    try:
        for _ in range(rounds):   # a fresh context captures the graphs of its first Davidson run
            with Caspt2Context(0) as c:
                load_factors(c, (4, 10, 10, 4), sp.h, sp.B, sp.ecore)
                c.set_option("casci_solver", "davidson")
                out.append((c.casci(1)[0], c.graph_stats()))
    finally:
        stop.set()
        t.join()
    assert len({e for e, _ in out}) == 1
    return [s for _, s in out]


def test_contexts_beside_captures():
    from dirac_caspt2_amd.api import Caspt2Context
    from gpu_helpers import say
    say("contexts beside graph captures")
    errors = []

    def work():
        try:
            Caspt2Context(0).close()
        except RuntimeError as e:   # reported by the main thread
            errors.append(e)

    stats = _energies(24, work)
    assert not errors, errors
    assert all(s["enabled"] == 1 and s["captures"] > 0 for s in stats)


def test_null_stream_beside_captures():
    import ctypes
    from dirac_caspt2_amd import _lib
    from gpu_helpers import say
    say("null stream beside graph captures")
    _lib.lib()
    with open("/proc/self/maps") as f:   # the HIP runtime that the library runs on
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    # a refusal while a capture runs is this thread's own affair: the status is dropped
    stats = _energies(24, hip.hipDeviceSynchronize)
    say("contexts whose captures were broken:", sum(s["enabled"] == 0 for s in stats))
    assert hip.hipDeviceSynchronize() == 0   # nothing is left behind

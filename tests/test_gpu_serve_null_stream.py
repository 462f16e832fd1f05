"""A program's own work on the null stream while a request server runs: HIP refuses it during a
graph capture, so the server's slots issue their launches directly.  Every synchronisation of the
program and every request must succeed, and graphs can still be asked for."""
import ctypes
import threading

import pytest

pytestmark = pytest.mark.gpu


def _served(server, sp, count):
    s = sp.spec
    mol = server.add_molecule((s.ninact, s.nact, s.nsec, s.nelec), sp.B)
    for _ in range(count):
        server.submit(mol, sp.h, sp.ecore)
    got = [server.wait(60.0) for _ in range(count)]
    assert all(r is not None and r.status == 0 for r in got), [r and r.error for r in got]
    return {r.total for r in got}


def test_null_stream_beside_server():
    from dirac_caspt2_amd import _lib, synth
    from dirac_caspt2_amd.api import Server
    from gpu_helpers import say
    say("null stream beside a request server")
    sp = synth.generate(synth.SynthSpec(4, 12, 24, 6, seed=31))   # 924 determinants: the Davidson path
    _lib.lib()
    with open("/proc/self/maps") as f:   # the HIP runtime that the library runs on
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    stop, refused = threading.Event(), []

    def work():
        while not stop.is_set():
            status = hip.hipDeviceSynchronize()
            if status:
                refused.append(status)

    with Server(0, nslots=4, lanes_per_slot=1) as server:
        t = threading.Thread(target=work)
        t.start()
        try:
            plain = _served(server, sp, 8)
        finally:
            stop.set()
            t.join()
    assert not refused, refused
    with Server(0, nslots=2, lanes_per_slot=1) as server:
        server.set_option("graphs", 1)
        replayed = _served(server, sp, 4)
    assert max(plain | replayed) - min(plain | replayed) < 1e-12

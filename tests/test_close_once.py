"""close() and free() call the library once, also when what follows the call fails, as it does at the
interpreter's exit with the module's names already gone: a program that ended with a context open
destroyed it twice, in its own __del__ and in the context's (CPU: the library is a stand-in)."""
import pytest


class _Lib:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *a: self.calls.append((name, a)) or 0


@pytest.fixture
def api(monkeypatch):
    from dirac_caspt2_amd import api
    monkeypatch.setattr(api, "check", None)
    return api


@pytest.mark.parametrize("kind", ["Caspt2Context", "Server"])
def test_close(api, kind):
    obj = object.__new__(getattr(api, kind))
    obj.lib, obj.h, obj._keep = _Lib(), 7, {}
    with pytest.raises(TypeError):
        obj.close()
    obj.close()
    assert len(obj.lib.calls) == 1


def test_free(api):
    ctx = object.__new__(api.Caspt2Context)
    ctx.lib, ctx.h, ctx._keep = _Lib(), 7, {}
    buf = object.__new__(api.DeviceArray)
    buf.ctx, buf.ptr, buf.nbytes = ctx, 4096, 16
    with pytest.raises(TypeError):
        buf.free()
    buf.free()
    assert [c[0] for c in ctx.lib.calls] == ["dc2_free"]
    ctx.h = None

"""The worker's record of the device memory it handed out (CPU: the library is a stand-in)."""

import pytest

from pypto_amd import _lib
from pypto_amd.runtime import ChipWorker


class _Library:
    """Hands out one address; `during_free` runs where another thread could, after the release and before the call returns."""

    during_free = None
    status = _lib.OK

    def pto_hip_malloc(self, nbytes, out):
        out._obj.value = 0x1000
        return _lib.OK

    def pto_hip_free(self, ptr):
        if self.during_free:
            self.during_free()
        return self.status


def _worker(lib):
    w = ChipWorker.__new__(ChipWorker)
    w._lib, w._owned = lib, {}
    w._require_ready = lambda what: None
    return w


def test_an_address_given_out_again_while_it_is_being_freed_stays_the_new_owners():
    lib = _Library()
    w = _worker(lib)
    ptr = w.malloc(16)
    lib.during_free = lambda: w.malloc(32)
    w.free(ptr)
    lib.during_free = None
    assert w._owned == {ptr: 32}
    w.free(ptr)
    with pytest.raises(ValueError, match="not allocated by this worker"):
        w.free(ptr)


def test_a_failed_free_keeps_the_entry(monkeypatch):
    lib = _Library()
    w = _worker(lib)
    ptr = w.malloc(16)
    lib.status = _lib.ERR_RUNTIME
    monkeypatch.setattr(_lib, "check", lambda status: (_ for _ in ()).throw(RuntimeError("free failed")) if status else None)
    with pytest.raises(RuntimeError, match="free failed"):
        w.free(ptr)
    assert w._owned == {ptr: 16}

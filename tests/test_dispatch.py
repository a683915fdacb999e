"""The native argument side of a program call against the general path's descriptors (CPU: pto_hip_run is a callback)."""

import ctypes as C
import subprocess
import sys

import numpy as np
import pytest
import torch

from pypto_amd import _lib, build, runtime

_RUN = C.CFUNCTYPE(C.c_int, C.c_int, C.POINTER(_lib.ChipTensor), C.c_int, C.POINTER(C.c_uint64), C.c_int, C.c_void_p)


class _Recorder:
    def __init__(self, status=0):
        self.calls, self.status = [], status
        self.fn = _RUN(self._run)

    def _run(self, cid, tensors, n_t, scalars, n_s, stream):
        self.calls.append((cid, [bytes(tensors[i]) for i in range(n_t)], [scalars[i] for i in range(n_s)], stream))
        return self.status

    def __call__(self, args, *, cid=3, flags=None, optional=0, n_scalars=0, stream=0):
        flags = b"\1" * (len(args) - n_scalars) if flags is None else flags
        return _lib.dispatch().run(C.cast(self.fn, C.c_void_p).value, cid, flags, optional, n_scalars, tuple(args), stream)


def _general(t):
    return bytes(runtime._descriptor(t.data_ptr(), tuple(t.shape), t.dtype, t.numel() * t.element_size()))


@pytest.mark.parametrize("dtype", list(runtime._DTYPE_CODES))
@pytest.mark.parametrize("shape", [(), (7,), (0, 4), (3, 5), (2, 3, 4), (2, 1, 2, 1, 2), (1, 6)])
def test_descriptors_are_those_of_the_general_path(dtype, shape):
    r = _Recorder()
    a, b = torch.zeros(shape).to(dtype), torch.zeros((4,) + shape[:4]).to(dtype)[1:]  # the second starts inside its storage
    assert r([a, b, torch.nn.Parameter(a, requires_grad=False)], cid=11, stream=77) == 0
    cid, tensors, scalars, stream = r.calls[0]
    assert (cid, scalars, stream) == (11, [], 77) and tensors == [_general(a), _general(b), _general(a)]


def test_scalars_travel_as_the_general_path_sends_them():
    r = _Recorder(status=5)
    values = [0, 5, -1, 2 ** 63, True, 1.5, -0.0, 1e-45, float("inf"), np.float64(2.25)]
    assert r([torch.zeros(2)] + values, n_scalars=len(values), stream=None) == 5
    assert r.calls[0][2] == [runtime.scalar_to_uint64(v) for v in values]


class _Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("args,kw", [
    ([torch.zeros(4, 4).t()], {}), ([torch.zeros(4, 4)[:, :2]], {}), ([torch.zeros(1, 1, 1, 1, 1, 1)], {}),
    ([torch.zeros(2, dtype=torch.float64)], {}), ([torch.zeros(2, dtype=torch.bool)], {}), ([torch.zeros(2, device="meta")], {}),
    ([torch.zeros(2).as_subclass(_Sub)], {}), ([torch.zeros(2).to_sparse()], {}), ([[1.0, 2.0]], {}), ([None], {}),
    ([runtime.DeviceTensor(4096, (2,), torch.float32)], {}), ([torch.zeros(2)], {"flags": b"\0"}),
    ([torch.zeros(2)], {"flags": b"\1\1"}), ([torch.zeros(2)] * 3, {"flags": b"\1\1"}), ([torch.zeros(2)] * 65, {}),
    ([torch.zeros(2), "x"], {"n_scalars": 1}), ([torch.zeros(2), np.int64(1)], {"n_scalars": 1}),
    ([torch.zeros(2), 1e39], {"n_scalars": 1}), ([torch.zeros(2)], {"stream": "0"})])
def test_everything_else_is_handed_back_without_a_launch(args, kw):
    r = _Recorder()
    assert r(args, **kw) is None and r.calls == []


def test_optional_tensors_may_be_left_out():
    r = _Recorder()
    t = torch.zeros(2)
    assert r([t, t], flags=b"\1" * 4, optional=2) == 0 and len(r.calls[0][1]) == 2
    assert r([t], flags=b"\1" * 4, optional=2) is None


def test_a_tensor_of_a_transform_is_handed_back():
    r = _Recorder()
    seen = []

    def f(x):
        seen.append(r([x]))
        return x

    torch.vmap(f)(torch.zeros(3, 4))
    assert seen == [None] and r.calls == []


def test_the_binary_is_named_after_the_torch_it_reads(monkeypatch):
    """Another torch's objects are never read through it, and a build for another torch never passes for up to date."""
    here = _lib.dispatch_path()
    assert here.exists() and torch.__version__ in here.name
    monkeypatch.setattr(torch, "__version__", "0.0.0")
    monkeypatch.setattr(_lib, "_dispatch", None)
    assert _lib.dispatch_path() != here
    with pytest.warns(RuntimeWarning):
        assert _lib.dispatch() is None


class _Library:
    """Stands for the C library of a worker: counts the ids it hands out."""

    def __init__(self):
        self.registered = 0

    def pto_hip_register(self, name, out):
        self.registered += 1
        return 0


def _worker():
    w = runtime.ChipWorker.__new__(runtime.ChipWorker)
    w._lib, w._initialized, w._handles, w._owned = _Library(), True, [], {}
    return w


def test_programs_are_called_without_the_binary(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_dispatch", None)
    monkeypatch.setattr(_lib, "dispatch_path", lambda: tmp_path / "absent.so")
    monkeypatch.setattr(_lib, "run_address", lambda: 0)
    w = _worker()
    seen = []
    w._dispatch = lambda cid, program, args, stream: seen.append((program, args, stream))
    with pytest.warns(RuntimeWarning):
        h = w.register(runtime.rms_norm)
    t = torch.zeros(2)
    h(t, t, t, 1e-5, stream=3)
    assert seen == [(runtime.rms_norm, (t, t, t, 1e-5), 3)]


def test_a_binary_that_does_not_load_leaves_no_program_registered(monkeypatch, tmp_path):
    broken = tmp_path / "broken.so"
    broken.write_bytes(b"no library")
    monkeypatch.setattr(_lib, "_dispatch", None)
    monkeypatch.setattr(_lib, "dispatch_path", lambda: broken)
    w = _worker()
    with pytest.raises(ImportError):
        w.register(runtime.rms_norm)
    assert w._lib.registered == 0 and w._handles == []


def test_the_library_is_linked_before_and_without_torch(monkeypatch, tmp_path, capsys):
    order = []

    def link(cmd, **kw):
        order.append("link")
        (tmp_path / "libpto_hip.so").write_bytes(b"")
        return subprocess.CompletedProcess(cmd, 0, "", "")

    def extension(force):
        order.append("extension")
        raise RuntimeError("no headers")

    monkeypatch.setattr(build, "OBJ_DIR", tmp_path)
    monkeypatch.setattr(build, "LIB_PATH", tmp_path / "libpto_hip.so")
    monkeypatch.setattr(build, "sources", lambda: [tmp_path / "a.hip"])
    monkeypatch.setattr(build, "_compile", lambda src, force: src)
    monkeypatch.setattr(build.subprocess, "run", link)
    monkeypatch.setattr(build, "_build_dispatch", extension)
    with pytest.raises(RuntimeError, match="no headers"):
        build.build(force=True)
    assert order == ["link", "extension"]
    order.clear()
    monkeypatch.setitem(sys.modules, "torch", None)
    assert build.build(force=True) == tmp_path / "libpto_hip.so" and order == ["link"]
    assert "torch is not installed" in capsys.readouterr().err

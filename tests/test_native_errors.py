"""Tests of the native wrappers' error paths: an operand without storage (a functorch wrapper) comes back as a Python
exception, as it does from a ctypes call, whichever operand it is, and an allocation that fails raises what torch.empty
raises."""
import contextlib
import subprocess
import sys
from pathlib import Path

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

ROOT = Path(__file__).resolve().parents[1]

# Fake GPU tensors pass the checks of shape, type and device (and read as null pointers, which the library refuses);
# the operand under vmap is the one whose pointer cannot be read.
_CHILD = """
import sys
sys.path.insert(0, ROOT)
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
import __graft_entry__ as ge
k2 = ge.load_package()
k2._lib._stream_of_index = lambda i: 0
native = k2._lib._fast()
native.device_checked(0)
M, K, N, r = 16, 256, 128, 16
with FakeTensorMode():
    def t(*shape, dtype=torch.float32):
        return torch.empty(shape, dtype=dtype, device="cuda:0")
    ops = dict(x=t(M, K, dtype=torch.bfloat16), qx=t(M, K, dtype=torch.int8), sx=t(M), A=t(r, K), B=t(N, r),
               qw=t(N, K, dtype=torch.int8), sw=t(N), bias=t(N))

    for name, w in ops.items():
        def call(wrapped):
            o = dict(ops, **{name: wrapped})
            native.linear_fwd(o["x"], o["qx"], o["sx"], False, o["A"], o["B"], 1.0, o["qw"], o["sw"], o["bias"], False,
                              True)
            return wrapped

        try:
            torch.func.vmap(call)(torch.empty((2, *w.shape), dtype=w.dtype, device="cuda:0"))
        except RuntimeError as e:
            assert "data pointer" in str(e), e
            print("raised:", name, flush=True)
"""


def test_operand_without_storage_raises():
    r = subprocess.run([sys.executable, "-c", _CHILD.replace("ROOT", repr(str(ROOT)))], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]
    assert [line.split()[1] for line in r.stdout.splitlines() if line.startswith("raised:")] == \
        ["x", "qx", "sx", "A", "B", "qw", "sw", "bias"]


def test_failed_allocation_keeps_its_class(k2):
    """A device that this build has no backend for is a NotImplementedError of torch's, not a plain RuntimeError."""
    with FakeTensorMode():
        x = torch.empty((4, 128), device="xpu:0")
    with pytest.raises(NotImplementedError):
        k2._lib.alloc_codes(x)


def test_extension_of_another_torch_is_refused(k2, monkeypatch):
    L = k2._lib
    lib = L.load()
    monkeypatch.setattr(L, "_native", None)
    monkeypatch.setattr(L.torch, "__version__", "0.0.0")
    with pytest.raises(RuntimeError, match="run krea-2_amd/build.py"):
        L._bind_native(lib)
    assert L._native is None
    monkeypatch.undo()
    L._bind_native(lib)
    assert L._native is not None


def test_device_is_known_to_the_wrappers_before_other_threads_see_it_checked(k2, monkeypatch):
    """A thread that finds the device checked calls the native wrapper again at once: it must not refuse it then."""
    L = k2._lib
    seen = []
    known = {}
    monkeypatch.setattr(L, "_device_ok", known)
    monkeypatch.setattr(L, "load", lambda: type("Lib", (), {"k2q_check_device": staticmethod(lambda: L.K2Q_OK)}))
    monkeypatch.setattr(L, "_native", type("Native", (), {"device_checked": staticmethod(
        lambda i: seen.append(dict(known)))}))
    monkeypatch.setattr(L.torch.cuda, "device", lambda i: contextlib.nullcontext())
    L._device_check(torch.device("cuda:0"))
    assert seen == [{}] and known == {0: True}


@pytest.mark.gpu
def test_out_of_memory_keeps_its_class(k2, dev):
    x = torch.zeros((1, 128), dtype=torch.bfloat16, device=dev).expand(1 << 36, 128)     # codes of 8 TiB
    with pytest.raises(torch.OutOfMemoryError):
        k2._lib.alloc_codes(x)

"""The native call path of Backend.matmul and its like (cyb_amd/csrc/torch_calls.cpp), without a GPU: what it cannot look over it
hands back to the Python checks, which answer as they did when they were the only path.

The tensors here claim to be on cuda:0 and have no memory; the handle and the context are blank memory that no call gets as far
as reading into.  Each case runs in a process of its own: a C++ exception that leaves an entry ends the process."""
import os
import subprocess
import sys

import pytest

torch = pytest.importorskip("torch")
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_PROLOGUE = """
import ctypes, torch
from torch._subclasses.fake_tensor import FakeTensorMode
from cyb_amd import backend as B
blank = ctypes.create_string_buffer(4096)
addr = ctypes.addressof(blank)
calls = B._load_calls()
assert calls is not None

class NoAnswers(torch.Tensor):
    @staticmethod
    def __new__(cls):
        return torch.Tensor._make_wrapper_subclass(cls, (1, 4), dtype=torch.float16, device="cuda:0", dispatch_sizes_strides_policy="strides")
    @classmethod
    def __torch_dispatch__(cls, f, types, args=(), kwargs=None):
        raise RuntimeError("not answered")

def hand_backs(t):
    return [calls.matmul(addr, 0, addr, t, t, None, None, None, 0), calls.matmul(addr, 0, addr, t, t, 1, None, None, 0),
            calls.matmul_static(addr, 0, addr, t, t, None, 0), calls.matmul_fused(addr, 0, addr, t, t, 1e-5, t, 0, t, None, 0)]

be = B.Backend.__new__(B.Backend)            # the Python checks alone: no context, no device
be.device, be._addr, be._ctx = 0, addr, ctypes.c_void_p()
be.weights, be._lib = {}, B.load_library()
w = B.QWeight.__new__(B.QWeight)
w._h, w._addr, w._backend, w.N, w.K = ctypes.c_void_p(addr), addr, be, 1, 4

def through_backend(t):
    assert hand_backs(t) == [1, 1, 1, 1]
    try:
        be.matmul(w, t, t)
    except RuntimeError as e:
        print("raised", type(e).__name__, flush=True)
        raise SystemExit(0)                  # (there is nothing to return to a transform)
"""

_CASES = {
    "subclass that raises": "through_backend(NoAnswers())",
    "vmap": "with FakeTensorMode():\n    torch.vmap(through_backend)(torch.empty((2, 1, 4), device='cuda', dtype=torch.float16))",
    "grad": "with FakeTensorMode():\n    torch.func.grad(through_backend)(torch.empty((1, 4), device='cuda'))",
    "fake": "with FakeTensorMode():\n    through_backend(torch.empty((1, 4), device='cuda', dtype=torch.float16))",
    "cpu": "through_backend(torch.empty((1, 4), dtype=torch.float16))",
}


@pytest.mark.parametrize("case", _CASES)
def test_tensors_without_an_address_are_handed_back_and_raise(case):
    p = subprocess.run([sys.executable, "-c", _PROLOGUE + _CASES[case]], cwd=ROOT, capture_output=True, text=True, timeout=110)
    assert p.returncode == 0, p.stderr[-2000:]
    assert "raised" in p.stdout, p.stdout + p.stderr[-2000:]


@pytest.mark.parametrize("args", ["(addr, 0, addr, x, x, True, None, None, 0)", "(addr, 0, addr, x, x, 1 << 70, None, None, 0)",
                                  "(0, 0, addr, x, x, None, None, None, 0)", "(addr, 0, 0, x, x, None, None, None, 0)",
                                  "(addr, 0, addr, None, x, None, None, None, 0)", "(addr, 0, addr, 4096, x, 1, None, None, 0)",
                                  "(addr, 0, addr, x, x, None, None, None, None)", "(addr, 0, addr, x, x)", "()"])
def test_arguments_that_are_not_a_plain_call_are_handed_back(args):
    code = _PROLOGUE + f"x = torch.empty((1, 4), dtype=torch.float16)\nassert calls.matmul{args} == 1"
    p = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=110)
    assert p.returncode == 0, p.stderr[-2000:]


@pytest.mark.parametrize("what", ["missing", "not a library", "another torch"])
def test_without_the_native_path_the_ctypes_calls_serve(what, tmp_path, monkeypatch):
    import ctypes

    from cyb_amd import backend as B
    monkeypatch.setattr(B, "_calls", None)
    if what == "another torch":
        monkeypatch.setattr(torch, "__version__", "1.0.0")
    else:
        path = tmp_path / "_torch_calls.so"
        if what == "not a library":
            path.write_bytes(b"not a library")
        monkeypatch.setattr(B, "_CALLS_PATH", str(path))
    be = B.Backend.__new__(B.Backend)
    be._lib, be._ctx, be._addr, be.device, be.weights = B.load_library(), ctypes.c_void_p(), 0, 0, {}
    w = B.QWeight.__new__(B.QWeight)
    w._h, w._addr, w._backend, w.N, w.K = ctypes.c_void_p(), 0, be, 4, 4
    x = torch.empty((1, 4), dtype=torch.float16)
    with pytest.warns(RuntimeWarning, match="_torch_calls.so"):
        with pytest.raises(B.CybqError, match="must live on cuda:0"):           # (the Python checks have the call)
            be.matmul(w, x, x)
    for call in (lambda: be.matmul_static(w, x, x), lambda: be.matmul_ex(w, x, x), lambda: be.matmul_norm(w, x, x, 1e-5, x)):
        with pytest.raises(B.CybqError, match="must live on cuda:0"):
            call()


def test_the_library_builds_without_torch():
    """`make` is also what the C++ and Rust users run."""
    p = subprocess.run(["make", "-n", "-B", "PYTHON=/bin/false"], cwd=os.path.join(ROOT, "cyb_amd", "csrc"), capture_output=True, text=True)
    assert p.returncode == 0 and "libcybq.so" in p.stdout, p.stderr
    assert "torch" not in p.stdout

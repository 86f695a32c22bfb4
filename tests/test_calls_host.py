"""The native operator calls (csrc/calls.cpp) without a GPU: built for CPU tensors, what they do with tensors that have no data
pointer; and the package without them, or without the library."""
import os
import subprocess
import sys
import sysconfig

import pytest
import torch

import unit_amd
from unit_amd import _lib, ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# calls.cpp with CPU tensors in the place of GPU ones and no stream; its headers first, so that the macros reach its own code only
SOURCE = """
#include <Python.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
namespace c10::hip {
struct NoStream { void *stream() const { return nullptr; } };
inline NoStream no_stream() { return {}; }
}
#define is_cuda is_cpu
#define getCurrentHIPStream no_stream
#include "%s"
"""

PROGRAM = """
import ctypes, sys
sys.path.insert(0, sys.argv[1])
sys.path.insert(0, sys.argv[2])
import torch
import _calls
from unit_amd import _lib, ops
L = _lib.load()
reached = []
kinds = {}
def answer(name):  # the library's function: notes the call, and takes the interpreter's lock to do so
    f = getattr(L, name)
    kinds[name] = ctypes.CFUNCTYPE(ctypes.c_int, *f.argtypes)(lambda *a: reached.append(name) or 0)
    return ctypes.cast(kinds[name], ctypes.c_void_p).value
_calls.bind(tuple(answer(f) if "gemm" in f or "dense" in f else ctypes.cast(getattr(L, f), ctypes.c_void_p).value
                  for f in ops._Calls._LIBRARY),
            ops.PreparedConvWeight, ops.PreparedDenseWeight, ops.PreparedGemmB, torch.int8, torch.float16)
h = lambda *s: torch.zeros(s, dtype=torch.float16)
u8 = lambda *s: torch.zeros(s, dtype=torch.uint8)
s8 = lambda *s: torch.zeros(s, dtype=torch.int8)
a, b, ws = h(4, 16), h(16, 8), u8(64)
assert _calls.gemm(a, b, False, None).shape == (4, 8) and reached == ["unit_gemm_f16"], reached
assert _calls.dense(u8(4, 64), s8(128, 64)).dtype == torch.int32
reached.clear()
declined = []
def mapped(call, *operands):
    def one(*x):
        declined.append(call(*x) is None)
        return x[0]
    torch.vmap(one)(*operands)
bias = torch.zeros(2, 16, dtype=torch.int32)
mapped(lambda x: _calls.gemm(x, b, False, None), h(3, 4, 16))
mapped(lambda x: _calls.gemm(a, x, True, None), h(3, 16, 8))
mapped(lambda x: _calls.gemm(a, b, True, x), u8(3, 64))
mapped(lambda x: _calls.dense(x, s8(128, 64)), u8(3, 4, 64))
mapped(lambda x: _calls.dense(u8(4, 64), x), s8(3, 128, 64))
mapped(lambda x: _calls.conv_u8(x, s8(1, 1, 1, 1, 4, 16, 4), 1, 0, 1), u8(3, 1, 1, 4, 4, 16))
mapped(lambda x: _calls.conv_u8(u8(1, 1, 4, 4, 16), x, 1, 0, 1), s8(3, 1, 1, 1, 1, 4, 16, 4))
mapped(lambda x: _calls.conv_fused(s8(1, 1, 4, 4, 16), s8(1, 1, 1, 1, 4, 16, 4), x, 3, 1, 0, 1), bias)
mapped(lambda x: _calls.conv3d(x, s8(1, 1, 1, 1, 1, 4, 16, 4), 1), s8(2, 1, 1, 4, 4, 4, 16))
mapped(lambda x: _calls.conv_f16(x, h(1, 1, 1, 1, 16, 16), 1, 1), h(3, 1, 1, 4, 4, 16))
mapped(lambda x: _calls.conv_f16(h(1, 16, 4, 4), x, 1, 1), h(3, 16, 16, 1, 1))
prepared = ops.PreparedGemmB(h(8, 16), 16, 8)
def inner(x):
    prepared.bt = x
    return _calls.gemm(a, prepared, False, None)
mapped(inner, h(3, 8, 16))
assert len(declined) == 12 and all(declined) and not reached, (declined, reached)
print("declined")
"""


@pytest.fixture(scope="module")
def module(tmp_path_factory):
    out = tmp_path_factory.mktemp("calls")
    src = out / "calls_cpu.cpp"
    src.write_text(SOURCE % os.path.join(ROOT, "unit_amd", "csrc", "calls.cpp"))
    base = os.path.dirname(torch.__file__)
    subprocess.check_call([os.environ.get("CXX", "g++"), "-O0", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-w",
                           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-I" + sysconfig.get_paths()["include"], f"-I{base}/include",
                           f"-I{base}/include/torch/csrc/api/include", "-I/opt/rocm/include", str(src), f"-L{base}/lib", "-ltorch_python",
                           "-ltorch_cpu", "-lc10", "-lc10_hip", "-o", str(out / "_calls.so")])
    return out


def test_tensors_without_storage_are_declined(module):
    """vmap's wrapped tensors are torch.Tensors of the right type and shape; asking one for its data throws."""
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(module), ROOT], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "declined", (r.returncode, r.stdout, r.stderr[-2000:])


def test_without_the_module_the_python_operators_take_the_call(monkeypatch):
    monkeypatch.delattr(unit_amd, "_calls", raising=False)
    monkeypatch.setitem(sys.modules, "unit_amd._calls", None)
    monkeypatch.setattr(ops, "_native", ops._Calls())
    a = torch.zeros((4, 16), dtype=torch.float16)
    with pytest.warns(RuntimeWarning, match="make -C"), pytest.raises(ValueError, match="must live on the GPU"):
        ops.gemm_fp16(a, a)
    with pytest.raises(ValueError, match="must live on the GPU"):  # said once
        ops.dense(a.to(torch.uint8), a.to(torch.int8))


def test_without_the_library_arguments_are_checked_first(monkeypatch):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", os.path.join(ROOT, "no such library"))
    monkeypatch.setattr(ops, "_native", ops._Calls())
    with pytest.raises(TypeError, match="expected a torch.Tensor"):
        ops.gemm_fp16([1.0], None)
    with pytest.raises(_lib.UnitError, match="make -C"):
        _lib.load()


def test_make_without_torch_builds_the_library_alone():
    make = ["make", "-n", "-C", os.path.join(ROOT, "unit_amd", "csrc"), "-W", "calls.cpp", "all"]
    assert "_calls.so" in subprocess.run(make, capture_output=True, text=True, check=True).stdout
    assert "_calls.so" not in subprocess.run(make + ["TORCH="], capture_output=True, text=True, check=True).stdout

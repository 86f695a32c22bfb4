"""The native operator calls against the Python operators of the same names: the same results, and the same errors for what
they hand on."""
import pytest
import torch

import unit_amd as U
from unit_amd import ops

pytestmark = pytest.mark.gpu


class _Declines:
    def __getattr__(self, name):
        return lambda *args: None


def _operands(dev):
    g = torch.Generator(device=dev).manual_seed(3)

    def i8(shape, lo=-128, hi=128, dtype=torch.int8):
        return torch.randint(lo, hi, shape, dtype=dtype, device=dev, generator=g)

    def f16(shape):
        return (torch.randn(shape, device=dev, generator=g) * 0.1).half()

    return i8, lambda shape: i8(shape, 0, 256, torch.uint8), f16


def _calls(dev):
    """name -> (function of no arguments, whether the native side takes it)"""
    i8, u8, f16 = _operands(dev)
    x, w, xs = u8((2, 3, 9, 8, 16)), i8((2, 3, 3, 3, 4, 16, 4)), i8((2, 3, 9, 8, 16))
    x4, w4 = u8((1, 1, 12, 11, 4)), i8((2, 1, 5, 7, 1, 16, 4))
    bias = i8((32,), -1000, 1000, torch.int32)
    xh, wh = f16((2, 2, 7, 9, 16)), f16((3, 2, 3, 3, 16, 16))
    xp, wp = f16((1, 32, 9, 9)), f16((48, 32, 3, 3))
    a, b = f16((33, 72)), f16((72, 40))
    d, e = u8((17, 64)), i8((128, 64))
    pw, pwh, pb, pe = U.prepare_conv2d_weight(w), U.prepare_conv2d_weight(wh), U.prepare_gemm_b(b), U.prepare_dense_weight(e)
    packed = U.prepack_dense_weight(e)
    x3, w3 = i8((1, 2, 4, 6, 5, 16)), i8((2, 2, 3, 3, 3, 4, 16, 4))
    ws = torch.empty(max(16, U.gemm_fp16_workspace_bytes(33, 40, 72)), dtype=torch.uint8, device=dev)
    strided = torch.empty((2, 3, 9, 16, 16), dtype=torch.uint8, device=dev)[:, :, :, ::2]
    strided.copy_(x)
    return {
        "conv": (lambda: U.conv2d_NCHWc_int8(x, w, 1, 1), True),
        "conv_pairs": (lambda: U.conv2d_NCHWc_int8(x, w, (2, 1), (1, 0, 2, 1), (1, 2)), True),
        "conv_list": (lambda: U.conv2d_NCHWc_int8(x, w, [2, 1], [1, 0]), False),
        "conv_prepared": (lambda: U.conv2d_NCHWc_int8(x, pw, 1, (1, 1)), True),
        "conv_c4": (lambda: U.conv2d_NCHWc_int8(x4, w4, 2, (2, 3)), True),
        "conv_layout": (lambda: U.conv2d_NCHWc_int8(x, w, 1, 1, 1, "int32", "NCHW4c", "NCHW16c"), False),
        "conv_strided": (lambda: U.conv2d_NCHWc_int8(strided, w, 1, 1), False),
        "fused": (lambda: U.conv2d_NCHWc_int8_fused(xs, w, bias, 11, 1, 1), True),
        "fused_prepared": (lambda: U.conv2d_NCHWc_int8_fused(xs, pw, None, -3, 2, 0), True),
        "fused_planar": (lambda: U.conv2d_NCHWc_int8_fused(xs, pw, bias, 2, 1, 1, 1, "int32", "NCHW16c", "NCHW", 30), False),
        "requant": (lambda: U.conv2d_NCHWc_int8_requant(x, pw, bias, 3, 14, 1, 1), True),
        "requant_plain": (lambda: U.conv2d_NCHWc_int8_requant(x, w, None, 3, 14, 1, 1), False),
        "conv3d": (lambda: U.conv3d_NCDHWc_int8(x3, w3, 1), True),
        "conv_f16": (lambda: U.conv2d_NCHW16c_OHWI16o(xh, wh, 1, 2), True),
        "conv_f16_prepared": (lambda: U.conv2d_NCHW16c_OHWI16o(xh, pwh, 2, 1), True),
        "conv_f16_plain": (lambda: U.conv2d_NCHW16c_OHWI16o(xp, wp, 2, 2), True),
        "gemm": (lambda: U.gemm_fp16(a, b), True),
        "gemm_half": (lambda: U.gemm_fp16(a, b, "float16"), True),
        "gemm_prepared": (lambda: U.gemm_fp16(a, pb), True),
        "gemm_workspace": (lambda: U.gemm_fp16(a, b, "float16", ws), True),
        "gemm_own_workspace": (lambda: U.gemm_fp16(a, b, "float32", True), False),
        "gemm_transposed": (lambda: U.gemm_fp16(a, b.t().contiguous().t()), False),
        "dense": (lambda: U.dense(d, e), True),
        "dense_prepared": (lambda: U.dense(d, pe), True),
        "dense_packed": (lambda: U.dense_dotprod(d, packed), True),
    }


def _errors(dev):
    i8, u8, f16 = _operands(dev)
    x, w = u8((1, 2, 5, 5, 16)), i8((1, 2, 3, 3, 4, 16, 4))
    pw = U.prepare_conv2d_weight(w)
    return {
        "cpu": lambda: U.conv2d_NCHWc_int8(x.cpu(), w, 1, 1),
        "dtype": lambda: U.conv2d_NCHWc_int8(x, w.half(), 1, 1),
        "channels": lambda: U.conv2d_NCHWc_int8(x[:, :1].contiguous(), pw, 1, 1),
        "window": lambda: U.conv2d_NCHWc_int8(x, i8((1, 2, 7, 7, 4, 16, 4)), 1, 0),
        "stride": lambda: U.conv2d_NCHWc_int8(x, w, 0, 1),
        "scale": lambda: U.conv2d_NCHWc_int8_fused(i8((1, 2, 5, 5, 16)), w, None, 2 ** 31, 1, 1),
        "bias": lambda: U.conv2d_NCHWc_int8_fused(i8((1, 2, 5, 5, 16)), w, torch.zeros(3, dtype=torch.int32, device=dev), 1, 1, 1),
        "shift": lambda: U.conv2d_NCHWc_int8_requant(x, pw, None, 1, 63, 1, 1),
        "gemm": lambda: U.gemm_fp16(f16((4, 16)), f16((24, 8))),
        "gemm_ws": lambda: U.gemm_fp16(f16((64, 4096)), f16((4096, 64)), "float16", torch.empty(16, dtype=torch.uint8, device=dev)),
        "dense_4d": lambda: U.dense(u8((4, 64)), U.prepack_dense_weight(i8((128, 64)))),
        "dense_k": lambda: U.dense(u8((4, 64)), i8((8, 32))),
        "conv3d": lambda: U.conv3d_NCDHWc_int8(i8((1, 1, 2, 4, 4, 16)), i8((1, 1, 3, 3, 3, 4, 16, 4)), 1),
    }


def test_native_calls_agree_with_the_python_operators(dev, monkeypatch):
    calls = _calls(dev)
    taken = {}

    class Notes:
        def __getattr__(self, name):
            def call(*args):
                out = getattr(ops._Calls.__getattr__(ops._Calls(), name), "__call__")(*args)
                taken[current] = out is not None
                return out
            return call

    got = {}
    monkeypatch.setattr(ops, "_native", Notes())
    for current, (fn, _) in calls.items():
        got[current] = fn()
    monkeypatch.setattr(ops, "_native", _Declines())
    for name, (fn, native) in calls.items():
        want = fn()
        assert got[name].dtype == want.dtype and got[name].device == want.device and torch.equal(got[name], want), name
        assert taken.get(name, False) == native, name


def test_native_calls_leave_errors_to_the_python_operators(dev, monkeypatch):
    for name, fn in _errors(dev).items():
        with pytest.raises((TypeError, ValueError)) as here:
            fn()
        with monkeypatch.context() as m:
            m.setattr(ops, "_native", _Declines())
            with pytest.raises((TypeError, ValueError)) as there:
                fn()
        assert type(here.value) is type(there.value) and str(here.value) == str(there.value), name


def test_wrapped_tensors_raise_as_in_the_python_operators(dev, monkeypatch):
    """torch.vmap's tensors have no data pointer: an error on the host, before any launch."""
    _, _, f16 = _operands(dev)
    batch, b = f16((3, 4, 16)), f16((16, 8))
    with pytest.raises(RuntimeError) as here:
        torch.vmap(lambda a: U.gemm_fp16(a, b))(batch)
    monkeypatch.setattr(ops, "_native", _Declines())
    with pytest.raises(RuntimeError) as there:
        torch.vmap(lambda a: U.gemm_fp16(a, b))(batch)
    assert str(here.value) == str(there.value)

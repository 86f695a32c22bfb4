"""Operator entry points of the tensorized conv2d / dense / GEMM path, on torch tensors that live
on the MI355X.  Same names, argument order and argument meaning as the reference operators they
replace; every one hands raw device pointers to the C ABI in libunit_amd.so (hand-written gfx950
kernels).  torch is used to allocate the result and to read shapes / pointers, nothing else.

Reference call sites:
  conv2d_NCHWc_int8        apps/cpu/kernel/conv2d.py:50-51   (topi.nn.conv2d_NCHWc_int8)
  dense_dotprod            apps/cpu/kernel/int8-gemm.py:13-16 (topi.x86.dense_dotprod)
  dense                    apps/cpu/relay/int8-gemm.py:14-16  (relay.nn.dense)
  conv2d_NCHW16c_OHWI16o   python/tensorizer/ops/gpu.py:8-53  (_conv2d_NCHW16c_OHWI16o_impl)
  gemm_fp16                apps/gpu/gemm.py:8-20
"""
import ctypes
import os
import re
import warnings
from functools import lru_cache

import torch

from . import _lib
from ._lib import ConvDesc, check

__all__ = [
    "conv2d_NCHWc_int8", "dense_dotprod", "dense", "conv2d_NCHW16c_OHWI16o", "gemm_fp16", "gemm_fp16_workspace_bytes",
    "pack_nchwc", "unpack_nchwc", "prepack_conv_weight", "prepack_dense_weight", "prepare_dense_weight", "PreparedDenseWeight",
    "prepack_conv_weight_f16", "conv_out_hw", "last_variant",
    "PreparedConvWeight", "prepare_conv2d_weight", "PreparedGemmB", "prepare_gemm_b",
    "conv2d_NCHWc_int8_requant",
]


# ------------------------------------------------------------------------------- helpers
_raw_stream, _device = (getattr(torch._C, name, None) for name in ("_cuda_getCurrentRawStream", "_cuda_getDevice"))


def _stream():
    # the handle of torch.cuda.current_stream(); without building the Stream object where torch allows (0.2 against 2.7 us)
    if _raw_stream is None or _device is None:
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(_device())


def _dev(t, name, dtype=None, ndim=None):
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{name}: expected a torch.Tensor, got {type(t).__name__}")
    if not t.is_cuda:
        raise ValueError(f"{name}: tensor must live on the GPU (there is no CPU implementation)")
    if dtype is not None and t.dtype != dtype:
        raise TypeError(f"{name}: expected dtype {dtype}, got {t.dtype}")
    if ndim is not None and t.dim() not in (ndim if isinstance(ndim, tuple) else (ndim,)):
        raise ValueError(f"{name}: expected {ndim}-D tensor, got shape {tuple(t.shape)}")
    return t if t.is_contiguous() else t.contiguous()


def _pair(v, name):
    if isinstance(v, int):
        return v, v
    v = tuple(int(x) for x in v)
    if len(v) != 2:
        raise ValueError(f"{name}: expected an int or a pair, got {v}")
    return v


def _pad4(padding):
    """TVM's get_pad_tuple: int -> all sides; (ph, pw) -> symmetric; (pt, pl, pb, pr)."""
    if isinstance(padding, int):
        return padding, padding, padding, padding
    p = tuple(int(x) for x in padding)
    if len(p) == 2:
        return p[0], p[1], p[0], p[1]
    if len(p) == 4:
        return p
    raise ValueError(f"padding: expected an int, (ph, pw) or (pt, pl, pb, pr), got {p}")


@lru_cache(maxsize=64)
def _layout_block(layout, name):
    m = re.fullmatch(r"NCHW(\d+)c", layout)
    if not m:
        raise ValueError(f"{name}: expected a layout of the form NCHW<x>c, got {layout!r}")
    return int(m.group(1))


def conv_out_hw(h, w, kh, kw, stride, padding=0, dilation=1):
    """Output height / width of a convolution, as the library computes it."""
    sh, sw = _pair(stride, "stride")
    dh, dw = _pair(dilation, "dilation")
    pt, pl, pb, pr = _pad4(padding)
    d = ConvDesc(1, 16, h, w, 16, kh, kw, sh, sw, pt, pl, pb, pr, dh, dw, 16)
    oh, ow = ctypes.c_int32(), ctypes.c_int32()
    check(_lib.load().unit_conv_out_hw(ctypes.byref(d), ctypes.byref(oh), ctypes.byref(ow)))
    return oh.value, ow.value


# Shapes, strides and padding of a convolution -> its descriptor and result shape.  A call costs the GPU as little as
# 4 us, less than checking the operands' shapes against each other and asking the library for the output size on
# every call did: that is a function of these plain values alone and is kept for the last 1024 combinations.
class _ConvPlan:
    __slots__ = ("desc", "ref", "ko", "n", "oh", "ow", "blocked")

    def __init__(self, n, c, h, w, k, kh, kw, stride, padding, dilation, cb):
        sh, sw = _pair(stride, "stride")
        dh, dw = _pair(dilation, "dilation")
        pt, pl, pb, pr = _pad4(padding)
        self.desc = ConvDesc(n, c, h, w, k, kh, kw, sh, sw, pt, pl, pb, pr, dh, dw, cb)
        self.ref = ctypes.byref(self.desc)
        oh, ow = ctypes.c_int32(), ctypes.c_int32()
        check(_lib.load().unit_conv_out_hw(self.ref, ctypes.byref(oh), ctypes.byref(ow)))
        self.n, self.ko, self.oh, self.ow = n, k // 16, oh.value, ow.value
        self.blocked = (n, self.ko, self.oh, self.ow, 16)  # shape of the blocked result


@lru_cache(maxsize=1024, typed=True)
def _plan_int8(dshape, kshape, stride, padding, dilation):
    """dshape: the data's; kshape: the blocked kernel's, or (K, C, KH, KW, cb) of a prepared one."""
    n, cc, h, w, cb = dshape
    if cb not in (4, 16):
        raise ValueError(f"data: channel block must be 16 or 4, got {cb}")
    if len(kshape) == 5:
        k, c, kh, kw, kcb = kshape
        if kcb != cb or c != cc * cb:
            raise ValueError(f"kernel: prepared for K={k}, C={c}, {kh} x {kw}, channel blocks of {kcb}: does not match data {tuple(dshape)}")
    else:
        ko, cc2, kh, kw, e, kb, i4 = kshape
        if (cc2, e, kb, i4) != (cc, cb // 4, 16, 4):
            raise ValueError(f"kernel: shape {tuple(kshape)} does not match data {tuple(dshape)}; "
                             f"expected (K/16, {cc}, KH, KW, {cb // 4}, 16, 4)")
        k = ko * 16
    return _ConvPlan(n, cc * cb, h, w, k, kh, kw, stride, padding, dilation, cb)


@lru_cache(maxsize=1024, typed=True)
def _plan_f16(dshape, kshape, stride_h, stride_w):
    """dshape (N, C/16, H, W, 16); kshape: the blocked kernel's, or (K, C, KH, KW, 16) of a prepared one."""
    n, cc, h, w, cb = dshape
    if len(kshape) == 5:
        k, c, kh, kw, kcb = kshape
        if kcb != cb or c != cc * cb:
            raise ValueError(f"kernel: prepared for K={k}, C={c}, {kh} x {kw}, channel blocks of {kcb}: does not match data {tuple(dshape)}")
    else:
        ko, ib, kh, kw, ic, ob = kshape
        if cb != 16 or ic != 16 or ob != 16 or ib != cc:
            raise ValueError(f"a {tuple(dshape)} / b {tuple(kshape)}: expected (N, C/16, H, W, 16) and "
                             f"(K/16, C/16, KH, KW, 16, 16)")
        k = ko * 16
    return _ConvPlan(n, cc * 16, h, w, k, kh, kw, (stride_h, stride_w), 0, 1, 16)


def _hashable(v):
    """A stride / padding / dilation argument as a key: ints and tuples as they are, other sequences as tuples of ints."""
    return v if type(v) is int else v if isinstance(v, int) else tuple(int(x) for x in v)


def _plan(data, kernel, stride, padding, dilation):
    kshape = kernel.key if isinstance(kernel, PreparedConvWeight) else kernel.shape
    return _plan_int8(data.shape, kshape, _hashable(stride), _hashable(padding), _hashable(dilation))


def last_variant():
    """Kernel variant chosen by the last compute call (the analogue of the tuned-schedule index
    the reference records per shape, python/tensorizer/tune.py:20-31)."""
    return _lib.last_variant()


# ------------------------------------------------------------------------------- native calls
class _Calls:
    """The operators' common case as native functions (csrc/calls.cpp): each returns the result, or None for a call that
    it does not take, which then runs through the Python below.  Bound on first use to the library that ctypes loaded.  The
    module is built against the installed torch (csrc/Makefile); where there is none that fits, the Python takes every call."""

    _NAMES = ("conv_u8", "conv_fused", "conv_requant", "conv3d", "conv_f16", "dense", "gemm")

    _LIBRARY = ("unit_conv_out_hw", "unit_conv2d_nchwc_u8s8s32", "unit_conv2d_nchwc_u8s8s32_prepared", "unit_conv2d_nchwc_s8s8s32_fused",
                "unit_conv2d_nchwc_s8s8s32_fused_prepared", "unit_conv2d_nchwc_u8s8u8_requant_prepared", "unit_conv3d_ncdhwc_s8s8s32",
                "unit_conv2d_nchw16c_f16f32", "unit_conv2d_nchw16c_f16f32_prepared", "unit_conv2d_nchw_f16f32",
                "unit_conv2d_nchw_f16f32_ws_bytes", "unit_dense_dotprod_u8s8s32", "unit_dense_u8s8s32", "unit_dense_u8s8s32_prepared",
                "unit_gemm_f16", "unit_gemm_f16_prepared", "unit_gemm_f16_ws")

    def __getattr__(self, name):  # the first use of each function
        if name not in self._NAMES:
            raise AttributeError(name)
        try:
            L = _lib.load()
        except _lib.UnitError:  # not built: said by the Python operator, after its checks
            return _declined
        try:
            from . import _calls
            _calls.bind(tuple(ctypes.cast(getattr(L, f), ctypes.c_void_p).value for f in self._LIBRARY), PreparedConvWeight,
                        PreparedDenseWeight, PreparedGemmB, torch.int8, torch.float16)
            fn = getattr(_calls, name)
        except (ImportError, AttributeError, ValueError) as e:
            fn = _declined
            if "_said" not in self.__dict__:
                self._said = True
                warnings.warn(f"unit_amd: the native operator calls do not fit this torch or are not built ({e}); every call goes "
                              f"through Python, about 2 us slower. Build them with `make -C {os.path.dirname(__file__)}/csrc`.",
                              RuntimeWarning, stacklevel=3)
        setattr(self, name, fn)
        return fn


def _declined(*args):
    return None


_native = _Calls()


# ------------------------------------------------------------------------------- prepared weights
class PreparedConvWeight:
    """Convolution weights in the MFMA fragment order of the kernels (see prepare_conv2d_weight).
    Accepted wherever conv2d_NCHWc_int8, conv2d_NCHWc_int8_fused and conv2d_NCHW16c_OHWI16o take
    a kernel."""

    def __init__(self, buf, K, C, KH, KW, cb, dtype):
        self.buf, self.K, self.C, self.KH, self.KW, self.cb, self.dtype = buf, K, C, KH, KW, cb, dtype

    @property
    def key(self):
        return self.K, self.C, self.KH, self.KW, self.cb

    def __repr__(self):
        return (f"PreparedConvWeight(K={self.K}, C={self.C}, KH={self.KH}, KW={self.KW}, cb={self.cb}, "
                f"dtype={self.dtype})")


def prepare_conv2d_weight(kernel):
    """Re-order a blocked convolution weight once for the direct kernels: the counterpart of the
    constant sub-graphs the reference's compiled models keep next to each convolution (weight
    layout chain apps/cpu/relay/result.log:8-13, sum(w) result.log:15-16).

    kernel int8 (K/16, C/16, KH, KW, 4, 16, 4), int8 (K/16, C/4, KH, KW, 1, 16, 4) with KW <= 8 (the stem's
           4-channel blocks), or fp16 (K/16, C/16, KH, KW, 16 in, 16 out)
    returns a PreparedConvWeight; convolutions on it give the same results as on `kernel`.
    """
    if isinstance(kernel, torch.Tensor) and kernel.dtype == torch.float16:
        kernel = _dev(kernel, "kernel", torch.float16, 6)
        ko, cc, kh, kw, ic, ob = kernel.shape
        if (ic, ob) != (16, 16):
            raise ValueError(f"kernel: expected (K/16, C/16, KH, KW, 16, 16), got {tuple(kernel.shape)}")
        eb, cb = 2, 16
    else:
        kernel = _dev(kernel, "kernel", torch.int8, 7)
        ko, cc, kh, kw, e, kb, i4 = kernel.shape
        if e not in (1, 4) or (kb, i4) != (16, 4):
            raise ValueError(f"kernel: expected (K/16, C/cb, KH, KW, cb/4, 16, 4) with cb 16 or 4, got {tuple(kernel.shape)}")
        eb, cb = 1, 4 * e
    L = _lib.load()
    nbytes = ctypes.c_size_t()
    check(L.unit_conv2d_prepared_weight_bytes(ko * 16, cc * cb, kh, kw, cb, eb, ctypes.byref(nbytes)))
    buf = torch.empty(nbytes.value, dtype=torch.uint8, device=kernel.device)
    check(L.unit_conv2d_prepare_weight(ko * 16, cc * cb, kh, kw, cb, eb, kernel.data_ptr(), buf.data_ptr(), _stream()))
    return PreparedConvWeight(buf, ko * 16, cc * cb, kh, kw, cb, kernel.dtype)


def _check_prepared(kernel, data, want_dtype):
    if kernel.dtype != want_dtype:
        raise TypeError(f"kernel: prepared from {kernel.dtype}, this operator takes {want_dtype}")
    if kernel.buf.device != data.device:
        raise ValueError("kernel: prepared on another device")


def _check_bias(bias, k, data):
    if bias.dtype != torch.int32 or bias.numel() != k or bias.device != data.device:
        raise ValueError(f"bias: expected {k} int32 values on {data.device}")
    return bias.contiguous()


# ------------------------------------------------------------------------------- int8
def conv2d_NCHWc_int8(data, kernel, stride, padding, dilation=1, out_dtype="int32", layout="NCHW16c",
                      out_layout="NCHW16c"):
    """u8 x s8 -> i32 convolution on blocked layouts.

    data   uint8 (N, C/cb, H, W, cb), cb in {16, 4}
    kernel int8  (K/16, C/cb, KH, KW, cb/4, 16, 4)
    returns int32 (N, K/16, OH, OW, 16)

    As in TVM the channel block is taken from the tensor shapes; `layout` / `out_layout` are
    checked for form only (the reference's driver passes 'NCHW4c' for 16-channel blocks too).
    """
    if out_dtype == "int32" and layout == "NCHW16c" and out_layout == "NCHW16c":
        out = _native.conv_u8(data, kernel, stride, padding, dilation)
        if out is not None:
            return out
    data = _dev(data, "data", torch.uint8, 5)
    prepared = isinstance(kernel, PreparedConvWeight)
    if not prepared:
        kernel = _dev(kernel, "kernel", torch.int8, 7)
    if out_dtype != "int32":
        raise ValueError(f"out_dtype: only 'int32' is supported, got {out_dtype!r}")
    _layout_block(layout, "layout")
    if _layout_block(out_layout, "out_layout") != 16:
        raise ValueError("out_layout: the output channel block is 16 (NCHW16c)")
    if prepared:
        _check_prepared(kernel, data, torch.int8)
    p = _plan(data, kernel, stride, padding, dilation)
    L = _lib.load()
    out = data.new_empty(p.blocked, dtype=torch.int32)
    if prepared:
        check(L.unit_conv2d_nchwc_u8s8s32_prepared(p.ref, data.data_ptr(), kernel.buf.data_ptr(), out.data_ptr(), _stream()))
    else:
        check(L.unit_conv2d_nchwc_u8s8s32(p.ref, data.data_ptr(), kernel.data_ptr(), out.data_ptr(), _stream()))
    return out


def conv2d_NCHWc_int8_fused(data, kernel, bias, scale, stride, padding, dilation=1, out_dtype="int32",
                            layout="NCHW16c", out_layout="NCHW16c", out_channels=None):
    """The quantized model form of the convolution,
    fused_nn_contrib_conv2d_NCHWc_subtract_add_multiply (apps/cpu/relay/result.log:3-26,35):

        out = (conv2d_NCHWc_int8(data + 128, kernel) - 128 * sum(kernel per out channel) + bias) * scale

    on signed activations, in int32.

    data   int8  (N, C/cb, H, W, cb), cb in {16, 4}
    kernel int8  (K/16, C/cb, KH, KW, cb/4, 16, 4)
    bias   int32 (K,) / any shape with K elements, or None
    scale  Python int
    returns int32 (N, K/16, OH, OW, 16)

    out_layout='NCHW' (prepared weights only) folds the graph's closing layout_transform
    (result.log:25) into the store: returns int32 (N, out_channels, OH, OW), out_channels
    (default K) being the channel count before the caller padded it up to a multiple of 16.
    """
    if out_dtype == "int32" and layout == "NCHW16c" and out_layout == "NCHW16c" and out_channels is None:
        out = _native.conv_fused(data, kernel, bias, scale, stride, padding, dilation)
        if out is not None:
            return out
    data = _dev(data, "data", torch.int8, 5)
    prepared = isinstance(kernel, PreparedConvWeight)
    if not prepared:
        kernel = _dev(kernel, "kernel", torch.int8, 7)
    if out_dtype != "int32":
        raise ValueError(f"out_dtype: only 'int32' is supported, got {out_dtype!r}")
    _layout_block(layout, "layout")
    planar = out_layout == "NCHW"
    if planar and not prepared:
        raise ValueError("out_layout: 'NCHW' needs prepared weights (prepare_conv2d_weight)")
    if not planar and out_channels is not None:
        raise ValueError("out_channels: only with out_layout='NCHW'")
    if not planar and _layout_block(out_layout, "out_layout") != 16:
        raise ValueError("out_layout: the output channel block is 16 (NCHW16c), or 'NCHW'")
    if prepared:
        _check_prepared(kernel, data, torch.int8)
    p = _plan(data, kernel, stride, padding, dilation)
    bias_ptr = None
    if bias is not None:
        bias = _check_bias(bias, p.ko * 16, data)
        bias_ptr = bias.data_ptr()
    scale = int(scale)
    if not -2 ** 31 <= scale < 2 ** 31:
        raise ValueError("scale: must fit int32")
    L = _lib.load()
    if planar:
        oc = p.ko * 16 if out_channels is None else int(out_channels)
        if not p.ko * 16 - 16 < oc <= p.ko * 16:
            raise ValueError(f"out_channels: {oc} does not round up to K = {p.ko * 16}")
        out = data.new_empty((p.n, oc, p.oh, p.ow), dtype=torch.int32)
        check(L.unit_conv2d_nchwc_s8s8s32_fused_prepared_nchw(p.ref, data.data_ptr(), kernel.buf.data_ptr(), bias_ptr, scale,
                                                              out.data_ptr(), oc, _stream()))
        return out
    out = data.new_empty(p.blocked, dtype=torch.int32)
    if prepared:
        check(L.unit_conv2d_nchwc_s8s8s32_fused_prepared(p.ref, data.data_ptr(), kernel.buf.data_ptr(), bias_ptr, scale,
                                                         out.data_ptr(), _stream()))
    else:
        check(L.unit_conv2d_nchwc_s8s8s32_fused(p.ref, data.data_ptr(), kernel.data_ptr(), bias_ptr, scale, out.data_ptr(),
                                                _stream()))
    return out


def conv2d_NCHWc_int8_requant(data, kernel, bias, scale, shift, stride, padding, dilation=1):
    """u8 x s8 convolution whose output is requantised to u8 in the blocked layout the next
    convolution reads (four times less output traffic than int32):

        q = clamp(((conv(data, kernel)[k] + bias[k]) * scale + 2**(shift - 1)) >> shift, 0, 255)

    data   uint8 (N, C/cb, H, W, cb)
    kernel a PreparedConvWeight (prepare_conv2d_weight), or the blocked int8 kernel (prepared here)
    bias   int32 (K,) or None;  scale int32;  shift 1..62
    returns uint8 (N, K/16, OH, OW, 16)

    The reference's graphs stop at the int32 subtract / add / multiply
    (apps/cpu/relay/result.log:15-24); this is the integer requantisation that follows it in a
    quantised network.
    """
    out = _native.conv_requant(data, kernel, bias, scale, shift, stride, padding, dilation)
    if out is not None:
        return out
    data = _dev(data, "data", torch.uint8, 5)
    if not isinstance(kernel, PreparedConvWeight):
        kernel = prepare_conv2d_weight(kernel)
    _check_prepared(kernel, data, torch.int8)
    p = _plan(data, kernel, stride, padding, dilation)
    bias_ptr = None
    if bias is not None:
        bias = _check_bias(bias, p.ko * 16, data)
        bias_ptr = bias.data_ptr()
    scale, shift = int(scale), int(shift)
    if not -2 ** 31 <= scale < 2 ** 31:
        raise ValueError("scale: must fit int32")
    out = data.new_empty(p.blocked)
    check(_lib.load().unit_conv2d_nchwc_u8s8u8_requant_prepared(p.ref, data.data_ptr(), kernel.buf.data_ptr(), bias_ptr, scale,
                                                                shift, out.data_ptr(), _stream()))
    return out


@lru_cache(maxsize=1024, typed=True)
def _plan_3d(dshape, kshape, stride):
    n, cc, dd, h, w, cb = dshape
    ko, cc2, kd, kh, kw, e, kb, i4 = kshape
    if cb not in (4, 16) or (cb == 4 and (cc * cb) % 16 == 0):
        raise ValueError(f"data: channel block must be 16, or 4 when C is not a multiple of 16 (got {cb}, C = {cc * cb})")
    if (cc2, e, kb, i4) != (cc, cb // 4, 16, 4):
        raise ValueError(f"kernel: shape {tuple(kshape)} does not match data {tuple(dshape)}; "
                         f"expected (K/16, {cc}, KD, KH, KW, {cb // 4}, 16, 4)")
    if stride <= 0 or kd > dd or kh > h or kw > w:
        raise ValueError("stride must be positive and the kernel window must fit the input")
    d = _lib.Conv3dDesc(n, cc * cb, dd, h, w, ko * 16, kd, kh, kw, stride)
    return d, ctypes.byref(d), (n, ko, (dd - kd) // stride + 1, (h - kh) // stride + 1, (w - kw) // stride + 1, 16)


def conv3d_NCDHWc_int8(data, kernel, stride=1):
    """The 3-D blocked convolution of apps/cpu/kernel/conv3d.py:39-64: valid, one stride for depth,
    height and width, int8 x int8 -> int32 (its te.compute casts both placeholders from int8).

    data   int8  (N, C/cb, D, H, W, cb), cb = 16, or 4 with KW <= 8 (the file's 3 -> 4 channel workload)
    kernel int8  (K/16, C/cb, KD, KH, KW, cb/4, 16, 4)
    returns int32 (N, K/16, OD, OH, OW, 16)
    """
    out = _native.conv3d(data, kernel, stride)
    if out is not None:
        return out
    data = _dev(data, "data", torch.int8, 6)
    kernel = _dev(kernel, "kernel", torch.int8, 8)
    _, ref, shape = _plan_3d(data.shape, kernel.shape, int(stride))
    out = data.new_empty(shape, dtype=torch.int32)
    check(_lib.load().unit_conv3d_ncdhwc_s8s8s32(ref, data.data_ptr(), kernel.data_ptr(), out.data_ptr(), _stream()))
    return out


def dense_dotprod(data, weight, bias=None, out_dtype="int32"):
    """u8 (M, K) x s8 packed (N/128, K/4, 128, 4) -> i32 (M, N) = data . W^T.
    A 2-D weight (N, K) is taken as the un-packed relay.nn.dense operand."""
    if bias is None and out_dtype == "int32" and not isinstance(weight, PreparedDenseWeight):
        out = _native.dense(data, weight)
        if out is not None:
            return out
    data = _dev(data, "data", torch.uint8, 2)
    weight = _dev(weight, "weight", torch.int8, (2, 4))
    if out_dtype != "int32":
        raise ValueError(f"out_dtype: only 'int32' is supported, got {out_dtype!r}")
    m, k = data.shape
    L = _lib.load()
    if weight.dim() == 4:
        nb, kg, t, four = weight.shape
        if (t, four) != (128, 4) or kg * 4 != k:
            raise ValueError(f"weight: expected (N/128, {k // 4}, 128, 4), got {tuple(weight.shape)}")
        n = nb * 128
        out = data.new_empty((m, n), dtype=torch.int32)
        check(L.unit_dense_dotprod_u8s8s32(data.data_ptr(), weight.data_ptr(), out.data_ptr(), m, n, k, _stream()))
    else:
        n, k2 = weight.shape
        if k2 != k:
            raise ValueError(f"weight: expected (N, {k}), got {tuple(weight.shape)}")
        out = data.new_empty((m, n), dtype=torch.int32)
        check(L.unit_dense_u8s8s32(data.data_ptr(), weight.data_ptr(), out.data_ptr(), m, n, k, _stream()))
    if bias is not None:
        out += _dev(bias, "bias", torch.int32)
    return out


class PreparedDenseWeight:
    """A dense weight (N, K) s8 with its row sums, computed once by `prepare_dense_weight`: the constant part of the
    u8 -> s8 shift, which the reference's compiled graphs fold the same way (apps/cpu/relay/result.log:15-16)."""

    def __init__(self, w, wsum):
        self.w, self.wsum = w, wsum
        self.shape = tuple(w.shape)


def prepare_dense_weight(weight):
    """(N, K) s8 -> PreparedDenseWeight, accepted by `dense`."""
    weight = _dev(weight, "weight", torch.int8, 2)
    n, k = weight.shape
    wsum = torch.empty((n,), dtype=torch.int32, device=weight.device)
    check(_lib.load().unit_dense_prepare_weight(weight.data_ptr(), wsum.data_ptr(), n, k, _stream()))
    return PreparedDenseWeight(weight, wsum)


def dense(data, weight, out_dtype="int32"):
    """relay.nn.dense(x u8 (M, K), w s8 (N, K)) -> i32 (M, N); `weight` may be a PreparedDenseWeight."""
    if out_dtype == "int32":
        out = _native.dense(data, weight) if not isinstance(weight, torch.Tensor) or weight.dim() == 2 else None
        if out is not None:
            return out
    if isinstance(weight, PreparedDenseWeight):
        data = _dev(data, "data", torch.uint8, 2)
        if out_dtype != "int32":
            raise ValueError(f"out_dtype: only 'int32' is supported, got {out_dtype!r}")
        m, k = data.shape
        n, k2 = weight.shape
        if k2 != k:
            raise ValueError(f"weight: expected (N, {k}), got {weight.shape}")
        out = data.new_empty((m, n), dtype=torch.int32)
        check(_lib.load().unit_dense_u8s8s32_prepared(data.data_ptr(), weight.w.data_ptr(), weight.wsum.data_ptr(),
                                                      out.data_ptr(), m, n, k, _stream()))
        return out
    weight = _dev(weight, "weight", torch.int8, 2)
    return dense_dotprod(data, weight, None, out_dtype)


# ------------------------------------------------------------------------------- fp16
class PreparedGemmB:
    """The b operand of gemm_fp16 re-laid once as (N, K) (see prepare_gemm_b)."""

    def __init__(self, bt, K, N):
        self.bt, self.K, self.N = bt, K, N

    def __repr__(self):
        return f"PreparedGemmB(K={self.K}, N={self.N})"


def prepare_gemm_b(b):
    """Re-lay the constant operand b (K, N) of gemm_fp16 once as (N, K), the counterpart of the one-time
    packing of b in apps/gpu/gemm-pack.py:9,17; gemm_fp16 accepts the result in place of b.  A 4-D b is taken
    as that file's packed operand (N/32, K/32, 32, 32)."""
    b = _dev(b, "b", torch.float16, (2, 4))
    if b.dim() == 4:  # already packed as the reference packs it: (N/32, K/32, 32, 32), [y/32][k/32][k%32][y%32]
        nb, kb, k32, n32 = b.shape
        if (k32, n32) != (32, 32):
            raise ValueError(f"b: a packed operand is (N/32, K/32, 32, 32), got {tuple(b.shape)}")
        k, n = kb * 32, nb * 32
        bt = torch.empty((n, k), dtype=torch.float16, device=b.device)
        check(_lib.load().unit_gemm_f16_prepare_b_packed32(b.data_ptr(), bt.data_ptr(), k, n, _stream()))
        return PreparedGemmB(bt, k, n)
    k, n = b.shape
    bt = torch.empty((n, k), dtype=torch.float16, device=b.device)
    check(_lib.load().unit_gemm_f16_prepare_b(b.data_ptr(), bt.data_ptr(), k, n, _stream()))
    return PreparedGemmB(bt, k, n)


def gemm_fp16(a, b, out_dtype="float32", workspace=None):
    """c[x, y] = sum_k f32(a[x, k]) * f32(b[k, y]); a (M, K), b (K, N) fp16 row-major, or b a
    PreparedGemmB, or b packed (N/32, K/32, 32, 32) with b4[y/32][k/32][k%32][y%32] = b[k][y] as
    apps/gpu/gemm-pack.py:9,14-18 takes it (re-laid on every call: prepare it once instead).
    workspace (b (K, N) only): True, or a uint8 tensor of `gemm_fp16_workspace_bytes(M, N, K)` bytes: k-splits keep
    their partial tiles in it and are added in split order (run-to-run identical results, also for float16 output)."""
    if out_dtype == "float32" or out_dtype == "float16":
        out = _native.gemm(a, b, out_dtype == "float16", workspace)
        if out is not None:
            return out
    a = _dev(a, "a", torch.float16, 2)
    if out_dtype not in ("float32", "float16"):
        raise ValueError(f"out_dtype: expected 'float32' or 'float16', got {out_dtype!r}")
    m, k = a.shape
    half = out_dtype == "float16"
    if isinstance(b, torch.Tensor) and b.dim() == 4:
        b = prepare_gemm_b(b)
    if isinstance(b, PreparedGemmB):
        if b.K != k or b.bt.device != a.device:
            raise ValueError(f"b: {b!r} does not match a {tuple(a.shape)} on {a.device}")
        out = a.new_empty((m, b.N), dtype=torch.float16 if half else torch.float32)
        check(_lib.load().unit_gemm_f16_prepared(a.data_ptr(), b.bt.data_ptr(), out.data_ptr(), m, b.N, k, int(half),
                                                 _stream()))
        return out
    b = _dev(b, "b", torch.float16, 2)
    k2, n = b.shape
    if k2 != k:
        raise ValueError(f"b: expected ({k}, N), got {tuple(b.shape)}")
    out = a.new_empty((m, n), dtype=torch.float16 if half else torch.float32)
    if workspace is not None and workspace is not False:
        need = gemm_fp16_workspace_bytes(m, n, k)
        if workspace is True:
            workspace = torch.empty((max(need, 16),), dtype=torch.uint8, device=a.device)
        workspace = _dev(workspace, "workspace", torch.uint8)
        check(_lib.load().unit_gemm_f16_ws(a.data_ptr(), b.data_ptr(), out.data_ptr(), m, n, k, int(half),
                                           workspace.data_ptr(), workspace.numel(), _stream()))
        return out
    check(_lib.load().unit_gemm_f16(a.data_ptr(), b.data_ptr(), out.data_ptr(), m, n, k, int(half), _stream()))
    return out


def gemm_fp16_workspace_bytes(m, n, k):
    """Bytes `gemm_fp16(..., workspace=...)` needs for this shape (0: the shape runs without k-splits)."""
    nbytes = ctypes.c_size_t()
    check(_lib.load().unit_gemm_f16_ws_bytes(m, n, k, ctypes.byref(nbytes)))
    return nbytes.value


def conv2d_NCHW16c_OHWI16o(a, b, stride_h, stride_w, out_type="float32"):
    """fp16 valid convolution (no padding argument: callers pre-pad), fp32 accumulate.

    Either a (N, C, H, W) + b (K, C, KH, KW), packed here exactly as the reference operator packs
    them in-op, or a (N, C/16, H, W, 16) + b (K/16, C/16, KH, KW, 16 in, 16 out).
    Returns float32 (N, K/16, OH, OW, 16)."""
    if out_type != "float32":
        raise ValueError(f"out_type: only 'float32' is supported, got {out_type!r}")
    out = _native.conv_f16(a, b, stride_h, stride_w)
    if out is not None:
        return out
    a = _dev(a, "a", torch.float16, (4, 5))
    L = _lib.load()
    if isinstance(b, PreparedConvWeight):
        if a.dim() != 5:
            raise ValueError("a: prepared weights take the blocked (N, C/16, H, W, 16) operand")
        _check_prepared(b, a, torch.float16)
        p = _plan_f16(a.shape, b.key, int(stride_h), int(stride_w))
        out = a.new_empty(p.blocked, dtype=torch.float32)
        check(L.unit_conv2d_nchw16c_f16f32_prepared(p.ref, a.data_ptr(), b.buf.data_ptr(), out.data_ptr(), _stream()))
        return out
    b = _dev(b, "b", torch.float16, (4, 6))
    if a.dim() == 4 and b.dim() == 4:
        p, need = _plan_f16_plain(a.shape, b.shape, int(stride_h), int(stride_w))
        if need:
            ws = a.new_empty((need,), dtype=torch.uint8)
            out = a.new_empty(p.blocked, dtype=torch.float32)
            check(L.unit_conv2d_nchw_f16f32(p.ref, a.data_ptr(), b.data_ptr(), out.data_ptr(), ws.data_ptr(), need, _stream()))
            return out
        a, b = pack_nchwc(a, 16), prepack_conv_weight_f16(b)
    if not (a.dim() == 5 and b.dim() == 6):
        raise ValueError("a, b: expected 4-D + 4-D or 5-D + 6-D operands")
    p = _plan_f16(a.shape, b.shape, int(stride_h), int(stride_w))
    out = a.new_empty(p.blocked, dtype=torch.float32)
    check(L.unit_conv2d_nchw16c_f16f32(p.ref, a.data_ptr(), b.data_ptr(), out.data_ptr(), _stream()))
    return out


@lru_cache(maxsize=1024, typed=True)
def _plan_f16_plain(ashape, bshape, stride_h, stride_w):
    n, c, h, w = ashape
    k, c2, kh, kw = bshape
    if c % 16 or k % 16 or c2 != c:
        raise ValueError("a, b: channel counts must match and be multiples of 16")
    p = _ConvPlan(n, c, h, w, k, kh, kw, (stride_h, stride_w), 0, 1, 16)
    need = ctypes.c_size_t()
    if -(-k // 32) * 64 * c * kh * kw > 2 ** 31 - 1:  # the prepared form fills 32-channel blocks: past the size limit
        return p, 0
    check(_lib.load().unit_conv2d_nchw_f16f32_ws_bytes(p.ref, ctypes.byref(need)))
    return p, need.value


# ------------------------------------------------------------------------------- layouts
_ELEM = {torch.uint8: 1, torch.int8: 1, torch.float16: 2, torch.int32: 4, torch.float32: 4}


def _elem(t, name):
    if t.dtype not in _ELEM:
        raise TypeError(f"{name}: unsupported dtype {t.dtype}")
    return _ELEM[t.dtype]


def pack_nchwc(x, cb):
    """layout_transform NCHW -> NCHW{cb}c; channels are zero-padded up to a multiple of cb."""
    x = _dev(x, "x", None, 4)
    n, c, h, w = x.shape
    out = torch.empty((n, -(-c // cb), h, w, cb), dtype=x.dtype, device=x.device)
    check(_lib.load().unit_pack_nchwc(x.data_ptr(), out.data_ptr(), n, c, h, w, cb, _elem(x, "x"), _stream()))
    return out


def unpack_nchwc(x, channels=None):
    """layout_transform NCHW{cb}c -> NCHW, keeping the first `channels` channels."""
    x = _dev(x, "x", None, 5)
    n, cc, h, w, cb = x.shape
    c = cc * cb if channels is None else int(channels)
    if not 0 < c <= cc * cb or -(-c // cb) != cc:
        raise ValueError(f"channels: {c} does not fit {cc} blocks of {cb}")
    out = torch.empty((n, c, h, w), dtype=x.dtype, device=x.device)
    check(_lib.load().unit_unpack_nchwc(x.data_ptr(), out.data_ptr(), n, c, h, w, cb, _elem(x, "x"), _stream()))
    return out


def prepack_conv_weight(w, cb):
    """int8 OIHW -> (ceil(O/16), ceil(I/cb), KH, KW, cb/4, 16, 4), zero-padded."""
    w = _dev(w, "w", torch.int8, 4)
    o, i, kh, kw = w.shape
    if cb not in (4, 16):
        raise ValueError(f"cb: must be 16 or 4, got {cb}")
    out = torch.empty((-(-o // 16), -(-i // cb), kh, kw, cb // 4, 16, 4), dtype=torch.int8, device=w.device)
    check(_lib.load().unit_prepack_conv_weight_s8(w.data_ptr(), out.data_ptr(), o, i, kh, kw, cb, _stream()))
    return out


def prepack_dense_weight(w):
    """int8 (N, K) -> (N/128, K/4, 128, 4)."""
    w = _dev(w, "w", torch.int8, 2)
    n, k = w.shape
    if n % 128 or k % 4:
        raise ValueError(f"w: N must be a multiple of 128 and K of 4, got {tuple(w.shape)}")
    out = torch.empty((n // 128, k // 4, 128, 4), dtype=torch.int8, device=w.device)
    check(_lib.load().unit_prepack_dense_weight_s8(w.data_ptr(), out.data_ptr(), n, k, _stream()))
    return out


def prepack_conv_weight_f16(w):
    """fp16 OIHW -> (O/16, I/16, KH, KW, 16 in, 16 out)."""
    w = _dev(w, "w", torch.float16, 4)
    o, i, kh, kw = w.shape
    if o % 16 or i % 16:
        raise ValueError(f"w: O and I must be multiples of 16, got {tuple(w.shape)}")
    out = torch.empty((o // 16, i // 16, kh, kw, 16, 16), dtype=torch.float16, device=w.device)
    check(_lib.load().unit_prepack_conv_weight_f16(w.data_ptr(), out.data_ptr(), o, i, kh, kw, _stream()))
    return out

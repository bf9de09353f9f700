"""ctypes binding of librnn_hip.so (include/rnn_hip.h) for Python callers.

Tensors are torch tensors already resident on the GPU (torch is used only for
device memory and the current stream). Every call goes through the C ABI; a
non-zero status raises RnnError carrying rnn_last_error(). There is no CPU
fallback: if the library is missing, load() raises.
"""
from __future__ import annotations

import ctypes
import os
import re

import torch

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "librnn_hip.so")
HEADER = os.path.join(os.path.dirname(HERE), "include", "rnn_hip.h")

RNN_OK = 0
RNN_ERR_INVALID_ARG = 1
RNN_ERR_HIP = 2
RNN_ERR_UNSUPPORTED = 3
RNN_ERR_OUT_OF_MEMORY = 4

FLAG_RELU = 0x1
ALGO_AUTO = 0x00
ALGO_TILED = 0x10
ALGO_GEMV = 0x20
ALGO_TILED_DMA = 0x30
ALGO_GEMV_MFMA = 0x40
ALGO_GEMV_BF16 = 0x50
FLAG_TERNARY_MFMA_LAYOUT = 0x100

TERNARY_ROWS = 0
TERNARY_ABSMEAN = 1

# QuantFormat (src/quantize.rs:37-56), declaration order
QF_FP16, QF_BF16, QF_INT8, QF_INT4, QF_NF4, QF_NVFP4, QF_GGUF_Q4, QF_GGUF_Q4K, QF_GGUF_Q8 = range(9)

# blas::Transpose (src/blas.rs:72-77)
NO_TRANS = 0
TRANS = 1


class RnnError(RuntimeError):
    def __init__(self, status: int, msg: str):
        super().__init__(f"[rnn status {status}] {msg}")
        self.status = status


_P = ctypes.c_void_p
_I64 = ctypes.c_int64
_INT = ctypes.c_int
_UINT = ctypes.c_uint

# name -> (argtypes, restype)
SIGNATURES = {
    "rnn_abi_version": ([], _INT),
    "rnn_last_error": ([], ctypes.c_char_p),
    "rnn_quant_rows_i8": ([_P, _I64, _I64, _P, _P, _P], _INT),
    "rnn_int8_dequantize": ([_P, _P, _I64, _I64, _P, _P], _INT),
    "rnn_int8_matmul_f32": ([_P, _P, _I64, _I64, _P, _I64, _P, _P], _INT),
    "rnn_int8_linear_forward": ([_P, _I64, _I64, _P, _P, _I64, _P, _P, _P], _INT),
    "rnn_igemm_workspace_size": ([_I64, _I64, _I64], ctypes.c_size_t),
    "rnn_igemm": ([_P, _P, _P, _I64, _I64, _I64, _P, ctypes.c_size_t, _P], _INT),
    "rnn_igemm_noalloc": ([_P, _P, _P, _I64, _I64, _I64, _P], _INT),
    "rnn_w8a8_linear": ([_P, _P, _P, _P, _P, _I64, _I64, _I64, _UINT, _P, _P, _P], _INT),
    "rnn_w8a8_forward": ([_P, _I64, _I64, _P, _P, _P, _I64, _UINT, _P, _P, ctypes.c_size_t, _P], _INT),
    "rnn_ternary_forward": ([_P, _I64, _I64, _P, _P, _P, _I64, _UINT, _P, _P, ctypes.c_size_t, _P],
                            _INT),
    "rnn_ternary_pack": ([_P, _I64, _P, _P], _INT),
    "rnn_ternary_unpack": ([_P, _I64, _P, _P], _INT),
    "rnn_ternary_quantize": ([_P, _I64, _I64, _INT, _P, _P, _P], _INT),
    "rnn_ternary_dequantize": ([_P, _I64, _P, _I64, _I64, _P, _P], _INT),
    "rnn_ternary_linear_forward": ([_P, _I64, _I64, _P, _P, _I64, _P, _P, _P], _INT),
    "rnn_ternary_gemm": ([_P, _P, _P, _P, _P, _I64, _I64, _I64, _UINT, _P, _P, _P], _INT),
    "rnn_ternary_prepack": ([_P, _I64, _I64, _P, _P], _INT),
    "rnn_rotor_rotation_matrices": ([_P, _I64, _P, _P], _INT),
    "rnn_rotorquant_quantize": ([_P, _I64, _I64, _INT, _P, _P, _P, _P, _P], _INT),
    "rnn_rotorquant_dequantize": ([_P, _P, _I64, _I64, _P, _P, _P], _INT),
    "rnn_qt_layout": ([_INT, _I64, _I64, _P, _P, _P], _INT),
    "rnn_qt_quantize": ([_INT, _P, _I64, _I64, _P, _P, _P], _INT),
    "rnn_qt_dequantize": ([_INT, _P, _I64, _P, _I64, _I64, _I64, _P, _P], _INT),
    "rnn_qt_linear_forward": ([_INT, _P, _I64, _I64, _P, _I64, _P, _I64, _I64, _I64, _P, _P,
                               _UINT, _P], _INT),
    "rnn_qt_linear_workspace_size": ([_I64, _I64], ctypes.c_size_t),
    "rnn_rotorquant_kv_attention_workspace_size": ([_I64, _I64, _I64, _I64], ctypes.c_size_t),
    "rnn_rotorquant_kv_attention_ws": ([_P, _I64, _I64, _P, _P, _P, _P, _P, _P, _I64, _I64,
                                        ctypes.c_float, _P, _P, ctypes.c_size_t, _P], _INT),
    "rnn_qt_linear_forward_ws": ([_INT, _P, _I64, _I64, _P, _I64, _P, _I64, _I64, _I64, _P, _P,
                                  _P, ctypes.c_size_t, _UINT, _P], _INT),
    "rnn_qt_linear_scratch_size": ([_INT, _I64, _I64, _P, _P, _I64, _I64, _I64], ctypes.c_size_t),
    "rnn_qt_linear_forward_scratch": ([_INT, _P, _I64, _I64, _P, _I64, _P, _I64, _I64, _I64, _P, _P,
                                       _P, ctypes.c_size_t, _P, ctypes.c_size_t, _UINT, _P], _INT),
    "rnn_rotorquant_kv_page_elems": ([_I64, _I64, _I64, _P, _P], _INT),
    "rnn_rotorquant_kv_pack": ([_P, _P, _I64, _I64, _I64, _INT, _INT, _P, _P, _P], _INT),
    "rnn_rotorquant_kv_attention": ([_P, _I64, _I64, _P, _P, _P, _P, _P, _P, _I64, _I64,
                                     ctypes.c_float, _P, _P], _INT),
    "rnn_sgemm": ([_INT, _INT, _I64, _I64, _I64, ctypes.c_float, _P, _I64, _P, _I64,
                   ctypes.c_float, _P, _I64, _P], _INT),
    "rnn_relu": ([_P, _I64, _P, _P], _INT),
    "rnn_w8a8_mlp": ([_P, _I64, _INT, _P, _P, _P, _P, _INT, _P, _P], _INT),
    "rnn_bias_act": ([_P, _P, _I64, _I64, _INT, _P], _INT),
    "rnn_linear_layer": ([_P, _I64, _I64, _P, _I64, _P, _INT, _P, _P], _INT),
    "rnn_linear_layer_workspace_size": ([_P, _I64, _I64, _I64], ctypes.c_size_t),
    "rnn_linear_layer_ws": ([_P, _I64, _I64, _P, _I64, _P, _INT, _P, _P, ctypes.c_size_t, _P], _INT),
}

_lib = None


def header_symbols() -> list[str]:
    """Function names declared in include/rnn_hip.h."""
    text = open(HEADER).read()
    return sorted(set(re.findall(r"^\s*(?:const\s+)?[\w\s\*]+?\b(rnn_\w+)\s*\(", text, re.M)))


def load():
    """Load librnn_hip.so (raises if it has not been built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RnnError(RNN_ERR_UNSUPPORTED,
                           f"{LIB_PATH} is missing: run rust-neural-network_amd/build.py")
        L = ctypes.CDLL(LIB_PATH)
        for name, (args, res) in SIGNATURES.items():
            fn = getattr(L, name)
            fn.argtypes = args
            fn.restype = res
        _lib = L
    return _lib


def last_error() -> str:
    return load().rnn_last_error().decode()


def _check(status: int):
    if status != RNN_OK:
        raise RnnError(status, last_error())


def _ptr(t):
    return None if t is None else t.data_ptr()


# The current stream's handle without building a Stream object (2.8 -> 0.1 us
# a call); torch versions without these names take the public one.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_raw_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream(stream):
    if stream is not None:
        return stream.cuda_stream
    if _raw_stream is None or _raw_device is None:
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(_raw_device())


def _dev(t, dtype, name):
    if t is None:
        return None
    if not t.is_cuda:
        raise RnnError(RNN_ERR_INVALID_ARG, f"{name} must be a device tensor")
    if t.dtype != dtype:
        raise RnnError(RNN_ERR_INVALID_ARG, f"{name} must be {dtype}, got {t.dtype}")
    if not t.is_contiguous():
        raise RnnError(RNN_ERR_INVALID_ARG, f"{name} must be contiguous")
    return t


def _need(t, n, name, at_least=False):
    """Raise unless tensor `t` (when given) holds exactly `n` elements (or at
    least `n` with at_least): a buffer shorter than the sizes passed to the C
    ABI would be read or written past its end on the device."""
    if t is None:
        return
    got = t.numel()
    if got < n or (got != n and not at_least):
        raise RnnError(RNN_ERR_INVALID_ARG,
                       f"{name} holds {got} elements, {'at least ' if at_least else ''}{n} needed")


def _out(t, dtype, n, name):
    """A caller-supplied output tensor: on the device, of `dtype`, contiguous,
    `n` elements."""
    if t is not None:
        _dev(t, dtype, name)
        _need(t, n, name)
    return t


def _dims(t, nd, name):
    if t.dim() != nd:
        raise RnnError(RNN_ERR_INVALID_ARG, f"{name} must be {nd}-D, got shape {tuple(t.shape)}")
    return tuple(t.shape)


def _empty(shape, dtype, like):
    return torch.empty(shape, dtype=dtype, device=like.device)


def _scratch(nbytes, like, stream):
    """(device bytes for one call, or None; the call's stream), from torch's
    allocator in the pool of that stream: freed at the end of the call, they
    are handed out again only to work ordered behind it."""
    if not nbytes:
        return None, _stream(stream)
    if stream is None:
        return torch.empty(nbytes, dtype=torch.uint8, device=like.device), _stream(None)
    with torch.cuda.stream(stream):
        return torch.empty(nbytes, dtype=torch.uint8, device=like.device), stream.cuda_stream


# ------------------------------------------------------------------ int8
def quant_rows_i8(x, q=None, scale=None, stream=None):
    """Per-row symmetric int8 (Int8Weights::quantize rule). Returns (q, scale)."""
    _dev(x, torch.float32, "x")
    rows, cols = _dims(x, 2, "x")
    q = _out(q, torch.int8, rows * cols, "q") if q is not None else _empty((rows, cols), torch.int8, x)
    scale = (_out(scale, torch.float32, rows, "scale") if scale is not None
             else _empty((rows,), torch.float32, x))
    _check(load().rnn_quant_rows_i8(_ptr(x), rows, cols, _ptr(q), _ptr(scale), _stream(stream)))
    return q, scale


def int8_dequantize(q, scale, stream=None):
    _dev(q, torch.int8, "q"), _dev(scale, torch.float32, "scale")
    rows, _ = _dims(q, 2, "q")
    _need(scale, rows, "scale")
    w = _empty(q.shape, torch.float32, q)
    _check(load().rnn_int8_dequantize(_ptr(q), _ptr(scale), q.shape[0], q.shape[1], _ptr(w),
                                      _stream(stream)))
    return w


def int8_matmul_f32(wq, ws, x, stream=None):
    _dev(wq, torch.int8, "wq"), _dev(ws, torch.float32, "ws"), _dev(x, torch.float32, "x")
    out_f, in_f = _dims(wq, 2, "wq")
    _need(ws, out_f, "ws")
    if in_f == 0 or x.numel() % in_f != 0:
        raise RnnError(RNN_ERR_INVALID_ARG, f"x ({x.numel()} elements) is not [m, {in_f}]")
    m = x.numel() // in_f
    y = _empty((m, out_f), torch.float32, x)
    _check(load().rnn_int8_matmul_f32(_ptr(wq), _ptr(ws), out_f, in_f, _ptr(x), m, _ptr(y),
                                      _stream(stream)))
    return y


def int8_linear_forward(x, wq, ws, bias=None, stream=None):
    _dev(x, torch.float32, "x"), _dev(wq, torch.int8, "wq"), _dev(ws, torch.float32, "ws")
    _dev(bias, torch.float32, "bias")
    batch, in_f = _dims(x, 2, "x")
    out_f, w_in = _dims(wq, 2, "wq")
    if w_in != in_f:
        raise RnnError(RNN_ERR_INVALID_ARG, f"x has {in_f} features, wq expects {w_in}")
    _need(ws, out_f, "ws"), _need(bias, out_f, "bias")
    y = _empty((batch, out_f), torch.float32, x)
    _check(load().rnn_int8_linear_forward(_ptr(x), batch, in_f, _ptr(wq), _ptr(ws), out_f,
                                          _ptr(bias), _ptr(y), _stream(stream)))
    return y


def igemm_workspace_size(m, k, n) -> int:
    return int(load().rnn_igemm_workspace_size(m, k, n))


def igemm(a_u8, b_i8, m, k, n, workspace=None, c=None, stream=None):
    """igemm contract: a u8 [m,k], b i8 [k,n] -> c i32 [m,n]."""
    _dev(a_u8, torch.uint8, "a"), _dev(b_i8, torch.int8, "b")
    if min(m, k, n) < 0:
        raise RnnError(RNN_ERR_INVALID_ARG, f"negative size m={m} k={k} n={n}")
    _need(a_u8, m * k, "a"), _need(b_i8, k * n, "b")
    c = _out(c, torch.int32, m * n, "c") if c is not None else _empty((m, n), torch.int32, a_u8)
    if workspace is not None and not (workspace.is_cuda and workspace.is_contiguous()):
        raise RnnError(RNN_ERR_INVALID_ARG, "workspace must be a contiguous device tensor")
    wsb = 0 if workspace is None else workspace.numel() * workspace.element_size()
    _check(load().rnn_igemm(_ptr(a_u8), _ptr(b_i8), _ptr(c), m, k, n, _ptr(workspace), wsb,
                            _stream(stream)))
    return c


IGEMM_NOALLOC_MAX_BYTES = 64 << 20  # RNN_IGEMM_NOALLOC_MAX_BYTES


def igemm_noalloc(a_u8, b_i8, m, k, n, c, stream=None):
    """igemm into a caller-allocated c (int32 [m, n]) with the library's
    device-array workspace: no allocation anywhere in the call."""
    _dev(a_u8, torch.uint8, "a"), _dev(b_i8, torch.int8, "b")
    if min(m, k, n) < 0:
        raise RnnError(RNN_ERR_INVALID_ARG, f"negative size m={m} k={k} n={n}")
    _need(a_u8, m * k, "a"), _need(b_i8, k * n, "b"), _out(c, torch.int32, m * n, "c")
    _check(load().rnn_igemm_noalloc(_ptr(a_u8), _ptr(b_i8), _ptr(c), m, k, n, _stream(stream)))
    return c


def w8a8_linear(aq, sa, wq, sw, bias=None, relu=False, algo=ALGO_AUTO, want_y=True,
                want_acc=False, y=None, acc=None, stream=None):
    """Returns (y f32 [m,n] or None, acc i32 [m,n] or None)."""
    _dev(aq, torch.int8, "aq"), _dev(wq, torch.int8, "wq")
    _dev(sa, torch.float32, "sa"), _dev(sw, torch.float32, "sw"), _dev(bias, torch.float32, "bias")
    m, k = _dims(aq, 2, "aq")
    n, wk = _dims(wq, 2, "wq")
    if wk != k:
        raise RnnError(RNN_ERR_INVALID_ARG, f"aq has k={k}, wq has k={wk}")
    _need(sa, m, "sa"), _need(sw, n, "sw"), _need(bias, n, "bias")
    _out(y, torch.float32, m * n, "y"), _out(acc, torch.int32, m * n, "acc")
    if want_y and y is None:
        y = _empty((m, n), torch.float32, aq)
    if want_acc and acc is None:
        acc = _empty((m, n), torch.int32, aq)
    flags = (FLAG_RELU if relu else 0) | algo
    _check(load().rnn_w8a8_linear(_ptr(aq), _ptr(sa), _ptr(wq), _ptr(sw), _ptr(bias), m, k, n,
                                  flags, _ptr(y), _ptr(acc), _stream(stream)))
    return y, acc


def w8a8_forward(x, wq, sw, bias=None, relu=False, stream=None):
    """quant_rows_i8 + w8a8_linear in one call (the codes and scales of x in
    the call's scratch): y [m, n] f32 of x [m, k] f32."""
    _dev(x, torch.float32, "x"), _dev(wq, torch.int8, "wq"), _dev(sw, torch.float32, "sw")
    _dev(bias, torch.float32, "bias")
    m, k = _dims(x, 2, "x")
    n, wk = _dims(wq, 2, "wq")
    if wk != k:
        raise RnnError(RNN_ERR_INVALID_ARG, f"x has k={k}, wq has k={wk}")
    _need(sw, n, "sw"), _need(bias, n, "bias")
    y = _empty((m, n), torch.float32, x)
    need = (m * k + 15) // 16 * 16 + 4 * m
    ws, s = _scratch(need, x, stream)
    _check(load().rnn_w8a8_forward(_ptr(x), m, k, _ptr(wq), _ptr(sw), _ptr(bias), n,
                                   FLAG_RELU if relu else 0, _ptr(y), _ptr(ws), need, s))
    return y


def w8a8_mlp(x, layers, relu=True, y=None, stream=None):
    """A chain of W8A8 layers in one launch (rnn_w8a8_mlp): `layers` is a list
    of (wq [n, k] int8, sw [n] f32, bias [n] f32 or None); x [m, k0] f32.
    Bit-identical to quant_rows_i8 + w8a8_linear per layer, ReLU between
    layers when `relu`. Raises RnnError (RNN_ERR_UNSUPPORTED) for chains the
    single launch does not take (more than 4 layers, widths over 1024,
    in-features not a multiple of 16)."""
    _dev(x, torch.float32, "x")
    m, k0 = _dims(x, 2, "x")
    nl = len(layers)
    dims = [k0]
    for i, (wq, sw, b) in enumerate(layers):
        _dev(wq, torch.int8, f"wq[{i}]"), _dev(sw, torch.float32, f"sw[{i}]")
        _dev(b, torch.float32, f"bias[{i}]")
        n, k = _dims(wq, 2, f"wq[{i}]")
        if k != dims[-1]:
            raise RnnError(RNN_ERR_INVALID_ARG, f"layer {i} takes {k} features, gets {dims[-1]}")
        _need(sw, n, f"sw[{i}]"), _need(b, n, f"bias[{i}]")
        dims.append(n)
    y = (_out(y, torch.float32, m * dims[-1], "y") if y is not None
         else _empty((m, dims[-1]), torch.float32, x))
    d = (ctypes.c_int64 * (nl + 1))(*dims)
    w = (ctypes.c_void_p * nl)(*[l[0].data_ptr() for l in layers])
    s_ = (ctypes.c_void_p * nl)(*[l[1].data_ptr() for l in layers])
    b_ = (ctypes.c_void_p * nl)(*[0 if l[2] is None else l[2].data_ptr() for l in layers])
    _check(load().rnn_w8a8_mlp(_ptr(x), m, nl, d, w, s_, b_, int(bool(relu)), _ptr(y),
                               _stream(stream)))
    return y


# ------------------------------------------------------------------ ternary
def ternary_pack(t, stream=None):
    _dev(t, torch.int8, "t")
    count = t.numel()
    packed = _empty(((count + 15) // 16,), torch.int32, t)
    _check(load().rnn_ternary_pack(_ptr(t), count, _ptr(packed), _stream(stream)))
    return packed


def ternary_unpack(packed, count, stream=None):
    _dev(packed, torch.int32, "packed")
    _need(packed, (count + 15) // 16, "packed", at_least=True)
    t = _empty((count,), torch.int8, packed)
    _check(load().rnn_ternary_unpack(_ptr(packed), count, _ptr(t), _stream(stream)))
    return t


def ternary_quantize(w, mode=TERNARY_ROWS, stream=None):
    """Returns (packed int32 words [ceil(numel/16)], scales f32 [rows])."""
    _dev(w, torch.float32, "w")
    rows, cols = _dims(w, 2, "w")
    packed = _empty(((rows * cols + 15) // 16,), torch.int32, w)
    scales = _empty((rows,), torch.float32, w)
    _check(load().rnn_ternary_quantize(_ptr(w), rows, cols, mode, _ptr(packed), _ptr(scales),
                                       _stream(stream)))
    return packed, scales


def ternary_dequantize(packed, numel, scales, cols, stream=None):
    _dev(packed, torch.int32, "packed"), _dev(scales, torch.float32, "scales")
    _need(packed, (numel + 15) // 16, "packed", at_least=True)
    w = _empty((numel,), torch.float32, packed)
    _check(load().rnn_ternary_dequantize(_ptr(packed), numel, _ptr(scales), scales.numel(), cols,
                                         _ptr(w), _stream(stream)))
    return w


def ternary_linear_forward(x, packed, scales, out_f, bias=None, stream=None):
    _dev(x, torch.float32, "x"), _dev(packed, torch.int32, "packed")
    _dev(scales, torch.float32, "scales"), _dev(bias, torch.float32, "bias")
    batch, in_f = _dims(x, 2, "x")
    _need(packed, (out_f * in_f + 15) // 16, "packed", at_least=True)
    _need(scales, out_f, "scales", at_least=True), _need(bias, out_f, "bias")
    y = _empty((batch, out_f), torch.float32, x)
    _check(load().rnn_ternary_linear_forward(_ptr(x), batch, in_f, _ptr(packed), _ptr(scales),
                                             out_f, _ptr(bias), _ptr(y), _stream(stream)))
    return y


def ternary_prepack(packed, rows, cols, stream=None):
    """The MFMA code layout of a ternary weight [rows, cols] (cols % 16 == 0):
    same size, read by ternary_gemm(..., mfma_layout=True)."""
    _dev(packed, torch.int32, "packed")
    _need(packed, rows * cols // 16, "packed", at_least=True)
    out = _empty((rows * cols // 16,), torch.int32, packed)
    _check(load().rnn_ternary_prepack(_ptr(packed), rows, cols, _ptr(out), _stream(stream)))
    return out


def ternary_gemm(aq, sa, packed, sw, n, bias=None, relu=False, want_y=True, want_acc=False,
                 y=None, stream=None, algo=ALGO_AUTO, mfma_layout=False):
    _dev(aq, torch.int8, "aq"), _dev(packed, torch.int32, "packed")
    _dev(sa, torch.float32, "sa"), _dev(sw, torch.float32, "sw"), _dev(bias, torch.float32, "bias")
    m, k = _dims(aq, 2, "aq")
    _need(packed, (n * k + 15) // 16, "packed", at_least=True)
    _need(sa, m, "sa"), _need(sw, n, "sw"), _need(bias, n, "bias")
    _out(y, torch.float32, m * n, "y")
    if want_y and y is None:
        y = _empty((m, n), torch.float32, aq)
    acc = _empty((m, n), torch.int32, aq) if want_acc else None
    flags = (FLAG_RELU if relu else 0) | (FLAG_TERNARY_MFMA_LAYOUT if mfma_layout else 0) | algo
    _check(load().rnn_ternary_gemm(_ptr(aq), _ptr(sa), _ptr(packed), _ptr(sw), _ptr(bias), m, k,
                                   n, flags, _ptr(y), _ptr(acc), _stream(stream)))
    return y, acc


def ternary_forward(x, packed, sw, n, bias=None, relu=False, mfma_layout=False, stream=None):
    """quant_rows_i8 + ternary_gemm in one call, as w8a8_forward."""
    _dev(x, torch.float32, "x"), _dev(packed, torch.int32, "packed")
    _dev(sw, torch.float32, "sw"), _dev(bias, torch.float32, "bias")
    m, k = _dims(x, 2, "x")
    _need(packed, (n * k + 15) // 16, "packed", at_least=True)
    _need(sw, n, "sw"), _need(bias, n, "bias")
    y = _empty((m, n), torch.float32, x)
    need = (m * k + 15) // 16 * 16 + 4 * m
    ws, s = _scratch(need, x, stream)
    flags = (FLAG_RELU if relu else 0) | (FLAG_TERNARY_MFMA_LAYOUT if mfma_layout else 0)
    _check(load().rnn_ternary_forward(_ptr(x), m, k, _ptr(packed), _ptr(sw), _ptr(bias), n, flags,
                                      _ptr(y), _ptr(ws), need, s))
    return y


# ------------------------------------------------------------------ RotorQuant
def rotation_matrices(rotors, stream=None):
    _dev(rotors, torch.float32, "rotors")
    n = rotors.shape[0] if rotors.dim() > 0 else 0
    _need(rotors, 4 * n, "rotors")
    out = _empty((n, 3, 3), torch.float32, rotors)
    _check(load().rnn_rotor_rotation_matrices(_ptr(rotors), n, _ptr(out), _stream(stream)))
    return out


def rotorquant_quantize(x, rotors, bits, want_y=True, want_codes=False, y=None, stream=None):
    """Returns (y or None, codes int8 [rows,padded] or None, scales [rows,groups] or None)."""
    _dev(x, torch.float32, "x"), _dev(rotors, torch.float32, "rotors")
    dim = x.shape[-1]
    rows = x.numel() // dim if dim else 0
    ng = (dim + 2) // 3
    _need(rotors, 4 * ng, "rotors", at_least=True)
    _out(y, torch.float32, x.numel(), "y")
    if want_y and y is None:
        y = _empty(tuple(x.shape), torch.float32, x)
    codes = _empty((rows, 3 * ng), torch.int8, x) if want_codes else None
    scales = _empty((rows, ng), torch.float32, x) if want_codes else None
    _check(load().rnn_rotorquant_quantize(_ptr(x), rows, dim, bits, _ptr(rotors), _ptr(y),
                                          _ptr(codes), _ptr(scales), _stream(stream)))
    return y, codes, scales


def rotorquant_dequantize(codes, scales, dim, rotors, stream=None):
    _dev(codes, torch.int8, "codes"), _dev(scales, torch.float32, "scales")
    _dev(rotors, torch.float32, "rotors")
    ng = (dim + 2) // 3
    rows = codes.shape[0]
    _need(codes, rows * 3 * ng, "codes"), _need(scales, rows * ng, "scales")
    _need(rotors, 4 * ng, "rotors", at_least=True)
    y = _empty((rows, dim), torch.float32, codes)
    _check(load().rnn_rotorquant_dequantize(_ptr(codes), _ptr(scales), rows, dim, _ptr(rotors),
                                            _ptr(y), _stream(stream)))
    return y


# ------------------------------------------------------------------ f32 GEMM
def sgemm(transa, transb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, stream=None):
    """blas::sgemm / BlasBackend::sgemm (src/blas.rs:104-118, :712-734):
    C = alpha*op(A)*op(B) + beta*C on device storage `a`, `b`, `c` (f32
    tensors holding the row-major matrices with row strides lda/ldb/ldc).
    `transa`/`transb` are NO_TRANS or TRANS. C is updated in place."""
    for t, nm in ((a, "a"), (b, "b"), (c, "c")):
        _dev(t, torch.float32, nm)

    def span(rows, cols, ld):  # elements a row-major [rows, cols] with row stride ld reaches
        return 0 if rows == 0 or cols == 0 else (rows - 1) * ld + cols
    if m > 0 and n > 0:
        _need(c, span(m, n, ldc), "c", at_least=True)
        if k > 0 and alpha != 0.0:
            _need(a, span(k, m, lda) if transa else span(m, k, lda), "a", at_least=True)
            _need(b, span(n, k, ldb) if transb else span(k, n, ldb), "b", at_least=True)
    _check(load().rnn_sgemm(int(transa), int(transb), m, n, k, float(alpha), _ptr(a), lda,
                            _ptr(b), ldb, float(beta), _ptr(c), ldc, _stream(stream)))
    return c


def matmul(a, b, stream=None):
    """blas::matmul (src/blas.rs:780-799): C = A.B for contiguous [m,k] @ [k,n]."""
    _dev(a, torch.float32, "a"), _dev(b, torch.float32, "b")
    m, k = _dims(a, 2, "a")
    kb, n = _dims(b, 2, "b")
    if kb != k:
        raise RnnError(RNN_ERR_INVALID_ARG, f"inner dimensions differ: {k} vs {kb}")
    c = _empty((m, n), torch.float32, a)
    return sgemm(NO_TRANS, NO_TRANS, m, n, k, 1.0, a, k, b, n, 0.0, c, n, stream)


def relu(x, out=None, stream=None):
    """Tensor::relu (src/tensor.rs:2025-2032): x.max(0.0) elementwise (NaN -> 0).
    `out` may be x itself."""
    _dev(x, torch.float32, "x")
    out = _out(out, torch.float32, x.numel(), "out") if out is not None else torch.empty_like(x)
    _check(load().rnn_relu(_ptr(x), x.numel(), _ptr(out), _stream(stream)))
    return out


def bias_act(y, bias=None, relu=False, stream=None):
    """The fused bias add + activation of Tensor::linear_layer
    (src/tensor.rs:771-786), in place on y [rows, cols]."""
    _dev(y, torch.float32, "y"), _dev(bias, torch.float32, "bias")
    rows, cols = _dims(y, 2, "y")
    _need(bias, cols, "bias")
    _check(load().rnn_bias_act(_ptr(y), _ptr(bias), rows, cols, int(bool(relu)), _stream(stream)))
    return y


def linear_layer(x, w, bias=None, relu=False, out=None, stream=None):
    """Tensor::linear_layer (src/tensor.rs:747-800): act(x [batch, in] . W^T +
    b) with W stored [out, in]; bias may be None (Linear without bias)."""
    _dev(x, torch.float32, "x"), _dev(w, torch.float32, "w"), _dev(bias, torch.float32, "bias")
    batch, in_f = _dims(x, 2, "x")
    out_f, w_in = _dims(w, 2, "w")
    if w_in != in_f:
        raise RnnError(RNN_ERR_INVALID_ARG, f"x has {in_f} features, w expects {w_in}")
    _need(bias, out_f, "bias")
    out = (_out(out, torch.float32, batch * out_f, "out") if out is not None
           else _empty((batch, out_f), torch.float32, x))
    need = load().rnn_linear_layer_workspace_size(_ptr(w), batch, in_f, out_f)
    ws, s = _scratch(need, x, stream)
    _check(load().rnn_linear_layer_ws(_ptr(x), batch, in_f, _ptr(w), out_f, _ptr(bias),
                                      int(bool(relu)), _ptr(out), _ptr(ws), need, s))
    return out


class HipBackend:
    """The BlasBackend trait (src/blas.rs:712-734) on the GPU: name() and
    sgemm() with the trait's argument order, operands on the device."""

    def name(self) -> str:
        return "hip-gfx950 (v_mfma_f32_16x16x4f32, 128x128 tiles)"

    def sgemm(self, transa, transb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc):
        return sgemm(transa, transb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc)


# ------------------------------------------------------------------ QuantizedTensor
def qt_layout(fmt, n, group_size):
    """(data bytes, scales.len(), stored group_size) of QuantizedTensor::quantize
    (src/quantize.rs:231-250)."""
    out = (ctypes.c_int64 * 3)()
    base = ctypes.addressof(out)
    _check(load().rnn_qt_layout(fmt, n, group_size, ctypes.c_void_p(base),
                                ctypes.c_void_p(base + 8), ctypes.c_void_p(base + 16)))
    return int(out[0]), int(out[1]), int(out[2])


def qt_quantize(fmt, x, group_size, stream=None):
    """QuantizedTensor::quantize of the flat data of device tensor x. Returns
    (data uint8 [bytes], scales f32 [groups], stored group_size)."""
    _dev(x, torch.float32, "x")
    n = x.numel()
    nb, ns, g = qt_layout(fmt, n, group_size)
    data = _empty((nb,), torch.uint8, x)
    scales = _empty((ns,), torch.float32, x)
    _check(load().rnn_qt_quantize(fmt, _ptr(x), n, group_size, _ptr(data), _ptr(scales),
                                  _stream(stream)))
    return data, scales, g


def qt_dequantize(fmt, data, scales, group, n, stream=None):
    """QuantizedTensor::dequantize (src/quantize.rs:252-269): flat f32 [n]."""
    _dev(data, torch.uint8, "data"), _dev(scales, torch.float32, "scales")
    out = _empty((n,), torch.float32, data)
    _check(load().rnn_qt_dequantize(fmt, _ptr(data), data.numel(), _ptr(scales), scales.numel(),
                                    group, n, _ptr(out), _stream(stream)))
    return out


def qt_linear_workspace_size(in_f, out_f) -> int:
    return int(load().rnn_qt_linear_workspace_size(in_f, out_f))


def qt_linear_forward(fmt, x, data, scales, group, out_f, bias=None, algo=ALGO_AUTO, y=None,
                      stream=None, workspace=None):
    """QuantizedLinear::forward (src/quantize.rs:744-754): x [m, in] -> y [m, out].
    `workspace`: a zeroed device byte tensor of at least
    qt_linear_workspace_size(in, out) bytes for the bf16 MFMA GEMV's scratch
    (else the call allocates); calls leave it reusable. Above 16 rows the
    call's other scratch comes from torch's allocator."""
    _dev(x, torch.float32, "x"), _dev(data, torch.uint8, "data")
    _dev(scales, torch.float32, "scales"), _dev(bias, torch.float32, "bias")
    _dev(workspace, torch.uint8, "workspace")
    m, in_f = _dims(x, 2, "x")
    _need(bias, out_f, "bias")
    y = _out(y, torch.float32, m * out_f, "y") if y is not None else _empty((m, out_f), torch.float32, x)
    ws_bytes = 0 if workspace is None else workspace.numel()
    need = (load().rnn_qt_linear_scratch_size(fmt, m, in_f, _ptr(data), _ptr(scales), scales.numel(),
                                              group, out_f) if m > 16 and algo == ALGO_AUTO else 0)
    scratch, s = _scratch(need, x, stream)
    _check(load().rnn_qt_linear_forward_scratch(fmt, _ptr(x), m, in_f, _ptr(data), data.numel(),
                                                _ptr(scales), scales.numel(), group, out_f,
                                                _ptr(bias), _ptr(y), _ptr(workspace), ws_bytes,
                                                _ptr(scratch), need, algo, s))
    return y


# ------------------------------------------------------------------ RotorQuant KV cache
RQ_PAGE_K = 0
RQ_PAGE_V = 1


def rotorquant_kv_page_elems(bh, seq, dim):
    """(u16 code elements, f32 scale elements) of one page."""
    out = (ctypes.c_int64 * 2)()
    base = ctypes.addressof(out)
    _check(load().rnn_rotorquant_kv_page_elems(bh, seq, dim, ctypes.c_void_p(base),
                                               ctypes.c_void_p(base + 8)))
    return int(out[0]), int(out[1])


def rotorquant_kv_pack(codes, scales, bh, seq, dim, bits, kind, stream=None):
    """Codes/scales of rotorquant_quantize (rows = bh*seq) -> a KV-cache page
    of the given kind (RQ_PAGE_K or RQ_PAGE_V): (u16 codes as int16, f32
    scales), both flat."""
    _dev(codes, torch.int8, "codes"), _dev(scales, torch.float32, "scales")
    ng = (dim + 2) // 3
    _need(codes, bh * seq * 3 * ng, "codes"), _need(scales, bh * seq * ng, "scales")
    nc, ns = rotorquant_kv_page_elems(bh, seq, dim)
    pc = _empty((nc,), torch.int16, codes)
    ps = _empty((ns,), torch.float32, codes)
    _check(load().rnn_rotorquant_kv_pack(_ptr(codes), _ptr(scales), bh, seq, dim, bits, kind,
                                         _ptr(pc), _ptr(ps), _stream(stream)))
    return pc, ps


def rotorquant_kv_attention_workspace_size(bh, nq, seq, dim) -> int:
    return int(load().rnn_rotorquant_kv_attention_workspace_size(bh, nq, seq, dim))


# Zeroed attention workspaces kept per (device, stream): every call leaves
# the counts at zero, so one is reused by the calls ordered on its stream.
_attn_ws = {}


def _attn_workspace(dev, nbytes):
    key = (dev, _raw_stream(dev.index) if _raw_stream and dev.index is not None
           else torch.cuda.current_stream(dev).cuda_stream)
    ws = _attn_ws.get(key)
    if ws is None or ws.numel() < nbytes:
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
        _attn_ws[key] = ws
    return ws


def rotorquant_kv_attention(q, k_page, v_page, k_rotors, v_rotors, seq, scale, out=None,
                            stream=None, workspace=None):
    """Tensor::flash_attention (src/tensor.rs:618-672) of q [bh, nq, dim] over
    a K page (RQ_PAGE_K) and a V page (RQ_PAGE_V) of rotorquant_kv_pack.
    Returns out [bh, nq, dim]. `workspace`: a zeroed device byte tensor of at
    least rotorquant_kv_attention_workspace_size(bh, nq, seq, dim) bytes for
    the sequence split's states (calls leave it reusable); on the current
    stream a cached one is used when none is given, on another stream the
    call allocates."""
    _dev(q, torch.float32, "q")
    for t, nm in ((k_page[0], "k codes"), (v_page[0], "v codes")):
        _dev(t, torch.int16, nm)
    for t, nm in ((k_page[1], "k scales"), (v_page[1], "v scales"), (k_rotors, "k rotors"),
                  (v_rotors, "v rotors")):
        _dev(t, torch.float32, nm)
    _dev(workspace, torch.uint8, "workspace")
    bh, nq, dim = _dims(q, 3, "q")
    nc, ns = rotorquant_kv_page_elems(bh, seq, dim)
    for t, n_, nm in ((k_page[0], nc, "k codes"), (v_page[0], nc, "v codes"),
                      (k_page[1], ns, "k scales"), (v_page[1], ns, "v scales")):
        _need(t, n_, nm, at_least=True)
    ng = (dim + 2) // 3
    _need(k_rotors, 4 * ng, "k rotors", at_least=True), _need(v_rotors, 4 * ng, "v rotors", at_least=True)
    out = (_out(out, torch.float32, bh * nq * dim, "out") if out is not None
           else _empty((bh, nq, dim), torch.float32, q))
    if workspace is None and stream is None:
        wsb = rotorquant_kv_attention_workspace_size(bh, nq, seq, dim)
        if wsb:
            workspace = _attn_workspace(q.device, wsb)
    ws_bytes = 0 if workspace is None else workspace.numel()
    _check(load().rnn_rotorquant_kv_attention_ws(_ptr(q), bh, nq, _ptr(k_page[0]), _ptr(k_page[1]),
                                                 _ptr(v_page[0]), _ptr(v_page[1]), _ptr(k_rotors),
                                                 _ptr(v_rotors), seq, dim, float(scale), _ptr(out),
                                                 _ptr(workspace), ws_bytes, _stream(stream)))
    return out

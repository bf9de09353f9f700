"""GPU parity of x . W^T on operands split into bf16 parts (rnn_linear_layer_ws
and the tiled QuantizedLinear route): every output within the f32 GEMM rounding
bound of the float64 product, which is also the bar of the f32 kernels; the
bound's k + 4 counts the bias addition and the dropped products (each below
2^-25 of its product, three of nine)."""
import numpy as np
import pytest

import rnn_hip as H

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def data(m, k, n, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((m, k), generator=g, device="cuda")
    x = torch.where(torch.rand((m, k), generator=g, device="cuda") < 0.01, x * 20, x)
    w = torch.randn((n, k), generator=g, device="cuda") * 0.02
    return x, w, torch.randn((n,), generator=g, device="cuda")


def check(y, x, w, b):
    xd, wd = x.double(), w.double()
    exact, scale = xd @ wd.t(), xd.abs() @ wd.abs().t()
    if b is not None:
        exact, scale = exact + b.double(), scale + b.double().abs()
    assert bool(((y.double() - exact).abs() <= (x.shape[1] + 4) * U * scale + 1e-30).all())


# every tile shape (32x32 to 128x256), K ranges added by the sum kernel, K below and past one
# stage, odd K (4-byte loads), m and n at 1 and one past a tile
@pytest.mark.parametrize("m,k,n", [(1, 512, 31), (17, 66, 1), (2, 3347, 32), (33, 128, 100),
                                   (64, 257, 300), (129, 1024, 257), (130, 4096, 300),
                                   (300, 1000, 2049), (1307, 965, 16), (129, 4800, 3776),
                                   (513, 512, 4100), (2000, 256, 4096), (700, 4132, 520),
                                   (64, 4096, 11008), (32, 14336, 130), (1, 33, 5)])
def test_linear_layer_split(dev, hip, m, k, n):
    import torch
    x, w, b = data(m, k, n, m + k + n)
    assert hip.load().rnn_linear_layer_workspace_size(w.data_ptr(), m, k, n) > 0
    y = torch.full((m * n + 16,), -5.0, device="cuda")
    out = y[:m * n].view(m, n)
    hip.linear_layer(x, w, None, out=out)
    check(out, x, w, None)
    assert bool((y[m * n:] == -5).all())
    again = hip.linear_layer(x, w)
    assert torch.equal(again, out)                      # the same bits on every call
    z = hip.linear_layer(x, w, b, relu=True)
    zb = hip.linear_layer(x, w, b)
    check(zb, x, w, b)
    assert torch.equal(z, zb.clamp_min(0.0))


def test_linear_layer_split_unaligned_operands(dev, hip):
    """x and W at odd float addresses (scalar and 4-byte loads), the same
    product; W's rows end at the end of its storage."""
    import torch
    m, k, n = 70, 256, 130
    x, w, b = data(m, k, n, 5)
    xs, ws = torch.empty(m * k + 1, device="cuda"), torch.empty(n * k + 1, device="cuda")
    xs[1:], ws[1:] = x.reshape(-1), w.reshape(-1)
    y = hip.linear_layer(xs[1:].view(m, k), ws[1:].view(n, k), b)
    check(y, x, w, b)


def test_linear_layer_split_values_the_parts_do_not_hold(dev, hip):
    """Infinities and NaN give the pattern of the f32 product (an infinite x
    times a W whose lower parts are zero is infinite, not NaN); x and W far
    below bf16's range and products that overflow are computed in f32; tiles
    without such values keep their bits."""
    import torch
    m, k, n = 140, 512, 300
    x, w, _ = data(m, k, n, 9)
    w[:, 3] = 1.0                                       # (h = 1, m = l = 0)
    clean = hip.linear_layer(x, w)
    bad_x, bad_w = x.clone(), w.clone()
    bad_x[2, 3], bad_x[5, 3], bad_x[9, 17] = float("inf"), float("-inf"), float("nan")
    bad_w[7, 11], bad_w[8, 12] = float("inf"), float("nan")
    y = hip.linear_layer(bad_x, bad_w)
    ref = bad_x.double() @ bad_w.double().t()
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))
    assert torch.equal(torch.sign(y[torch.isinf(ref)]).double(), torch.sign(ref[torch.isinf(ref)]))
    fine = torch.isfinite(ref)
    lim = (k + 4) * U * (bad_x.nan_to_num(0, 0, 0).double().abs() @
                         bad_w.nan_to_num(0, 0, 0).double().abs().t())
    assert bool(((y.double() - ref).abs() <= lim)[fine].all())
    assert torch.equal(y[128:, 256:], clean[128:, 256:])
    # rows of x near 2^-120 against W near 2^90, and the reverse: full f32 precision
    for sx, sw in ((2.0 ** -120, 2.0 ** 90), (2.0 ** 90, 2.0 ** -120), (2.0 ** -120, 1.0)):
        xs, ws = x * sx, w * sw
        check_scaled = (xs.double() @ ws.double().t())
        err = (hip.linear_layer(xs, ws).double() - check_scaled).abs()
        lim = (k + 4) * U * (xs.double().abs() @ ws.double().abs().t()) + k * 2.0 ** -149
        assert bool((err <= lim).all())
    big = hip.linear_layer(x * 2.0 ** 100, w * 2.0 ** 40)
    assert bool(torch.isinf(big).any())
    assert torch.equal(clean, hip.linear_layer(x, w))


@pytest.mark.parametrize("k", [481, 497, 510, 543])
def test_linear_layer_split_computed_again_k_remainders(dev, hip, k):
    """Tiles computed again in f32 where K ends within a pass of 32: the bound
    of an f32 sum in any order, (k + 4) U sum |x||w|."""
    import torch
    m, n = 140, 300
    x, w, b = data(m, k, n, k)
    x[::16, 5] = 2.0 ** -120
    w[::32, k - 1] = 2.0 ** -125
    assert hip.load().rnn_linear_layer_workspace_size(w.data_ptr(), m, k, n) > 0
    ref = x.double() @ w.double().t() + b.double()
    lim = (k + 4) * U * (x.double().abs() @ w.double().abs().t() + b.double().abs())
    assert bool(((hip.linear_layer(x, w, b).double() - ref).abs() <= lim).all())


def test_linear_layer_split_capture_and_streams(dev, hip):
    """Replays of a captured call, and a call on another stream, give the
    eager bits (the parts live in the call's own scratch)."""
    import torch
    x, w, b = data(200, 1024, 700, 11)
    eager = hip.linear_layer(x, w, b)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    other = torch.empty_like(eager)
    hip.linear_layer(x, w, b, out=other, stream=s)
    s.synchronize()
    assert torch.equal(other, eager)
    with torch.cuda.stream(s):
        hip.linear_layer(x, w, b)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = hip.linear_layer(x, w, b)
    for i in range(3):
        x.mul_(1.5)
        g.replay()
        assert torch.equal(out, hip.linear_layer(x, w, b)), i


FORMATS = {"INT4-g128": (H.QF_INT4, 128), "Q4_0": (H.QF_GGUF_Q4, 32), "INT8-g64": (H.QF_INT8, 64),
           "Q8_0": (H.QF_GGUF_Q8, 32), "BF16": (H.QF_BF16, 0), "NVFP4-g32": (H.QF_NVFP4, 32),
           "INT8-rows": (H.QF_INT8, 1024), "INT4-tensor": (H.QF_INT4, 0), "INT8-2rows": (H.QF_INT8, 2048)}


def quantized(fmt, gs, n, k, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randn((n, k), generator=g, device="cuda") * 0.02
    d, s, gg = H.qt_quantize(fmt, w, gs if gs else n * k)
    return d, s, gg, H.qt_dequantize(fmt, d, s, gg, n * k).view(n, k)


# tiles of 32x32, 32x64 and 64x128, one and several ranges of K, ragged m and n
@pytest.mark.parametrize("m,k,n", [(49, 1024, 33), (300, 1024, 2049), (130, 4096, 1000),
                                   (1000, 1024, 4096), (65, 11264, 64)])
@pytest.mark.parametrize("name", FORMATS)
def test_quantized_linear_tiles(dev, hip, name, m, k, n):
    import torch
    fmt, gs = FORMATS[name]
    if gs > 32 and (k % gs and gs % k):
        pytest.skip("a group that neither divides nor is divided by a row")
    if gs == 2048 and n % 2:
        n += 1
    d, s, g, w = quantized(fmt, gs, n, k, m + n)
    x, _, b = data(m, k, n, m)
    size = hip.load().rnn_qt_linear_scratch_size(fmt, m, k, d.data_ptr(), s.data_ptr(), s.numel(), g, n)
    parts = -(-m // 128) * 128 * -(-k // 32) * 192 + 8 * 4 * m * n
    assert 0 <= size <= parts                           # the tiles' scratch (or the slices': none)
    y = torch.full((m * n + 16,), -5.0, device="cuda")
    out = y[:m * n].view(m, n)
    hip.qt_linear_forward(fmt, x, d, s, g, n, b, y=out)
    check(out, x, w, b)
    assert bool((y[m * n:] == -5).all())
    assert torch.equal(out, hip.qt_linear_forward(fmt, x, d, s, g, n, b))


@pytest.mark.parametrize("name", ["INT4-g128", "Q8_0", "BF16", "NVFP4-g32"])
def test_quantized_linear_tiles_nonfinite(dev, hip, name):
    """Non-finite x, scales and BF16 weights, and x below bf16's range, on the
    tiles: the pattern of the f32 product of the dequantized weight."""
    import torch
    fmt, gs = FORMATS[name]
    m, k, n = 200, 1024, 700
    d, s, g, _ = quantized(fmt, gs, n, k, 3)
    x, _, _ = data(m, k, n, 4)
    x[1, 5], x[3, 6], x[70, 9] = float("inf"), float("nan"), 2.0 ** -130
    x[90] *= 2.0 ** -115
    if name == "BF16":
        d.view(torch.int16)[11 * k + 7] = 0x7F80        # +inf
        d.view(torch.int16)[12 * k + 7] = 0x7FC0        # NaN
    else:
        s[11 * k // g] = float("inf")
    w = hip.qt_dequantize(fmt, d, s, g, n * k).view(n, k)
    assert hip.load().rnn_qt_linear_scratch_size(fmt, m, k, d.data_ptr(), s.data_ptr(), s.numel(), g, n) > 0
    y = hip.qt_linear_forward(fmt, x, d, s, g, n)
    ref = x.double() @ w.double().t()
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))
    fine = torch.isfinite(ref)
    lim = (k + 4) * U * (x.nan_to_num(0, 0, 0).double().abs() @ w.nan_to_num(0, 0, 0).double().abs().t())
    assert bool(((y.double() - ref).abs() <= lim + k * 2.0 ** -149)[fine].all())


def test_quantized_linear_dequantize_in_scratch(dev, hip):
    """Formats and groups the tiles do not take, m above the slices: the weight
    is dequantized into the call's scratch."""
    import torch
    for fmt, gs, m, k, n in ((H.QF_NF4, 64, 700, 512, 300), (H.QF_FP16, 0, 700, 512, 300),
                             (H.QF_INT4, 33, 100, 201, 70), (H.QF_NF4, 64, 20, 200, 70)):
        d, s, g, w = quantized(fmt, gs, n, k, m)
        x, _, b = data(m, k, n, m)
        check(hip.qt_linear_forward(fmt, x, d, s, g, n, b), x, w, b)

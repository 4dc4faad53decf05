"""How far the convolutions' gradients are from their sums in 64 bits, and what their rarer forms return and take."""
import ctypes
import itertools

import numpy as np
import pytest
import torch

from neurotensor_amd import _lib
from neurotensor_amd import functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


def randn(shape, dtype, seed, scale=1.0):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    return (torch.randn(shape, device=DEV, generator=gen) * scale).to(dtype)


def windows(x, k, s, p, d, out):
    """(tap, the [B, C, *out] elements that it meets) for every tap of the window."""
    nd = len(k)
    xp = torch.nn.functional.pad(x, [q for a in reversed(range(nd)) for q in (p[a], p[a])]) if any(p) else x
    for t in itertools.product(*[range(i) for i in k]):
        yield t, xp[(slice(None), slice(None)) + tuple(slice(t[a] * d[a], t[a] * d[a] + (out[a] - 1) * s[a] + 1, s[a]) for a in range(nd))]


def exact_dw(x, g, k, s, p, d, groups):
    """The weight gradient in Float64: one product of matrices per tap and group."""
    x, g = x.double(), g.double()
    O, cg, og = g.shape[1], x.shape[1] // groups, g.shape[1] // groups
    dw = torch.zeros((O, cg) + tuple(k), device=x.device, dtype=torch.float64)
    for t, win in windows(x, k, s, p, d, g.shape[2:]):
        for gi in range(groups):
            xg = win[:, gi * cg:(gi + 1) * cg].transpose(0, 1).reshape(cg, -1).t().contiguous()
            gg = g[:, gi * og:(gi + 1) * og].transpose(0, 1).reshape(og, -1).contiguous()
            dw[(slice(gi * og, (gi + 1) * og), slice(None)) + t] = gg @ xg
    return dw


def exact_dx(size, w, g, k, s, p, d, groups):
    """The image gradient in Float64: one product of matrices per tap and group, added at the elements that the tap meets."""
    w, g = w.double(), g.double()
    B, O, out = g.shape[0], g.shape[1], tuple(g.shape[2:])
    cg, og = w.shape[1], O // groups
    dx = torch.zeros((B, cg * groups) + tuple(size[a] + 2 * p[a] for a in range(len(size))), device=w.device, dtype=torch.float64)
    for t, win in windows(dx, k, s, (0,) * len(k), d, out):
        for gi in range(groups):
            gg = g[:, gi * og:(gi + 1) * og].transpose(0, 1).reshape(og, -1)
            col = w[(slice(gi * og, (gi + 1) * og), slice(None)) + t].t().contiguous() @ gg
            win[:, gi * cg:(gi + 1) * cg] += col.reshape((cg, B) + out).transpose(0, 1)
    return dx[(slice(None), slice(None)) + tuple(slice(p[a], p[a] + size[a]) for a in range(len(size)))]


def relative(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


def backward(nd):
    return {1: F.conv1d_backward, 2: F.conv2d_backward, 3: F.conv3d_backward}[nd]


@pytest.mark.parametrize("geom", [
    # (B, C, size, O, kernel, stride, padding, groups)
    (2, 256, (32, 32), 1024, (3, 3), 1, 1, 1),      # two k ranges in 256 x 256 tiles
    (64, 512, (14, 14), 512, (7, 7), 1, 3, 1),      # a few ranges over 64 images
    (64, 256, (28, 28), 256, (3, 3), 1, 1, 1),      # as many as fill the CUs
    (26, 96, (13, 13, 13), 256, (3, 3, 3), 1, 1, 1),
    (6, 24, (9, 9, 9), 64, (3, 3, 3), 2, 1, 1),
    (10, 128, (19, 19), 48, (7, 7), 1, 3, 1),       # rows that miss the 16-byte rule: dY through its copy
    (16, 16, (7, 17), 32, (3, 3), 1, 1, 4),
    (2, 192, (40, 40), 256, (3, 3), 2, 1, 1),
], ids=lambda g: "x".join(map(str, g)))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_16_bit_weight_gradients_are_rounded_once(geom, dtype):
    """A gradient that is one rounding of its Float32 sum is as far from the exact sum as that sum's own rounding (the Float32 chain
    adds some 1e-6 of it); a second rounding, of partial sums, makes that sqrt(2) times as much.  1.1 lies between."""
    B, C, size, O, k, s, p, groups = geom
    nd = len(size)
    out = [(size[a] + 2 * p - k[a]) // s + 1 for a in range(nd)]
    x, w, g = randn((B, C) + size, dtype, 1), randn((O, C // groups) + k, dtype, 2, 0.05), randn([B, O] + out, dtype, 3)
    _, dw = backward(nd)(x, w, g, stride=s, padding=p, groups=groups)
    want = exact_dw(x, g, k, (s,) * nd, (p,) * nd, (1,) * nd, groups)
    assert relative(dw, want) <= 1.1 * relative(want.to(dtype), want), (relative(dw, want), relative(want.to(dtype), want))


@pytest.mark.parametrize("geom", [
    # (B, C, size, O, kernel, stride, padding)
    (22, 23, (1, 69), 4, (1, 5), (1, 3), (0, 0)),      # 22 pixels per image, rows of dY that miss the 16-byte rule
    (38, 8, (1, 19), 168, (1, 5), (1, 2), (0, 2)),
    (43, 8, (4, 4), 208, (2, 2), (1, 1), (1, 0)),
], ids=lambda g: "x".join(map(str, g)))
def test_fp32_weight_gradients_of_small_maps_are_as_close_as_the_reference_order(geom):
    """Over small maps the reference sums short chains (the pixels of one image, then the images), which the host entry point follows
    bit for bit.  The rounding errors of a chain of n sums grow as sqrt(n): a few long chains through all images were 1.4 to 2 times
    as far from the exact gradient, chains of one or two K-steps (16 or 32 pixels) differ by less than 1.2; 1.3 lies between."""
    B, C, size, O, k, s, p = geom
    out = [(size[a] + 2 * p[a] - k[a]) // s[a] + 1 for a in range(2)]
    x, w, g = randn((B, C) + size, torch.float32, 1), randn((O, C) + k, torch.float32, 2, 0.05), randn([B, O] + out, torch.float32, 3)
    _, dw = F.conv2d_backward(x, w, g, stride=s, padding=p)
    hx, hw, hg = (t.cpu().numpy() for t in (x, w, g))
    hdx, hdw = np.empty_like(hx), np.empty_like(hw)
    vp = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    _lib.check(_lib.load().ntg_conv2d_backward(_lib.FLOAT32, vp(hx), vp(hw), vp(hg), vp(hdx), vp(hdw), B, C, size[0], size[1], O, k[0], k[1],
                                               s[0], s[1], p[0], p[1], 1, 1, 1, 0))
    want = exact_dw(x, g, k, s, p, (1, 1), 1)
    ours, reference = relative(dw, want), relative(torch.from_numpy(hdw).to(DEV), want)
    assert ours <= 1.3 * reference, (ours, reference)


def microseconds(fn, passes=10):
    for _ in range(3):
        fn()
    best = float("inf")
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(passes):
            fn()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) / passes * 1e3)
    return best


@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_many_weights_over_one_small_image(nd, dtype):
    """A single small image (a copy of eight blocks beside a million weights) takes no longer than sixteen of them, and gives the
    first of the sixteen's results bit for bit."""
    size, k = (4,) * nd, (3,) * nd
    x, w, g = randn((16, 512) + size, dtype, 1), randn((192, 512) + k, dtype, 2, 0.02), randn((16, 192) + size, dtype, 3)
    fwd = {2: F.conv2d, 3: F.conv3d}[nd]
    calls = (lambda n: fwd(x[:n], w, padding=1), lambda n: backward(nd)(x[:n], w, g[:n], padding=1)[0])
    for call in calls:
        assert torch.equal(call(1)[0], call(16)[0])
        one, sixteen = microseconds(lambda: call(1)), microseconds(lambda: call(16))
        assert one <= 1.2 * sixteen, (one, sixteen)


@pytest.mark.parametrize("geom", [
    # (B, C, size, O, kernel, stride, padding, groups)
    (4, 32, (8, 64), 32, (8, 8), 2, (0, 0), 1),            # one row of outputs: the border is 7 times dY
    (3, 64, (9, 130), 48, (8, 7), (2, 3), (0, 3), 2),
    (2, 32, (7, 40), 32, (7, 4), (1, 4), (0, 1), 1),       # a stride along one axis: a border of 6 rows on each side of one row
    (4096, 1024, (4, 4), 16, (3, 3), 2, (1, 1), 1),        # four million planes of four elements
], ids=lambda g: "x".join(map(str, g)))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_16_bit_strided_image_gradients_are_rounded_once(geom, dtype):
    """Image gradients by phases of the strides are one rounding of their Float32 sums (bound as above); the GEMM + col2im form rounds
    every entry of the col matrix and then their sum."""
    B, C, size, O, k, s, p, groups = geom
    s = s if isinstance(s, tuple) else (s, s)
    out = [(size[a] + 2 * p[a] - k[a]) // s[a] + 1 for a in range(2)]
    x, w, g = randn((B, C) + size, dtype, 1), randn((O, C // groups) + k, dtype, 2, 0.05), randn([B, O] + out, dtype, 3)
    dx, _ = F.conv2d_backward(x, w, g, stride=s, padding=p, groups=groups)
    want = exact_dx(size, w, g, k, s, p, (1, 1), groups)
    assert relative(dx, want) <= 1.1 * relative(want.to(dtype), want), (relative(dx, want), relative(want.to(dtype), want))


def _arr(v):
    return (ctypes.c_int64 * len(v))(*v)


@pytest.mark.parametrize("geom", [
    # (B, C, size, O, kernel, stride, padding, dilation, groups)
    (2, 32, (6, 7, 8), 48, (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), 1),
    (3, 32, (5, 8, 12), 32, (3, 2, 3), (1, 2, 1), (1, 0, 1), (1, 1, 2), 2),
    (1, 64, (8, 8, 8), 32, (2, 2, 2), (2, 2, 2), (0, 0, 0), (1, 1, 1), 1),
    (70, 16, (4, 4, 4), 16, (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), 1),   # the weight gradient's ranges fit into the smaller workspace
], ids=lambda g: "x".join(map(str, g)))
def test_fp32_three_axes_keep_the_reference_order_in_the_smaller_workspace(geom):
    """Device calls with ntg_convnd_workspace_bytes of workspace sum in the order of the host entry points: the same bits.  Either
    gradient alone takes the form that it takes beside the other."""
    B, C, size, O, k, s, p, d, groups = geom
    out = tuple((size[a] + 2 * p[a] - d[a] * (k[a] - 1) - 1) // s[a] + 1 for a in range(3))
    x, w, g = randn((B, C) + size, torch.float32, 1), randn((O, C // groups) + k, torch.float32, 2, 0.05), randn((B, O) + out, torch.float32, 3)
    hx, hw, hg = (t.cpu().numpy() for t in (x, w, g))
    hy, hdx, hdw = np.empty((B, O) + out, np.float32), np.empty_like(hx), np.empty_like(hw)
    vp = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    geo = tuple(_arr(v) for v in (size, k, s, p, d))
    lib = _lib.load()
    _lib.check(lib.ntg_convnd(_lib.FLOAT32, vp(hx), vp(hw), vp(hy), B, C, O, 3, *geo, groups))
    _lib.check(lib.ntg_convnd_backward(_lib.FLOAT32, vp(hx), vp(hw), vp(hg), vp(hdx), vp(hdw), B, C, O, 3, *geo, groups, 0))
    st = torch.cuda.current_stream().cuda_stream
    fwd, bwd = (lib.ntg_convnd_workspace_bytes(_lib.FLOAT32, B, C, O, 3, *geo, groups, b) for b in (0, 1))
    ws = torch.empty((max(fwd, bwd, 1),), dtype=torch.uint8, device=DEV)
    y, dx, dw, dx1, dw1 = torch.empty((B, O) + out, device=DEV), torch.empty_like(x), torch.empty_like(w), torch.empty_like(x), torch.empty_like(w)
    _lib.check(lib.ntg_convnd_dev(_lib.FLOAT32, x.data_ptr(), w.data_ptr(), y.data_ptr(), ws.data_ptr(), fwd, B, C, O, 3, *geo, groups, st))
    for pdx, pdw in ((dx, dw), (dx1, None), (None, dw1)):
        _lib.check(lib.ntg_convnd_backward_dev(_lib.FLOAT32, x.data_ptr(), w.data_ptr(), g.data_ptr(), None if pdx is None else pdx.data_ptr(),
                                               None if pdw is None else pdw.data_ptr(), ws.data_ptr(), bwd, B, C, O, 3, *geo, groups, 0, st))
    for got, want in ((y, hy), (dx, hdx), (dw, hdw), (dx1, hdx), (dw1, hdw)):
        assert torch.equal(got.cpu(), torch.from_numpy(want))


def exact_y(x, w, s, p, d, out, groups):
    """The convolution in Float64: one product of matrices per tap and group."""
    x, w = x.double(), w.double()
    B, O = x.shape[0], w.shape[0]
    cg, og = w.shape[1], O // groups
    y = torch.zeros((B, O) + tuple(out), device=w.device, dtype=torch.float64)
    for t, win in windows(x, w.shape[2:], s, p, d, out):
        for gi in range(groups):
            xg = win[:, gi * cg:(gi + 1) * cg].transpose(0, 1).reshape(cg, -1)
            part = w[(slice(gi * og, (gi + 1) * og), slice(None)) + t].contiguous() @ xg
            y[:, gi * og:(gi + 1) * og] += part.reshape((og, B) + tuple(out)).transpose(0, 1)
    return y


@pytest.mark.parametrize("geom,dtype", [
    # (B, C, size, O, kernel, stride, groups), and the tiles that the planners choose:
    ((4, 128, (32, 32, 32), 128, (3, 3, 3), 1, 1), torch.float32),      # 128 x 128 in all three
    ((4, 128, (31, 33, 31), 128, (3, 3, 3), 1, 1), torch.float32),      # ... dY through its copy, outputs that end inside a tile
    ((16, 128, (16, 16, 16), 128, (3, 3, 3), 2, 1), torch.float32),     # the phases 128 x 128
    ((16, 64, (16, 16, 16), 256, (3, 3, 3), 1, 2), torch.float32),      # groups: forward 128 x 128
    ((16, 32, (16, 16, 17), 256, (3, 3, 3), 1, 1), torch.bfloat16),     # forward 256 x 256 and the last 256 outputs on 64 x 64, dW 128 x 128
    ((16, 256, (16, 16, 17), 32, (3, 3, 3), 1, 1), torch.float16),      # the same of the image gradient
    ((16, 256, (16, 16, 16), 32, (3, 3, 3), 2, 1), torch.bfloat16),     # the phases 256 x 256
    ((16, 128, (16, 16, 16), 32, (3, 3, 3), 2, 1), torch.float16),      # the phases 128 x 128
    ((8, 256, (15, 17, 17), 256, (3, 3, 3), 1, 1), torch.bfloat16),     # 256 x 256 in all three, dY through its copy
    ((24, 256, (16, 16, 16), 256, (1, 3, 3), 1, 1), torch.float16),     # 256 x 256, the last eight images 128 x 128; dW 256 x 256
    ((16, 64, (16, 16, 16), 256, (3, 3, 3), 1, 2), torch.bfloat16),     # groups: 128 x 128 in all three
], ids=str)
def test_three_axes_on_the_large_tiles(geom, dtype):
    """Three axes at sizes that reach the 128- and 256-row tiles of the channels-last kernels, against Float64.  16 bits: one
    rounding (bound as above).  Float32: each of the K roundings of a sum of K random products errs by 2^-24 of a partial sum at most, which is
    no larger than the results in the mean, and independent errors add up as sqrt(K): sqrt(K) * 2^-24 of the results' norm."""
    B, C, size, O, k, s, groups = geom
    p = tuple(i // 2 for i in k)
    out = tuple((size[a] + 2 * p[a] - k[a]) // s + 1 for a in range(3))
    x, w, g = randn((B, C) + size, dtype, 1), randn((O, C // groups) + k, dtype, 2, 0.05), randn((B, O) + out, dtype, 3)
    y = F.conv3d(x, w, stride=s, padding=p, groups=groups)
    dx, dw = F.conv3d_backward(x, w, g, stride=s, padding=p, groups=groups)
    taps = k[0] * k[1] * k[2]
    for name, got, exact, depth in (("y", y, lambda: exact_y(x, w, (s,) * 3, p, (1,) * 3, out, groups), C // groups * taps),
                                    ("dx", dx, lambda: exact_dx(size, w, g, k, (s,) * 3, p, (1,) * 3, groups), O // groups * taps),
                                    ("dw", dw, lambda: exact_dw(x, g, k, (s,) * 3, p, (1,) * 3, groups), B * out[0] * out[1] * out[2])):
        want = exact()
        bound = 2.0 ** -24 * depth ** 0.5 if dtype == torch.float32 else 1.1 * relative(want.to(dtype), want)
        assert relative(got, want) <= bound, (name, relative(got, want), bound)
        # (no element is off on its own: a misplaced one differs by about its neighbours' size)
        worst = ((got.double() - want).abs().max() / want.square().mean().sqrt()).item()
        assert worst <= (1e-6 * depth ** 0.5 if dtype == torch.float32 else 0.06), (name, worst)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("geom", [
    # (B, C, size, O, kernel, stride, groups)
    (2, 32, (6, 7, 8), 48, (3, 3, 3), 1, 1),
    (3, 32, (9, 8, 11), 64, (3, 3, 3), 2, 2),
], ids=str)
def test_three_axes_gradients_add_to_what_is_there(geom, dtype):
    """accumulate = 1 on the channels-last forms.  16 bits: Float32 sums with the incoming value in them, rounded once -- but the image
    gradient at strides > 1 is rounded in its phase's plane first, an error of sqrt(1 + 1/2) of one rounding where both terms are of one
    size; bounds of 1.1 times these.  Float32 as above."""
    B, C, size, O, k, s, groups = geom
    p = (1,) * 3
    out = tuple((size[a] + 2 - k[a]) // s + 1 for a in range(3))
    x, w, g = randn((B, C) + size, dtype, 1), randn((O, C // groups) + k, dtype, 2, 0.05), randn((B, O) + out, dtype, 3)
    want_dx, want_dw = exact_dx(size, w, g, k, (s,) * 3, p, (1,) * 3, groups), exact_dw(x, g, k, (s,) * 3, p, (1,) * 3, groups)
    dx0 = randn(x.shape, dtype, 4, want_dx.std().item())
    dw0 = randn(w.shape, dtype, 5, want_dw.std().item())
    dx, dw = dx0.clone(), dw0.clone()
    lib, code = _lib.load(), F.ntg_dtype(x)
    geo = tuple(_arr(v) for v in (size, k, (s,) * 3, p, (1,) * 3))
    need = lib.ntg_convnd_fast_workspace_bytes(code, B, C, O, 3, *geo, groups, 1)
    ws = torch.empty((need,), dtype=torch.uint8, device=DEV)
    _lib.check(lib.ntg_convnd_backward_dev(code, x.data_ptr(), w.data_ptr(), g.data_ptr(), dx.data_ptr(), dw.data_ptr(), ws.data_ptr(), need,
                                           B, C, O, 3, *geo, groups, 1, torch.cuda.current_stream().cuda_stream))
    for name, got, want, depth, roundings in (("dx", dx, dx0.double() + want_dx, O // groups * 27, 1.5 if s > 1 else 1.0),
                                              ("dw", dw, dw0.double() + want_dw, B * out[0] * out[1] * out[2], 1.0)):
        bound = 2.0 ** -24 * depth ** 0.5 if dtype == torch.float32 else 1.1 * roundings ** 0.5 * relative(want.to(dtype), want)
        assert relative(got, want) <= bound, (name, relative(got, want), bound)


@pytest.mark.parametrize("geom", [
    # (B, C, size, O, kernel, stride, padding, groups)
    (7, 128, (8, 8, 8), 48, (3, 3, 3), 2, 1, 1),           # image gradient by phases: three K-steps of out channels per tap
    (37, 192, (10, 10, 10), 32, (3, 3, 3), 2, 1, 1),       # ... two; 125 pixels per image
    (4, 32, (9, 9, 9), 16, (4, 4, 4), 2, 1, 1),            # ... one
    (4, 128, (9, 9, 9), 192, (3, 3, 3), 2, 1, 1),
    (16, 128, (16, 16, 16), 256, (4, 4, 4), 2, 1, 2),      # 128 x 128 tiles
    (25, 128, (12, 12), 192, (3, 3), 1, 1, 1),
    (15, 96, (7, 7), 96, (5, 5), 2, 2, 1),                 # 16 pixels per image: chains of one K-step
    (20, 256, (1, 512), 256, (1, 4), (1, 2), (0, 1), 1),
], ids=str)
def test_fp32_gradients_are_as_close_as_sums_per_tap_and_per_image(geom):
    """The reference adds up one product per tap (the image gradient, on three axes at strides) and per image (the weight gradient); the
    host entry points follow it bit for bit.  The device's chains are no longer than these, so their rounding errors are of the same
    size: over the 10^4 values and more of a gradient the ratio of the two norms is 1 within some percent; one chain through everything was
    1.4 to 2.5."""
    B, C, size, O, k, s, p, groups = geom
    nd = len(size)
    s, p = (s,) * nd if isinstance(s, int) else s, (p,) * nd if isinstance(p, int) else p
    out = tuple((size[a] + 2 * p[a] - k[a]) // s[a] + 1 for a in range(nd))
    x, w, g = randn((B, C) + size, torch.float32, 1), randn((O, C // groups) + k, torch.float32, 2, 0.05), randn((B, O) + out, torch.float32, 3)
    dx, dw = backward(nd)(x, w, g, stride=s, padding=p, groups=groups)
    hx, hw, hg = (t.cpu().numpy() for t in (x, w, g))
    hdx, hdw = np.empty_like(hx), np.empty_like(hw)
    vp = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    geo = tuple(_arr(v) for v in (size, k, s, p, (1,) * nd))
    _lib.check(_lib.load().ntg_convnd_backward(_lib.FLOAT32, vp(hx), vp(hw), vp(hg), vp(hdx), vp(hdw), B, C, O, nd, *geo, groups, 0))
    checks = [("dw", dw, hdw, exact_dw(x, g, k, s, p, (1,) * nd, groups))]
    if nd == 3:
        checks.append(("dx", dx, hdx, exact_dx(size, w, g, k, s, p, (1,) * nd, groups)))
    for name, got, host, want in checks:
        ours, reference = relative(got, want), relative(torch.from_numpy(host).to(DEV), want)
        assert ours <= 1.15 * reference, (name, ours, reference)


@pytest.mark.parametrize("geom", [
    # (B, C, size, O, groups): 32 rows and fewer in the forward product, in the image gradient
    (2, 128, (8, 12), 16, 1), (2, 256, (8, 12), 32, 2), (1, 64, (96,), 8, 1), (3, 16, (8, 12), 192, 1), (2, 32, (96,), 256, 2),
], ids=str)
def test_fp32_one_tap_through_the_host_entry_points_is_the_reference_product(geom):
    """unfold + matmult bit for bit, also where the device entry points split k over the wavefronts of the kernels for few rows."""
    B, C, size, O, groups = geom
    nd, L, cg, og = len(size), int(np.prod(size)), C // groups, O // groups
    x, w, g = (randn(shape, torch.float32, i).cpu().numpy() for i, shape in enumerate(((B, C) + size, (O, cg) + (1,) * nd, (B, O) + size)))
    y, dx = np.empty_like(g), np.empty_like(x)
    vp = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    geo = tuple(_arr(v) for v in (size, (1,) * nd, (1,) * nd, (0,) * nd, (1,) * nd))
    lib = _lib.load()
    _lib.check(lib.ntg_convnd(_lib.FLOAT32, vp(x), vp(w), vp(y), B, C, O, nd, *geo, groups))
    _lib.check(lib.ntg_convnd_backward(_lib.FLOAT32, vp(x), vp(w), vp(g), vp(dx), None, B, C, O, nd, *geo, groups, 0))
    for b in range(B):
        for q in range(groups):
            wq = np.ascontiguousarray(w.reshape(O, cg)[q * og:(q + 1) * og])
            for got, a, rhs, m, k in ((y, wq, x, og, cg), (dx, np.ascontiguousarray(wq.T), g, cg, og)):
                want, rhs = np.zeros((m, L), np.float32), np.ascontiguousarray(rhs.reshape(B, groups, k, L)[b, q])
                _lib.check(lib.ntg_matmult(_lib.FLOAT32, vp(a), vp(rhs), vp(want), m, k, k, L, 0, 0))
                assert np.array_equal(got.reshape(B, groups, m, L)[b, q], want), (b, q, m, k)


@pytest.mark.parametrize("geom", [
    # (B, C, size, O, groups): up to 32 rows in the forward product or the image gradient, 64 k and more; a pitch of one strip, of odd strips, of one column block
    (8, 256, (28, 28), 64, 4), (3, 64, (32, 5), 256, 2), (2, 512, (28, 28), 32, 2), (5, 1040, (4,), 32, 4), (2, 128, (2044,), 16, 1),
    (6, 64, (5992,), 32, 4), (2, 256, (4004,), 16, 1),
], ids=str)
def test_fp32_few_rows_in_groups_err_no_more_than_the_products_of_each_group(geom):
    """The kernels for up to 32 rows add up eight short chains, and layers in groups go through them in one launch: the same bits as each group's layer
    by itself.  The weight gradient of one tap is no further from the sums in 64 bits than the images' products added up (ratio 1 within some percent; one
    chain an image was 2.9)."""
    B, C, size, O, groups = geom
    nd, cg, og = len(size), C // groups, O // groups
    forward = {1: F.conv1d, 2: F.conv2d}[nd]
    x, w, g = (randn(shape, torch.float32, i) for i, shape in enumerate(((B, C) + size, (O, cg) + (1,) * nd, (B, O) + size)))
    y = forward(x, w, groups=groups)
    dx, dw = backward(nd)(x, w, g, groups=groups)
    per_image = torch.zeros_like(dw)
    for q in range(groups):
        c, o = slice(q * cg, (q + 1) * cg), slice(q * og, (q + 1) * og)
        xq, wq, gq = x[:, c].contiguous(), w[o].contiguous(), g[:, o].contiguous()
        assert torch.equal(y[:, o], forward(xq, wq)), q
        assert torch.equal(dx[:, c], backward(nd)(xq, wq, gq)[0]), q
        for b in range(B):
            per_image[o] += F.matmult(gq[b].reshape(og, -1), xq[b].reshape(cg, -1), None, False, True).reshape(wq.shape)
    want = exact_dw(x, g, (1,) * nd, (1,) * nd, (0,) * nd, (1,) * nd, groups)
    assert relative(dw, want) <= 1.15 * relative(per_image, want), (relative(dw, want), relative(per_image, want))


def test_fp32_few_rows_in_groups_of_more_images_than_a_launch_holds():
    """65535 items: 33000 images in two groups go out group by group."""
    x, w = randn((33000, 128, 4), torch.float32, 1), randn((32, 64, 1), torch.float32, 2)
    y = F.conv1d(x, w, groups=2)
    for q in range(2):
        assert torch.equal(y[:, 16 * q:16 * q + 16], F.conv1d(x[:, 64 * q:64 * q + 64].contiguous(), w[16 * q:16 * q + 16].contiguous())), q


@pytest.mark.parametrize("geom", [
    # (B, C, size, O, kernel, stride, groups)
    (4, 24, (64, 64), 32, (5, 5), 1, 4), (8, 96, (28, 28), 48, (3, 3), 1, 4), (1, 192, (29, 29, 29), 48, (3, 3, 3), 2, 4),
], ids=str)
def test_fp32_weight_gradients_in_groups_are_as_close_as_each_group_by_itself(geom):
    """Groups share the ranges that fill the CUs, so each has fewer and longer ones than its layer by itself; the chains are short enough that the
    gradient is as close all the same (chains of 256 multiply-adds: ratios of 1.33, 1.0 and 1.15).  Over 5000 values and more the ratio of the two norms
    is known to 2 %."""
    B, C, size, O, k, s, groups = geom
    nd, p = len(size), tuple(v // 2 for v in k)
    out = tuple((size[a] + 2 * p[a] - k[a]) // s + 1 for a in range(nd))
    x, w, g = randn((B, C) + size, torch.float32, 1), randn((O, C // groups) + k, torch.float32, 2, 0.05), randn((B, O) + out, torch.float32, 3)
    _, dw = backward(nd)(x, w, g, stride=s, padding=p[0], groups=groups)
    want = exact_dw(x, g, k, (s,) * nd, p, (1,) * nd, groups)
    cg, og = C // groups, O // groups
    alone = torch.cat([backward(nd)(x[:, q * cg:(q + 1) * cg].contiguous(), w[q * og:(q + 1) * og].contiguous(), g[:, q * og:(q + 1) * og].contiguous(),
                                    stride=s, padding=p[0])[1] for q in range(groups)])
    assert relative(dw, want) <= 1.1 * relative(alone, want), (relative(dw, want), relative(alone, want))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("width", [2040, 2048])
@pytest.mark.parametrize("groups", [1, 2])
def test_16_bit_weight_gradients_of_one_tap_on_rows_of_8_mib(width, dtype, groups):
    """Rows of 2^23 bytes are the first that the kernels that can write Float32 sums do not take as a pitch.  One rounding to 16 bits, on both sides of it (one
    image); the sums of 2^22 products in 32 bits add at most 2^-24 sqrt(2^22) = 1.2e-4 of the result, 1 / 2 of Float16's rounding in the norm of both."""
    x, g = randn((1, 16, 2048, width), dtype, 1), randn((1, 16, 2048, width), dtype, 3)
    w = randn((16, 16 // groups, 1, 1), dtype, 2)
    _, dw = F.conv2d_backward(x, w, g, groups=groups)
    want = exact_dw(x, g, (1, 1), (1, 1), (0, 0), (1, 1), groups)
    assert relative(dw, want) <= 1.25 * relative(want.to(dtype), want), (relative(dw, want), relative(want.to(dtype), want))


@pytest.mark.parametrize("geom", [
    # (B, C, size, O, kernel, stride, groups): out channels of a group that are no multiple of 16
    (8, 32, (56, 56), 24, (3, 3), 2, 1),
    (8, 32, (56, 56), 24, (7, 7), 2, 1),
    (8, 64, (56, 56), 48, (5, 5), 2, 2),
    (8, 48, (28, 28), 72, (4, 4), 2, 1),                   # 72: two K-steps and a half
    (8, 32, (56, 56), 8, (3, 3), 2, 1),                    # fewer than a K-step's 16
    (8, 64, (40, 40), 16, (4, 4), 2, 4),
    (8, 32, (33, 35), 24, (3, 3), 2, 2),
    (4, 24, (4000,), 24, (7,), 2, 1),
    (2, 16, (24, 24, 24), 8, (3, 3, 3), 2, 1),
    (2, 16, (24, 24, 24), 16, (3, 3, 3), 2, 4),
], ids=str)
def test_fp32_strided_image_gradients_of_any_channels_are_as_close_as_sums_per_tap(geom):
    """Image gradients at strides, and the transposed convolution that is the same sum: the col matrix adds up one product per tap, and the
    host entry point forms it.  The phases' chains are no longer than that, so the two norms' ratio is 1 within some percent; one chain through all
    taps was 1.4 (3 x 3) to 2.7 (7 x 7)."""
    B, C, size, O, k, s, groups = geom
    nd, p = len(size), tuple(v // 2 for v in k)
    out = tuple((size[a] + 2 * p[a] - k[a]) // s + 1 for a in range(nd))
    x, w, g = randn((B, C) + size, torch.float32, 1), randn((O, C // groups) + k, torch.float32, 2, 0.05), randn((B, O) + out, torch.float32, 3)
    dx, _ = backward(nd)(x, w, g, stride=s, padding=p[0], groups=groups)
    rest = {size[a] - ((out[a] - 1) * s - 2 * p[a] + k[a]) for a in range(nd)}
    hx, hw, hg = (t.cpu().numpy() for t in (x, w, g))
    hdx, hdw = np.empty_like(hx), np.empty_like(hw)
    vp = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    geo = tuple(_arr(v) for v in (size, k, (s,) * nd, p, (1,) * nd))
    _lib.check(_lib.load().ntg_convnd_backward(_lib.FLOAT32, vp(hx), vp(hw), vp(hg), vp(hdx), vp(hdw), B, C, O, nd, *geo, groups, 0))
    want = exact_dx(size, w, g, k, (s,) * nd, p, (1,) * nd, groups)
    reference = relative(torch.from_numpy(hdx).to(DEV), want)
    assert relative(dx, want) <= 1.15 * reference, (relative(dx, want), reference)
    if len(rest) == 1:
        transposed = {1: F.conv_transpose1d, 2: F.conv_transpose2d, 3: F.conv_transpose3d}[nd]
        y = transposed(g, w, stride=s, padding=p[0], output_padding=rest.pop(), groups=groups)
        assert relative(y, want) <= 1.15 * reference, (relative(y, want), reference)


def test_fp32_weight_gradient_takes_the_large_tiles_where_they_are_faster(monkeypatch):
    """128 x 128 tiles take 77 % of the time of four 64 x 64 ones (profiles/conv_weight_gradient_gather_sweep.txt): the planned gradient of this
    layer is faster than fourteen ranges on 64 x 64 tiles (the knob's tile), which a plan that charged both alike chose; by 15 % without
    the copy of the image."""
    x, w, g = (randn(s, torch.float32, i) for i, s in enumerate(((64, 128, 28, 28), (128, 128, 3, 3), (64, 128, 28, 28))))
    call = lambda: F._conv2d_gradients(x, w, g, 1, 1, 1, 1, want_dx=False)[1]
    planned, small = [], []
    for _ in range(2):
        monkeypatch.delenv("NTG_DW_RANGES", raising=False)
        planned.append(microseconds(call))
        monkeypatch.setenv("NTG_DW_RANGES", "14")
        small.append(microseconds(call))
    assert min(planned) <= 0.96 * min(small), (planned, small)

"""Image gradients at a column stride of two: rows that are stored 16 bytes at a time from two pieces of a phase's row each.

The same call with an image that starts one element past a 16-byte boundary takes the element-wise path: the bits have to agree.  Values against
float64: one rounding to the type (2^-11 Float16, 2^-8 BFloat16, 2^-24 Float32, relative) of a sum whose k multiply-adds each err by 2^-24 of
sum |a||b| at most.  C added to is one rounding of (result + C) in Float32, exactly.
"""
import ctypes

import pytest
import torch

from neurotensor_amd import _lib
from neurotensor_amd import functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
UNIT = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}
GEOMS = [
    # (B, C, H, W, O, kh, kw, stride rows, padding rows, padding columns): rows of one piece, of several; a row that starts in either phase
    (2, 16, 4, 8, 16, 3, 3, 2, 1, 1),
    (1, 32, 5, 24, 32, 4, 4, 2, 1, 1),
    (2, 16, 6, 16, 32, 2, 2, 2, 0, 0),
    (3, 32, 3, 40, 16, 3, 1, 1, 1, 0),          # a column phase without taps
    (1, 16, 9, 56, 48, 5, 7, 3, 2, 3),
    (2, 16, 7, 64, 16, 1, 3, 2, 0, 2),          # a row phase without taps, padding wider than the window's half
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("geom", GEOMS, ids=lambda g: "x".join(map(str, g)))
def test_rows_from_two_column_phases(geom, dtype):
    B, C, H, W, O, kh, kw, sh, ph, pw = geom
    gen = torch.Generator().manual_seed(B + C + H + W)
    w = torch.randn(O, C, kh, kw, generator=gen).to(dtype)
    Ho, Wo = (H + 2 * ph - kh) // sh + 1, (W + 2 * pw - kw) // 2 + 1
    g = torch.randn(B, O, Ho, Wo, generator=gen).to(dtype)
    c0 = torch.randn(B, C, H, W, generator=gen).to(dtype)
    rows = (H - ((Ho - 1) * sh - 2 * ph + kh), W - ((Wo - 1) * 2 - 2 * pw + kw))
    exact = torch.nn.functional.conv_transpose2d(g.double(), w.double(), None, (sh, 2), (ph, pw), rows)
    terms = torch.nn.functional.conv_transpose2d(g.double().abs(), w.double().abs(), None, (sh, 2), (ph, pw), rows)
    lib = _lib.load()
    x, dw, dg, dk = torch.zeros(B, C, H, W, dtype=dtype, device=DEV), torch.zeros_like(w, device=DEV), g.to(DEV), w.to(DEV)
    geo = (B, C, H, W, O, kh, kw, sh, 2, ph, pw, 1, 1, 1)
    need = lib.ntg_conv2d_backward_workspace_bytes(F.ntg_dtype(x), *geo)
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=DEV)
    out = {}
    for accumulate in (0, 1):
        for shift in (0, 1):
            buf = torch.zeros(c0.numel() + 8, dtype=dtype, device=DEV)
            dx = buf[shift:shift + c0.numel()]
            dx.copy_(c0.reshape(-1))
            _lib.check(lib.ntg_conv2d_backward_dev(F.ntg_dtype(x), x.data_ptr(), dk.data_ptr(), dg.data_ptr(), dx.data_ptr(), dw.data_ptr(), ws.data_ptr(), need,
                                                   *geo, accumulate, torch.cuda.current_stream().cuda_stream))
            out[accumulate, shift] = dx.cpu().reshape(c0.shape)
            assert (buf[:shift] == 0).all() and (buf[shift + c0.numel():] == 0).all()
        assert torch.equal(out[accumulate, 0], out[accumulate, 1])
    got = out[0, 0]
    bound = UNIT[dtype] * exact.abs() + (O * kh * kw + 8) * 2.0 ** -24 * terms + (2.0 ** -24 if dtype == torch.float16 else 0)
    assert ((got.double() - exact).abs() <= bound).all()
    assert torch.equal(out[1, 0], (got.float() + c0.float()).to(dtype))


GEOMS3 = [
    # (B, C, (D, H, W), O, window, strides of the slower axes, padding)
    (1, 16, (4, 5, 16), 16, (3, 3, 4), (2, 1), (1, 1, 1)),
    (2, 32, (3, 4, 24), 16, (2, 3, 3), (1, 2), (0, 1, 1)),
    (1, 16, (5, 4, 8), 32, (3, 2, 1), (2, 2), (1, 0, 0)),         # a column phase without taps
    (1, 16, (3, 6, 48), 16, (1, 2, 5), (3, 1), (0, 1, 2)),        # slice phases without taps, columns that start in the second phase
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("geom", GEOMS3, ids=lambda g: "x".join(map(str, g[2])))
def test_rows_from_two_column_phases_over_three_axes(geom, dtype):
    B, C, size, O, window, slow, pad = geom
    stride = (*slow, 2)
    gen = torch.Generator().manual_seed(B + C + sum(size))
    outs = tuple((n + 2 * p - k) // s + 1 for n, p, k, s in zip(size, pad, window, stride))
    w, g = torch.randn(O, C, *window, generator=gen).to(dtype), torch.randn(B, O, *outs, generator=gen).to(dtype)
    c0 = torch.randn(B, C, *size, generator=gen).to(dtype)
    rest = tuple(n - ((o - 1) * s - 2 * p + k) for n, o, s, p, k in zip(size, outs, stride, pad, window))
    exact = torch.nn.functional.conv_transpose3d(g.double(), w.double(), None, stride, pad, rest)
    terms = torch.nn.functional.conv_transpose3d(g.double().abs(), w.double().abs(), None, stride, pad, rest)
    lib = _lib.load()
    arr = lambda v: (ctypes.c_int64 * 3)(*v)
    x, dw, dg, dk = torch.zeros(B, C, *size, dtype=dtype, device=DEV), torch.zeros_like(w, device=DEV), g.to(DEV), w.to(DEV)
    geo = (arr(size), arr(window), arr(stride), arr(pad), arr((1, 1, 1)))
    need = lib.ntg_convnd_fast_workspace_bytes(F.ntg_dtype(x), B, C, O, 3, *geo, 1, 1)
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=DEV)
    out = {}
    for accumulate in (0, 1):
        for shift in (0, 1):
            buf = torch.zeros(c0.numel() + 8, dtype=dtype, device=DEV)
            dx = buf[shift:shift + c0.numel()]
            dx.copy_(c0.reshape(-1))
            _lib.check(lib.ntg_convnd_backward_dev(F.ntg_dtype(x), x.data_ptr(), dk.data_ptr(), dg.data_ptr(), dx.data_ptr(), dw.data_ptr(), ws.data_ptr(), need,
                                                   B, C, O, 3, *geo, 1, accumulate, torch.cuda.current_stream().cuda_stream))
            out[accumulate, shift] = dx.cpu().reshape(c0.shape)
            assert (buf[:shift] == 0).all() and (buf[shift + c0.numel():] == 0).all()
        assert torch.equal(out[accumulate, 0], out[accumulate, 1])
    k = O * window[0] * window[1] * window[2]
    bound = UNIT[dtype] * exact.abs() + (k + 8) * 2.0 ** -24 * terms + (2.0 ** -24 if dtype == torch.float16 else 0)
    assert ((out[0, 0].double() - exact).abs() <= bound).all()
    assert torch.equal(out[1, 0], (out[0, 0].float() + c0.float()).to(dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("geom", [
    # rows shorter than a piece, a piece and one element, one less than two: the last piece moves back over the one before, or adds element by element
    (2, 16, 4, 3, 16, 3, 3, 2, 1, 1),
    (2, 16, 5, 7, 16, 3, 3, 2, 1, 1),
    (1, 32, 5, 9, 32, 4, 4, 2, 1, 1),
    (2, 16, 6, 15, 32, 2, 2, 2, 0, 0),
    (3, 32, 3, 17, 16, 3, 1, 1, 1, 0),
    (1, 16, 9, 52, 48, 5, 7, 3, 2, 3),
    (2, 16, 7, 41, 16, 1, 3, 2, 0, 2),
], ids=lambda g: "x".join(map(str, g)))
def test_rows_that_are_no_whole_pieces(geom, dtype):
    test_rows_from_two_column_phases(geom, dtype)

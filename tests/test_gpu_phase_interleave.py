"""Image gradients at a column stride of two: rows that are stored 16 bytes at a time from two pieces of a phase's row each.

The same call with an image that starts one element past a 16-byte boundary takes the element-wise path: the bits have to agree.  Values against
float64: one rounding to the type (2^-11 Float16, 2^-8 BFloat16, 2^-24 Float32, relative) of a sum whose k multiply-adds each err by 2^-24 of
sum |a||b| at most.  C added to is one rounding of (result + C) in Float32, exactly.
"""
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

"""The native side of functional.py (face/face.cpp) against the general Python ways: the same results, the same refusals."""
import os

import pytest
import torch

from neurotensor_amd import _lib
from neurotensor_amd import functional as F

gpu = pytest.mark.gpu


def both(monkeypatch, call):
    """What a call gives with the native side and without: tensors, or the exception's type and text."""
    def run():
        try:
            r = call()
        except Exception as e:
            return type(e), str(e)
        return r if isinstance(r, tuple) else (r,)
    assert F._face is not None
    native = run()
    monkeypatch.setattr(F, "_face", None)
    general = run()
    monkeypatch.undo()
    assert len(native) == len(general)
    for a, b in zip(native, general):
        if isinstance(b, torch.Tensor):
            assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b) and a.is_contiguous()
        else:
            assert a == b


def t(*shape, dtype=torch.float32, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed + sum(shape))
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


MATRICES = {
    "plain": lambda: (t(33, 40), t(40, 24)), "views of transposes": lambda: (t(40, 33).t(), t(24, 40).t()), "a row": lambda: (t(1, 40), t(40, 24)),
    "a column": lambda: (t(33, 40), t(40, 1)), "views with a side of one": lambda: (t(40, 1).t(), t(1, 40).t()), "slices": lambda: (t(33, 80)[:, ::2], t(80, 24)[::2]),
    "rows of a wider matrix": lambda: (t(33, 80)[:, :40], t(40, 24)), "batch": lambda: (t(3, 33, 40), t(3, 40, 24)), "batch, one right side": lambda: (t(3, 33, 40), t(40, 24)),
    "batch, one left side": lambda: (t(33, 40), t(5, 40, 24)), "batch of one": lambda: (t(1, 33, 40), t(1, 40, 24)), "batch of one against many": lambda: (t(1, 33, 40), t(4, 40, 24)),
    "two batch axes": lambda: (t(2, 3, 8, 40), t(2, 3, 40, 24)), "two against one": lambda: (t(2, 3, 8, 40), t(3, 40, 24)), "batched transposes": lambda: (t(3, 40, 33).mT, t(3, 40, 24)),
    "empty k": lambda: (t(3, 0), t(0, 4)), "empty rows": lambda: (t(0, 4), t(4, 5)), "empty batch": lambda: (t(0, 3, 4), t(0, 4, 5)), "wrong k": lambda: (t(3, 4), t(5, 6)),
    "a vector": lambda: (t(4), t(4, 3)), "two types": lambda: (t(3, 4), t(4, 5, dtype=torch.float16)), "outer sizes differ": lambda: (t(2, 3, 4), t(3, 4, 5)),
    "needs a gradient": lambda: (t(3, 4).requires_grad_(), t(4, 5)), "bool": lambda: (t(3, 4) > 0, t(4, 5) > 0), "split along k": lambda: (t(40, 2080, dtype=torch.bfloat16), t(2080, 704, dtype=torch.bfloat16)),
}


@gpu
@pytest.mark.parametrize("form", MATRICES)
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)], ids=["nn", "tt"])
def test_products(monkeypatch, form, ta, tb):
    a, b = MATRICES[form]()
    if ta and "empty" not in form:
        a, b = (a.transpose(-1, -2), b.transpose(-1, -2)) if a.dim() > 1 else (a, b)
    both(monkeypatch, lambda: F.matmult(a, b, None, ta, tb))


@gpu
@pytest.mark.parametrize("bias", [(24,), (1, 24), (33, 24), (1,), (33,), (2, 24)], ids=str)
@pytest.mark.parametrize("layer", [F.linear, F.linear_relu], ids=["linear", "relu"])
def test_linear(monkeypatch, bias, layer):
    x, w = t(33, 40), t(24, 40)
    both(monkeypatch, lambda: layer(x, w, t(*bias), False, True))
    both(monkeypatch, lambda: layer(x, w.t(), t(48)[::2], False, False))
    both(monkeypatch, lambda: layer(t(2, 33, 40), w, t(*bias), False, True))


CONVOLUTIONS = {
    1: ((2, 8, 20), (12, 8, 3)), 2: ((2, 8, 10, 9), (12, 8, 3, 3)), 3: ((2, 8, 5, 6, 7), (12, 8, 3, 3, 3)),
}


@gpu
@pytest.mark.parametrize("axes", CONVOLUTIONS)
@pytest.mark.parametrize("options", [
    {}, {"padding": 1}, {"stride": 2, "padding": 1, "dilation": 2}, {"groups": 2}, {"groups": 3}, {"groups": 0}, {"stride": 0}, {"padding": -1}, {"dilation": 9},
    {"stride": (2, 1), "padding": (1, 0)}, {"stride": [1, 2, 1]}, {"padding": True},
], ids=str)
def test_convolutions(monkeypatch, axes, options):
    forward, backward = {1: (F.conv1d, F.conv1d_backward), 2: (F.conv2d, F.conv2d_backward), 3: (F.conv3d, F.conv3d_backward)}[axes]
    xs, ws = CONVOLUTIONS[axes]
    groups = options.get("groups", 1)
    if groups == 2:
        ws = (12, 4) + ws[2:]
    for dtype in (torch.float32, torch.float16):
        x, w = t(*xs, dtype=dtype), t(*ws, dtype=dtype)
        both(monkeypatch, lambda: forward(x, w, **options))
        both(monkeypatch, lambda: forward(x.transpose(0, 1).contiguous().transpose(0, 1), w, **options))
        both(monkeypatch, lambda: forward(x[0], w, **options))
        try:
            y = forward(x, w, **options)
        except Exception:
            continue
        dy = t(*y.shape, dtype=dtype)
        both(monkeypatch, lambda: backward(x, w, dy, **options))
        both(monkeypatch, lambda: backward(x, w, dy.flatten(1), **options))


@gpu
@pytest.mark.parametrize("axes", [1, 2, 3])
@pytest.mark.parametrize("options", [{}, {"stride": 2}, {"stride": 2, "output_padding": 1}, {"stride": 2, "output_padding": 2}, {"groups": 2, "padding": 1}, {"padding": 40}, {"dilation": 2}], ids=str)
def test_transposed_convolutions(monkeypatch, axes, options):
    forward = {1: F.conv_transpose1d, 2: F.conv_transpose2d, 3: F.conv_transpose3d}[axes]
    backward = {1: F.conv_transpose1d_backward, 2: F.conv_transpose2d_backward, 3: F.conv_transposend_backward}[axes]
    x, w = t(2, 8, *(5, 6, 4)[:axes]), t(8, 6, *(3, 2, 3)[:axes])
    both(monkeypatch, lambda: forward(x, w, **options))
    try:
        y = forward(x, w, **options)
    except Exception:
        return
    dy = t(*y.shape)
    both(monkeypatch, lambda: backward(x, w, dy, **options))
    both(monkeypatch, lambda: backward(x, w, dy[..., :-1], **options))


def test_tensors_on_the_host_are_refused_as_before():
    with pytest.raises(ValueError, match="device memory"):
        F.matmult(torch.ones(2, 2), torch.ones(2, 2))
    with pytest.raises(ValueError, match="device memory"):
        F.conv2d(torch.ones(1, 1, 3, 3), torch.ones(1, 1, 1, 1))


def test_the_native_side_leaves_everything_but_plain_device_tensors_to_the_general_ways():
    assert F._face is not None
    m = torch.ones(2, 2)
    assert F._face.gemm(m, m, None, False, False, False, 0) is None
    assert F._face.gemm(m, [1], None, False, False, False, 0) is None
    assert F._face.conv(2, torch.ones(1, 1, 3, 3), torch.ones(1, 1, 1, 1), 1, 0, 1, 1, 0) is None
    assert F._face.conv(7, m, m, 1, 0, 1, 1, 0) is None
    assert F._face.conv_backward(2, m, m) is None


@gpu
@pytest.mark.parametrize("large", [2 ** 31, 2 ** 62, 2 ** 63 - 1], ids=hex)
def test_options_whose_sums_would_wrap_are_left_to_the_general_ways(large):
    """(2 x padding and dilation x (kernel - 1) of 2^63 - 1 are -2 in 64 bits: a geometry that looks sound.)"""
    for axes in (1, 2, 3):
        x, w = t(2, 8, *(8,) * axes), t(8, 8, *(3,) * axes)
        for options in ((1, large, 1, 1), (1, large, large, 1), (large, 0, large, 1), (1, 0, 1, large), (1, (large,) * axes, 1, 1)):
            assert F._face.conv(axes, x, w, *options, 0) is None, options
            assert F._face.conv_backward(axes, x, w, t(2, 8, *(6,) * axes), *options, 0) is None, options
            assert F._face.conv_backward(axes, x, w, t(0), *options, 0) is None, options
            s, p, d, groups = options
            assert F._face.conv_transpose(axes, x, w, s, p, 0, d, groups, 0) is None, options
            assert F._face.conv_transpose_backward(axes, x, w, t(2, 8, *(10,) * axes), *options, 0) is None, options
        assert F._face.conv_transpose(axes, x, w, 2, 0, large, 1, 1, 0) is None
    # two output sizes of 2^32 are no pixels in 64 bits
    assert F._face.conv_backward(2, t(2, 8, 8, 8), t(8, 8, 1, 1), t(0), 1, 2 ** 31 - 4, 1, 1, 0) is None


def test_a_native_side_that_does_not_load_is_done_without(monkeypatch, tmp_path):
    assert F._load_native() is not None
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libntgemm.so"))
    assert F._load_native() is None                                     # none there
    (tmp_path / "_face.so").write_bytes(b"built for something else")
    with pytest.warns(RuntimeWarning, match="_face.so does not load"):
        assert F._load_native() is None
    # another build of the library in the same directory: the native side calls libntgemm.so only
    monkeypatch.setattr(_lib, "LIB_PATH", os.path.join(os.path.dirname(_lib.__file__), "lib", "libntgemm_other.so"))
    assert F._load_native() is None

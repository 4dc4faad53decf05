"""The forms a convolution is computed in on the device, each against the sums in 64 bits: that every product is there once, at the edges of tiles, slots,
ranges and groups.  (The bound holds for any order of summation; what an order costs in precision is held to in test_gpu_conv_precision.py.)

The bound: an output of n products is rounded once to its type (unit roundoff u; Float16 below 2^-14: 2^-25) after a sum in 32 bits whose error
is at most n 2^-24 times the sum of the products' magnitudes.  Where parts of the sum are stored in the type on the way (the entries of a col
matrix, the products per image of a layer of one tap) each is rounded too: u times those magnitudes more."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from neurotensor_amd import _lib
from neurotensor_amd import functional as F

pytestmark = pytest.mark.gpu

UNIT = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}
CONV = {1: torch.nn.functional.conv1d, 2: torch.nn.functional.conv2d, 3: torch.nn.functional.conv3d}
TRANS = {1: torch.nn.functional.conv_transpose1d, 2: torch.nn.functional.conv_transpose2d, 3: torch.nn.functional.conv_transpose3d}
OURS = {(1, False): (F.conv1d, F.conv1d_backward), (2, False): (F.conv2d, F.conv2d_backward), (3, False): (F.conv3d, F.conv3d_backward),
        (1, True): (F.conv_transpose1d, F.conv_transpose1d_backward), (2, True): (F.conv_transpose2d, F.conv_transpose2d_backward),
        (3, True): (F.conv_transpose3d, F.conv_transposend_backward)}


def operands(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed, seed=1):
    gen = torch.Generator().manual_seed(seed)
    nd = len(size)
    wshape = ((cin, cout // groups) if transposed else (cout, cin // groups)) + (kernel,) * nd
    x = torch.randn((batch, cin) + size, generator=gen).to(dtype)
    w = (torch.randn(wshape, generator=gen) * 0.2).to(dtype)
    out = tuple((s - 1) * stride - 2 * pad + kernel if transposed else (s + 2 * pad - kernel) // stride + 1 for s in size)
    return x, w, torch.randn((batch, cout) + out, generator=gen).to(dtype)


def sums(x, w, dy, stride, pad, groups, transposed):
    """(y, dx, dw) in float64 on the CPU."""
    x, w = x.double().requires_grad_(), w.double().requires_grad_()
    y = (TRANS if transposed else CONV)[x.dim() - 2](x, w, stride=stride, padding=pad, groups=groups)
    dx, dw = torch.autograd.grad(y, (x, w), dy.double())
    return y.detach(), dx, dw


def check(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed, parts=()):
    x, w, dy = operands(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed)
    forward, backward = OURS[(len(size), transposed)]
    opt = {"stride": stride, "padding": pad, "groups": groups}
    dev = [t.cuda() for t in (x, w, dy)]
    got = (forward(dev[0], dev[1], **opt),) + tuple(backward(*dev, **opt))
    want = sums(x, w, dy, stride, pad, groups, transposed)
    mags = sums(x.abs(), w.abs(), dy.abs(), stride, pad, groups, transposed)
    taps = kernel ** len(size)
    terms = (cin // groups * taps, cout // groups * taps, batch * dy[0, 0].numel() if not transposed else batch * x[0, 0].numel())
    for name, g, r, m, n in zip(("y", "dx", "dw"), got, want, mags, terms):
        assert g.shape == r.shape and g.dtype == dtype
        bound = UNIT[dtype] * (r.abs() + (m if name in parts else 0.0)) + 2.0 ** -24 * (n + 32) * m + (2.0 ** -25 if dtype == torch.float16 else 0.0)
        err = (g.double().cpu() - r).abs()
        assert bool((err <= bound).all()), f"{name}: {float((err - bound).max())} over the bound"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("batch,cin,cout,size,kernel,stride,pad,groups,transposed,parts", [
    (2, 64, 96, (13, 11), 3, 1, 1, 2, False, ()),        # channels-last, ragged pixels
    (3, 128, 128, (17,), 5, 1, 2, 4, False, ()),
    (2, 64, 64, (5, 6, 7), 3, 1, 1, 2, False, ()),
    (3, 24, 32, (12, 12), 3, 2, 1, 4, False, ("dx",)),        # few channels a group: taps merged, image gradient through the col matrix
    (2, 256, 144, (8, 8), 1, 1, 0, 4, False, ("dw",)),        # one tap: plain products (36 out channels a group: the images' products are rounded)
    (5, 48, 48, (9, 9), 1, 1, 0, 3, False, ()),          # ... on rows that miss 16 bytes
    (2, 64, 96, (6, 6), 4, 2, 1, 2, True, ()),
    (2, 16, 16, (7, 5), 2, 2, 0, 4, True, ("y",)),
    (2, 30, 18, (10, 9), 3, 1, 1, 3, False, ()),         # element-wise gathers
], ids=str)
def test_groups_as_items_of_one_launch(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed, parts):
    check(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed, parts)


def test_a_batch_of_groups_split_in_two_launches_keeps_whole_images():
    """One round of 256 x 256 tiles and a rest: the first launch takes whole images of all groups, each group with its own weights."""
    batch, groups, c = 23, 3, 256
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((batch, groups * c, 32, 32), generator=gen, device="cuda").to(torch.bfloat16)
    w = (torch.randn((groups * c, c, 1, 1), generator=gen, device="cuda") * 0.1).to(torch.bfloat16)
    y = F.conv2d(x, w, groups=groups)
    for g in range(groups):
        part = slice(g * c, (g + 1) * c)
        assert torch.equal(y[:, part], F.conv2d(x[:, part].contiguous(), w[part].contiguous()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("batch,cin,cout,size,kernel,stride,pad,groups,transposed", [
    (1, 64, 1, (127,), 3, 1, 1, 1, False),           # 32 x 128 tiles: one row, one column short of a tile
    (2, 32, 32, (129,), 5, 1, 2, 1, False),          # ... all rows, one column more
    (3, 64, 33, (12, 12), 3, 1, 1, 1, False),        # one row too many
    (2, 32, 17, (4, 5, 7), 3, 1, 1, 1, False),        # (out channels padded for the weight gradient)
    (1040, 32, 31, (33,), 3, 1, 1, 1, False),        # 16 bits: 32 x 256 tiles
    (2, 16, 96, (9, 10), 3, 2, 1, 1, False),         # image gradient by phases
    (2, 64, 64, (16, 8), 4, 2, 1, 2, True),
    (2, 20, 32, (4, 6, 6), 2, 2, 0, 1, False),
    (2, 96, 96, (11, 12), 3, 1, 1, 1, False),        # Float32: three rows of flat tiles
], ids=str)
def test_flat_tiles(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed):
    check(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed)


@pytest.mark.parametrize("size,kernel,stride,pad,dil", [
    ((7,), (3,), (2,), (1,), (1,)), ((9,), (2,), (4,), (0,), (1,)),                     # (positions that no window reaches)
    ((6, 9), (3, 5), (2, 1), (1, 2), (1, 1)),
    ((5, 6, 7), (4, 4, 4), (2, 2, 2), (1, 1, 1), (1, 1, 1)), ((4, 8, 3), (1, 1, 1), (2, 2, 2), (0, 0, 0), (1, 1, 1)),
    ((3, 5, 20), (2, 3, 9), (1, 3, 2), (0, 1, 5), (1, 1, 1)), ((6, 5, 7), (2, 3, 2), (1, 2, 1), (1, 0, 2), (2, 1, 1)),      # (dilated: the general kernel)
    ((3, 4, 3, 5), (2, 2, 3, 3), (1, 2, 1, 2), (1, 0, 1, 1), (1, 1, 1, 1)),
], ids=str)
def test_col_matrix_back_onto_an_image_in_tap_order(size, kernel, stride, pad, dil):
    """Up to four axes, bit for bit: every position adds its taps in ascending order."""
    nd, batch, channels = len(size), 2, 3
    out = [(s + 2 * p - d * (k - 1) - 1) // st + 1 for s, k, st, p, d in zip(size, kernel, stride, pad, dil)]
    rng = np.random.default_rng(5)
    col = rng.standard_normal((batch, channels * int(np.prod(kernel)), int(np.prod(out)))).astype(np.float32)
    arr = lambda v: (ctypes.c_int64 * nd)(*v)
    image = torch.empty((batch, channels) + size, device="cuda")
    _lib.check(_lib.load().ntg_unfoldnd_backward_dev(_lib.FLOAT32, torch.from_numpy(col).cuda().data_ptr(), image.data_ptr(), batch, channels, nd, arr(size), arr(kernel),
                                                     arr(stride), arr(pad), arr(dil), 0, torch.cuda.current_stream().cuda_stream))
    want = oracle.unfoldnd_backward(col, size, kernel, dil, pad, stride)
    assert np.array_equal(image.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("batch,cin,cout,size,kernel,stride,pad,groups,transposed", [
    (3, 16, 1, (9, 9), 3, 1, 1, 1, False),           # one out channel, planes that miss 16 bytes
    (2, 1, 9, (11, 7), 5, 1, 2, 1, False),           # one channel
    (2, 24, 21, (13,), 3, 2, 1, 3, False),
    (2, 8, 10, (5, 5, 5), 3, 1, 1, 2, False),
    (1, 6, 260, (15, 15), 3, 1, 1, 1, False),
    (2, 18, 24, (6, 5), 4, 2, 1, 2, True),
], ids=str)
def test_weight_gradients_of_odd_planes_and_channels(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed):
    parts = ("dx",) if stride > 1 and not transposed else ("y",) if transposed else ()      # (through the col matrix)
    check(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed, parts)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("batch,cin,cout,size,groups", [
    (1, 16, 16, (256,), 1), (2, 64, 136, (8, 24), 1), (3, 32, 48, (20, 10), 2), (1, 8, 264, (1024,), 1), (5, 24, 8, (4, 6), 1),
], ids=str)
def test_weight_gradient_of_one_tap_in_ranges(dtype, batch, cin, cout, size, groups):
    check(dtype, batch, cin, cout, size, 1, 1, 0, groups, False)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=["f16", "f32"])
@pytest.mark.parametrize("batch,cin,cout,size,kernel,stride,pad,groups,transposed", [
    (3, 64, 64, (9, 15), 3, 1, 1, 1, False),         # planes that miss 16 bytes: the last piece of a row element by element
    (2, 72, 72, (63,), 5, 1, 2, 1, False),           # a tile and a part in each direction
    (2, 65, 70, (13, 5), 3, 1, 3, 5, False),         # padded channels of five groups in one tile, a border wider than the window
    (4, 3, 64, (10, 9), 5, 1, 2, 1, False),          # a thread a pixel
    (1, 5, 16, (300,), 7, 2, 3, 1, False),
    (2, 64, 64, (3, 4, 5), 3, 1, 1, 1, False),       # slices in front and behind
    (2, 32, 64, (7, 6, 5), 3, 3, 1, 2, False),       # phases of stride 3: their weights and table beside the copies
    (1, 64, 48, (2, 3), 4, 4, 0, 1, True),
], ids=str)
def test_copies_borders_and_weights_in_one_launch(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed):
    parts = ("dx",) if stride > 1 and not transposed else ()
    check(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed, parts)


def test_tensors_at_any_element_of_a_buffer():
    """Images, weights and gradients two bytes off any alignment."""
    gen = torch.Generator(device="cuda").manual_seed(4)
    x, w, dy = (torch.randn(s, generator=gen, device="cuda").to(torch.bfloat16) for s in ((2, 40, 12, 12), (24, 40, 3, 3), (2, 24, 12, 12)))
    off = []
    for t in (x, w, dy):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
        buf[1:].copy_(t.flatten())
        off.append(buf[1:].view(t.shape))
    assert torch.equal(F.conv2d(off[0], off[1], padding=1), F.conv2d(x, w, padding=1))
    dx, _ = F.conv2d_backward(*off, padding=1)
    assert torch.equal(dx, F.conv2d_backward(x, w, dy, padding=1)[0])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("batch,cin,cout,size,kernel,stride,pad,groups,transposed", [
    (2, 1, 1, (9, 15), 3, 1, 1, 1, False),           # one slot a tap, nine taps: K-steps across tap rows, a last one of a single slot
    (2, 24, 40, (8, 9), 3, 1, 1, 1, False),          # three and five slots (Float32: six and ten)
    (1, 3, 33, (40, 33), 7, 2, 3, 1, False),
    (3, 20, 12, (60,), 5, 1, 2, 1, False),
    (2, 12, 24, (6, 5, 7), 3, 1, 1, 2, False),       # three axes, two groups
    (2, 24, 16, (12, 11), 3, 1, 2, 1, False),        # dilated windows below
    (1, 48, 12, (5, 5, 6), 2, 2, 0, 3, False),       # phases
    (5, 36, 20, (6, 5), 4, 2, 1, 1, True),
    (2, 8, 24, (129, 1), 1, 1, 0, 1, False),         # one tap: a K-step that is mostly past the end
    (1, 40, 300, (12, 12), 3, 1, 1, 1, False),       # larger tiles
], ids=str)
def test_taps_in_slots(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed):
    parts = ("dx", "y") if stride > 1 or transposed else ("dw", "y", "dx") if kernel == 1 else ()
    check(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed, parts)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("batch,cin,cout,size,kernel,stride,pad,groups,transposed", [
    (8, 104, 8, (64, 63), 3, 1, 1, 1, False), (8, 104, 8, (64, 64), 3, 1, 1, 1, False),      # 13 slots of 16: under 32768 pixels and from there
    (2, 8, 136, (64, 63), 3, 1, 1, 1, False), (2, 8, 136, (64, 64), 3, 1, 1, 1, False),      # 17 of 20, the image gradient: 8192
    (1, 104, 24, (16, 16, 31), 3, 1, 1, 1, False), (1, 104, 24, (16, 16, 32), 3, 1, 1, 1, False),
    (2, 24, 104, (128, 128), 3, 2, 1, 1, False),                                             # the phases of 32768 image pixels
    (2, 208, 16, (64, 64), 2, 2, 0, 2, True),
], ids=str)
def test_wide_groups_in_slots_or_whole_runs(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed):
    check(dtype, batch, cin, cout, size, kernel, stride, pad, groups, transposed)


def test_taps_in_slots_dilated_and_the_longest_table():
    gen = torch.Generator(device="cuda").manual_seed(6)
    for shape, w, opt in (((2, 24, 20, 20), (8, 24, 3, 3), {"dilation": 3, "padding": 3}), ((1, 40, 12, 12), (8, 40, 8, 8), {"padding": 3}),
                          ((1, 328, 12, 12), (8, 328, 7, 7), {"padding": 3})):          # 320 and 2009 slots; 2048 at most
        x = torch.randn(shape, generator=gen, device="cuda").to(torch.bfloat16)
        k = torch.randn(w, generator=gen, device="cuda").to(torch.bfloat16)
        want = torch.nn.functional.conv2d(x.double().cpu(), k.double().cpu(), **opt)
        mags = torch.nn.functional.conv2d(x.double().abs().cpu(), k.double().abs().cpu(), **opt)
        err = (F.conv2d(x, k, **opt).double().cpu() - want).abs()
        assert bool((err <= 2.0 ** -8 * want.abs() + 2.0 ** -24 * (k[0].numel() + 32) * mags).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("batch,cin,cout,size,kernel,stride,pad", [
    (2, 256, 65, (13, 5), 3, 1, 1),                  # a tile and a part in each direction
    (1, 256, 256, (9,), 7, 1, 3),                    # pixels that miss the rows of the sums
    (3, 320, 24, (11, 12), 3, 2, 1),                 # five ranges in 16 bits; strides
    (1, 64, 30, (9, 9), 7, 1, 3),                    # flat tiles; two ranges in 16 bits
    (1, 128, 64, (4, 5, 6), 3, 1, 1),
], ids=str)
def test_channels_in_ranges(dtype, batch, cin, cout, size, kernel, stride, pad):
    check(dtype, batch, cin, cout, size, kernel, stride, pad, 1, False, ("dx",) if stride > 1 else ())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("batch,cin,cout,size,kernel,stride,pad,groups", [
    (2, 256, 130, (13, 5), 5, 1, 2, 2),              # 65 rows a group
    (3, 192, 9, (9, 10), 5, 2, 2, 3),                # three rows a group
    (1, 256, 128, (5, 6, 7), 3, 2, 1, 4),
    (2, 512, 32, (11,), 7, 1, 3, 2),                 # (an axis of more than eight taps has no such form: its image gradient goes through a col matrix)
    (4, 1, 256, (8, 8), 7, 1, 3, 1),                 # a border of twice the map
    (2, 128, 96, (8, 8), 7, 1, 3, 2),
], ids=str)
def test_channels_of_groups_in_ranges(dtype, batch, cin, cout, size, kernel, stride, pad, groups):
    check(dtype, batch, cin, cout, size, kernel, stride, pad, groups, False, ("dx",) if stride > 1 else ())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("ranges", [None, "0", "1"])
@pytest.mark.parametrize("batch,cin,cout,size,kernel,stride,pad,groups", [
    (3, 16, 16, (1600,), 3, 1, 1, 1),            # chunks of 512 pixels that images cross, one row of flat tiles
    (2, 24, 33, (40, 40), 3, 1, 1, 1),           # one row past a flat tile
    (5, 8, 64, (32, 32), 5, 1, 2, 1),            # 200 columns: a wide tile and part of one
    (2, 32, 65, (65, 63), 3, 2, 1, 1),           # strides, one row past a tile
    (2, 16, 48, (12, 16, 20), 3, 1, 1, 2),       # three axes, groups of 24 rows
    (1, 8, 8, (23, 41), 1, 1, 0, 1),             # under two chunks
    (40, 64, 128, (8, 8), 3, 1, 1, 1),           # many images a chunk
])
def test_weight_gradients_through_the_table_of_pixels(monkeypatch, dtype, ranges, batch, cin, cout, size, kernel, stride, pad, groups):
    """As planned, one product an image, and one range over all images (the last two where the gradient's rows allow)."""
    if ranges is not None:
        monkeypatch.setenv("NTG_DW_RANGES", ranges)
    check(dtype, batch, cin, cout, size, kernel, stride, pad, groups, False)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_channels_in_ranges_with_the_columns_split(dtype):
    """289 output pixels of 1536 rows of partial sums go out as 256 columns and a rest, whose sums start 256 Float32 elements in."""
    x, w, _ = operands(dtype, 8, 256, 192, (17, 17), 7, 1, 3, 1, False)
    got = F.conv2d(x.cuda(), w.cuda(), padding=3)[::7].double().cpu()
    want, mags = (CONV[2](a.double(), b.double(), padding=3) for a, b in ((x[::7], w), (x[::7].abs(), w.abs())))
    bound = UNIT[dtype] * want.abs() + 2.0 ** -24 * (256 * 49 + 32) * mags + (2.0 ** -25 if dtype == torch.float16 else 0.0)
    assert bool(((got - want).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("cin,cout,size,kernel,batches", [
    (256, 256, (13, 13), 3, (1, 9, 10)),             # 12 tiles an image
    (256, 256, (16, 16), 3, (1, 6, 7, 8)),           # 16: 128 of them
    (512, 32, (9,), 3, (1, 2, 128)),
    (64, 64, (11, 11), 7, (1, 3, 64)),
], ids=str)
def test_an_image_is_the_same_bits_alone_and_among_others(dtype, cin, cout, size, kernel, batches):
    """Channels in ranges, up to 128 tiles in all: forward product and image gradient."""
    x, w, dy = (t.cuda() for t in operands(dtype, max(batches), cin, cout, size, kernel, 1, kernel // 2, 1, False))
    forward, backward = OURS[(len(size), False)]
    opt = {"padding": kernel // 2}
    alone = [(forward(x[i:i + 1], w, **opt)[0], backward(x[i:i + 1], w, dy[i:i + 1], **opt)[0][0]) for i in (0, max(batches) - 1)]
    for n in batches:
        y, dx = forward(x[:n], w, **opt), backward(x[:n], w, dy[:n], **opt)[0]
        assert torch.equal(y[0], alone[0][0]) and torch.equal(dx[0], alone[0][1]), n
    assert torch.equal(y[-1], alone[1][0]) and torch.equal(dx[-1], alone[1][1])

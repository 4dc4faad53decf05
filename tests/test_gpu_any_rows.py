"""Products whose rows start anywhere (odd sizes, views inside a 16-byte chunk): whole and cut into k ranges, at the edges of tiles, K-steps and chunks.

Exact for Int8 (wrapping) and Float32 without a workspace (the reference's chain, bit for bit).  Otherwise against the product in 64 bits: one
rounding to the type (half a last place: 2^-11 Float16, 2^-8 BFloat16, relative) on a sum whose k multiply-adds each err by 2^-24 of sum |a||b| at most.
"""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from neurotensor_amd import _lib
from neurotensor_amd import functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "i8": torch.int8}
UNIT = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8, "f32": 2.0 ** -24}
TRANS = [(False, False), (False, True), (True, False), (True, True)]
# one element past / before a tile, a K-step, a chunk; one row; the shortest rows that hold a chunk; k ranges with a short last one
SIZES = [(33, 17, 17), (63, 65, 64), (64, 63, 65), (65, 129, 127), (40, 16, 19), (1, 33, 18), (129, 257, 31), (1700, 40, 1030),
         (70, 2049, 66), (37, 3001, 130), (200, 1100, 77), (1025, 401, 2049)]


def values(shape, name, gen):
    if name == "i8":
        return torch.randint(-128, 128, shape, dtype=torch.int8, generator=gen)
    return torch.randn(*shape, generator=gen).to(DTYPES[name])


def check(got, a, b, c0, name, k):
    if name == "i8":
        want = torch.matmul(a.double(), b.double()).to(torch.int64) + (0 if c0 is None else c0.to(torch.int64))
        assert torch.equal(((want + 128) % 256 - 128).to(torch.int8), got)
        return
    exact = torch.matmul(a.double(), b.double()) + (0 if c0 is None else c0.double())
    terms = torch.matmul(a.double().abs(), b.double().abs()) + (0 if c0 is None else c0.double().abs())
    bound = UNIT[name] * exact.abs() + (k + 40) * 2.0 ** -24 * terms + (2.0 ** -24 if name == "f16" else 0)      # (40: the sums of k ranges; Float16's smallest step)
    assert ((got.double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("name", sorted(DTYPES))
@pytest.mark.parametrize("ta,tb", TRANS)
def test_sizes_at_the_edges(name, ta, tb):
    gen = torch.Generator().manual_seed(5)
    for m, k, n in SIZES:
        a, b = values((k, m) if ta else (m, k), name, gen), values((n, k) if tb else (k, n), name, gen)
        got = F.matmult(a.to(DEV), b.to(DEV), None, ta, tb).cpu()
        check(got, a.t() if ta else a, b.t() if tb else b, None, name, k)


@pytest.mark.parametrize("name", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("ta,tb", TRANS)
def test_infinities_stay_in_their_row_and_column(name, ta, tb):
    """What a chunk on the edge reads of the next k-row reaches no sum."""
    gen = torch.Generator().manual_seed(9)
    for m, k, n in ((67, 300, 69), (131, 1100, 130)):
        a, b = values((m, k), name, gen).abs() + 1, values((k, n), name, gen).abs() + 1
        a[0, 1:] = float("inf")
        b[1:, 0] = float("inf")
        got = F.matmult((a.t() if ta else a).contiguous().to(DEV), (b.t() if tb else b).contiguous().to(DEV), None, ta, tb).cpu()
        assert torch.isinf(got[0]).all() and torch.isinf(got[:, 0]).all() and torch.isfinite(got[1:, 1:]).all()


@pytest.mark.parametrize("name", sorted(DTYPES))
def test_batches_pitches_and_what_is_added_to(name):
    """Items of a batch are the same bits alone, rows lie further apart than they are long, C is added to and starts inside a chunk."""
    lib = _lib.load()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    gen = torch.Generator().manual_seed(6)
    for m, k, n, batch in ((66, 70, 37, 3), (45, 2051, 97, 3), (45, 2051, 97, 160)):       # (160: the ranges of a float inside a workgroup)
        lda, ldb, ldc = k + 2, n + 1, n + 3
        a, b, c0 = values((batch, m, lda), name, gen), values((batch, k, ldb), name, gen), values((1 + batch * m * ldc,), name, gen)
        ta, tb, one = a.to(DEV), b.to(DEV), c0.to(DEV)
        both = [c0.to(DEV), one]
        for c, items in ((both[0], [(0, batch)]), (both[1], [(i, 1) for i in range(batch)])):
            for first, count in items:
                d = _lib.GemmDesc()
                d.dtype, d.c_mode, d.m, d.k, d.n, d.batches = F.ntg_dtype(ta), _lib.C_ACCUMULATE, m, k, n, count
                d.lda, d.ldb, d.ldc, d.stride_a, d.stride_b, d.stride_c = lda, ldb, ldc, m * lda, k * ldb, m * ldc
                need = lib.ntg_gemm_workspace_bytes(ctypes.byref(d))
                ws = torch.empty(max(need, 1), dtype=torch.uint8, device=DEV)
                d.workspace, d.workspace_bytes = ws.data_ptr(), need
                es = c.element_size()
                _lib.check(lib.ntg_gemm_dev(ctypes.byref(d), ta[first].data_ptr(), tb[first].data_ptr(), c.data_ptr() + (1 + first * m * ldc) * es, st))
        torch.cuda.synchronize()
        assert torch.equal(both[0].view(torch.uint8), both[1].view(torch.uint8))
        got, before = both[0].cpu()[1:].view(batch, m, ldc), c0[1:].view(batch, m, ldc)
        assert torch.equal(got[..., n:], before[..., n:])                # what lies between the rows stays
        check(got[..., :n], a[..., :k], b[..., :n], before[..., :n], name, k)


def product(lib, a, b, c, m, k, n, batch, strides, ta, tb, mode, bias=None, relu=False, entry="dev", first=0):
    """Items first .. first + batch - 1 of one call; the bytes of workspace that it was offered."""
    es = c.element_size()
    d = _lib.GemmDesc()
    d.dtype, d.transpose_a, d.transpose_b, d.c_mode = F.ntg_dtype(c), int(ta), int(tb), mode
    d.m, d.k, d.n, d.batches = m, k, n, batch
    d.stride_a, d.stride_b, d.stride_c = strides
    if bias is not None:
        d.bias, d.bias_batch_stride, d.bias_col_stride = bias.data_ptr() + first * n * es, n, 1
    need = lib.ntg_gemm_workspace_bytes(ctypes.byref(d))
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=DEV)
    if entry == "dev":
        d.workspace, d.workspace_bytes = ws.data_ptr(), need
    call = lib.ntg_gemm_noalloc_dev if entry == "noalloc" else lib.ntg_gemm_relu_dev if relu else lib.ntg_gemm_dev
    _lib.check(call(ctypes.byref(d), a.data_ptr() + first * strides[0] * es, b.data_ptr() + first * strides[1] * es, c.data_ptr() + first * strides[2] * es,
                    ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    return need


# batches that fill the chip by themselves; ranges of whole and of broken length, a last K-step that is cut
FULL = [(70, 2049, 66, 200), (129, 2057, 130, 64), (200, 2501, 77, 70), (40, 3001, 201, 200), (128, 2002, 250, 130)]


@pytest.mark.parametrize("name", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("ta,tb", TRANS)
def test_a_batch_that_fills_the_chip_takes_no_room_and_gives_the_bits_of_its_items(name, ta, tb):
    lib = _lib.load()
    gen = torch.Generator().manual_seed(12)
    for (m, k, n, batch), mode, relu, shared in zip(FULL, (_lib.C_ACCUMULATE, _lib.C_BIAS, _lib.C_OVERWRITE, _lib.C_BIAS, _lib.C_ACCUMULATE),
                                                    (False, True, False, False, True), (False, False, True, True, False)):
        a, b = values((batch, m, k), name, gen), values((1 if shared else batch, k, n), name, gen)
        c0, bias = values((batch, m, n), name, gen), values((batch, n), name, gen)
        da, db = (a.transpose(1, 2) if ta else a).contiguous().to(DEV), (b.transpose(1, 2) if tb else b).contiguous().to(DEV)
        dbias = bias.to(DEV) if mode == _lib.C_BIAS else None
        strides = (m * k, 0 if shared else k * n, m * n)
        together, alone = c0.to(DEV), c0.to(DEV)
        room = product(lib, da, db, together, m, k, n, batch, strides, ta, tb, mode, dbias, relu)
        some = [0, 1, batch // 2, batch - 1]
        for i in some:
            one = product(lib, da, db, alone, m, k, n, 1, strides, ta, tb, mode, dbias, relu, first=i)
            assert one >= 2 * m * n * 4 and room == 256                  # the item alone is cut into ranges that go through memory
            assert torch.equal(together[i].view(torch.uint8), alone[i].view(torch.uint8)), (m, k, n, i)
        start = c0 if mode == _lib.C_ACCUMULATE else bias[:, None, :].expand(batch, m, n) if mode == _lib.C_BIAS else torch.zeros_like(c0)
        if relu:
            assert (together >= 0).all() and (together > 0).any()
        else:
            check(together.cpu()[some], a[some], b.expand(batch, k, n)[some], start[some], name, k)
            unallocated = c0.to(DEV)
            product(lib, da, db, unallocated, m, k, n, batch, strides, ta, tb, mode, dbias, entry="noalloc")
            assert torch.equal(unallocated.view(torch.uint8), together.view(torch.uint8))


@pytest.mark.parametrize("name", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("relu", [False, True])
def test_bias_and_relu(name, relu):
    gen = torch.Generator().manual_seed(7)
    for m, k, n in ((37, 67, 129), (65, 2001, 100), (300, 300, 333)):
        x, w, bias = values((m, k), name, gen), values((n, k), name, gen), values((n,), name, gen)
        got = (F.linear_relu if relu else F.linear)(x.to(DEV), w.to(DEV), bias.to(DEV), False, True).cpu()
        if relu:
            assert (got >= 0).all()
            keep = got > 0
            plain = F.linear(x.to(DEV), w.to(DEV), bias.to(DEV), False, True).cpu()
            assert torch.equal(got, torch.where(plain > 0, plain, torch.zeros_like(plain))) and keep.any()
        else:
            check(got, x, w.t(), bias, name, k)


def test_float32_without_workspace_is_the_reference_chain_bit_for_bit():
    lib = _lib.load()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rng = np.random.default_rng(8)
    for (m, k, n), (ta, tb) in zip(((65, 67, 130), (70, 131, 33), (130, 35, 65), (61, 1003, 63)), TRANS):
        a, b, c0 = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (k, n), (m, n)))
        sa, sb = np.ascontiguousarray(a.T) if ta else a, np.ascontiguousarray(b.T) if tb else b
        da, db, dc = (torch.from_numpy(v).to(DEV) for v in (sa, sb, c0))
        d = _lib.GemmDesc()
        d.dtype, d.transpose_a, d.transpose_b, d.c_mode = _lib.FLOAT32, int(ta), int(tb), _lib.C_ACCUMULATE
        d.m, d.k, d.n, d.batches = m, k, n, 1
        _lib.check(lib.ntg_gemm_dev(ctypes.byref(d), da.data_ptr(), db.data_ptr(), dc.data_ptr(), st))
        want = oracle.matmult2d(sa, sb, c0.copy(), ta, tb)
        assert np.array_equal(dc.cpu().numpy().view(np.uint32), want.view(np.uint32))


INTS = {"i16": (np.int16, torch.int16), "i32": (np.int32, torch.int32), "i64": (np.int64, torch.int64)}


@pytest.mark.parametrize("name", sorted(INTS))
@pytest.mark.parametrize("ta,tb", TRANS)
def test_wide_integers_from_digits(name, ta, tb):
    """The whole range of values, wrapping: edges of tiles, K-steps and groups of eight, k ranges, both tile heights, a broadcast operand, C added to."""
    rng = np.random.default_rng(9)
    npdt, dt = INTS[name]
    full = lambda *shape: rng.integers(-2**63, 2**63 - 1, shape, dtype=np.int64, endpoint=True).astype(npdt)
    for m, k, n, batch in ((33, 9, 8, 1), (8, 8, 9, 1), (63, 33, 65, 1), (65, 31, 63, 2), (1, 40, 70, 1), (129, 64, 66, 1), (140, 1031, 150, 1), (200, 40, 299, 64), (5, 7, 6, 1)):
        lead = (batch,) if batch > 1 else ()
        a, b = full(*lead, *((k, m) if ta else (m, k))), full(*((n, k) if tb else (k, n)))
        c0 = full(*lead, m, n)
        a[..., 0, 0], b[0, 0] = np.iinfo(npdt).min, np.iinfo(npdt).min
        A = (np.swapaxes(a, -1, -2) if ta else a).astype(np.int64).view(np.uint64)
        B = (b.T if tb else b).astype(np.int64).view(np.uint64)
        want = A @ B
        got = F.matmult(torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV), None, ta, tb).cpu().numpy()
        assert np.array_equal(got, want.astype(npdt)), (m, k, n)
        out = torch.from_numpy(c0.copy()).to(DEV)
        F.matmult(torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV), out, ta, tb)
        assert np.array_equal(out.cpu().numpy(), (want + c0.astype(np.int64).view(np.uint64)).astype(npdt)), (m, k, n)


@pytest.mark.parametrize("name", sorted(INTS))
@pytest.mark.parametrize("ta,tb", TRANS)
def test_wide_integers_with_a_side_under_a_tile_are_cut_into_k_ranges(name, ta, tb):
    """Few tiles and a deep k, down to the smallest sides; the last range is shorter than a group of eight."""
    lib = _lib.load()
    rng = np.random.default_rng(10)
    npdt, dt = INTS[name]
    full = lambda *shape: rng.integers(-2**63, 2**63 - 1, shape, dtype=np.int64, endpoint=True).astype(npdt)
    for m, n, batch in ((64, 64, 1), (8, 8, 1), (9, 300, 1), (40, 70, 3)):
        d = _lib.GemmDesc()
        d.dtype, d.transpose_a, d.transpose_b, d.m, d.n, d.batches = F.ntg_dtype(torch.empty(0, dtype=dt)), int(ta), int(tb), m, n, batch
        for k in range(1300, 1500):
            d.k, d.stride_a, d.stride_b, d.stride_c = k, m * k, k * n, m * n
            ranges = lib.ntg_gemm_workspace_bytes(ctypes.byref(d)) // (batch * m * ((n + 3) // 4 * 4) * np.dtype(npdt).itemsize)
            assert ranges >= 2
            steps = (k + 31) // 32
            if 0 < k - (ranges - 1) * -(-steps // ranges) * 32 < 8:
                break
        else:
            assert False, "no k with a short last range"
        a, b, c0 = full(batch, *((k, m) if ta else (m, k))), full(batch, *((n, k) if tb else (k, n))), full(batch, m, n)
        A = (np.swapaxes(a, -1, -2) if ta else a).astype(np.int64).view(np.uint64)
        B = (np.swapaxes(b, -1, -2) if tb else b).astype(np.int64).view(np.uint64)
        out = torch.from_numpy(c0.copy()).to(DEV)
        F.matmult(torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV), out, ta, tb)
        assert np.array_equal(out.cpu().numpy(), (A @ B + c0.astype(np.int64).view(np.uint64)).astype(npdt)), (m, k, n)


def test_int64_of_few_k_on_either_side_of_the_line():
    """16 and 17 k on 256 and more tiles: the vector ALU's kernel and the digits give the wrapping result."""
    rng = np.random.default_rng(11)
    for m, k, n, batch in ((1024, 16, 1024, 1), (1025, 16, 1024, 1), (1025, 17, 1024, 1), (70, 8, 40, 200), (16, 17, 16, 300)):
        a, b = (rng.integers(-2**63, 2**63 - 1, s, dtype=np.int64, endpoint=True) for s in ((batch, m, k), (batch, k, n)))
        got = F.matmult(torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV)).cpu().numpy()
        assert np.array_equal(got, (a.view(np.uint64) @ b.view(np.uint64)).view(np.int64)), (m, k, n, batch)


@pytest.mark.parametrize("name", sorted(DTYPES) + sorted(INTS))
@pytest.mark.parametrize("ta,tb", TRANS)
def test_lists_behind_pointer_tables_have_the_bits_of_their_items(name, ta, tb):
    """Repeated pointers in no order, entries inside a chunk, C added to: one launch for a long list; a list whose items are split
    along k on 16-byte rows is refused."""
    lib = _lib.load()
    rng, gen = np.random.default_rng(13), torch.Generator().manual_seed(13)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    if name in INTS:
        draw = lambda *s: torch.from_numpy(rng.integers(-2**63, 2**63 - 1, s, dtype=np.int64, endpoint=True).astype(INTS[name][0]))
    else:
        draw = lambda *s: values(s, name, gen)
    m, k, n, mats = 67, 4051, 97, 3
    d = _lib.GemmDesc()
    d.transpose_a, d.transpose_b, d.c_mode, d.m, d.k, d.n = int(ta), int(tb), _lib.C_ACCUMULATE, m, k, n
    a, b = draw(mats, m * k + 3), draw(mats, k * n + 3)                  # (odd pitches: the matrices start anywhere)
    da, db = a.to(DEV), b.to(DEV)
    d.dtype = F.ntg_dtype(da)
    for items in (60, 2):
        d.flags, d.batches = _lib.GEMM_PTRS_ITEM_ORDER, items
        ia, ib = rng.integers(0, mats, items), rng.integers(0, mats, items)
        c0 = draw(items, m * n + 1)
        c, alone = c0.to(DEV), c0.to(DEV)
        need = lib.ntg_gemm_workspace_bytes(ctypes.byref(d))
        assert need == 0 or items == 2
        tab = torch.tensor([da[i].data_ptr() for i in ia] + [db[i].data_ptr() for i in ib] + [x.data_ptr() for x in c], dtype=torch.int64, device=DEV)
        _lib.check(lib.ntg_gemm_ptrs_dev(ctypes.byref(d), tab.data_ptr(), tab.data_ptr() + 8 * items, tab.data_ptr() + 16 * items, st))
        d.flags, d.batches = 0, 1
        one = lib.ntg_gemm_workspace_bytes(ctypes.byref(d))
        assert one > 0 and need in (0, one)
        ws = torch.empty(one, dtype=torch.uint8, device=DEV)
        d.workspace, d.workspace_bytes = ws.data_ptr(), one
        for j in range(items):
            _lib.check(lib.ntg_gemm_dev(ctypes.byref(d), da[ia[j]].data_ptr(), db[ib[j]].data_ptr(), alone[j].data_ptr(), st))
        d.workspace, d.workspace_bytes = None, 0
        torch.cuda.synchronize()
        assert torch.equal(c.view(torch.uint8), alone.view(torch.uint8))
        assert torch.equal(c[:, m * n:].cpu(), c0[:, m * n:])
        j = items - 1
        left, right = a[ia[j], :m * k].view(k, m).t() if ta else a[ia[j], :m * k].view(m, k), b[ib[j], :k * n].view(n, k).t() if tb else b[ib[j], :k * n].view(k, n)
        if name in INTS:
            want = left.numpy().astype(np.int64).view(np.uint64) @ right.numpy().astype(np.int64).view(np.uint64) + c0[j, :m * n].view(m, n).numpy().astype(np.int64).view(np.uint64)
            assert np.array_equal(c[j, :m * n].cpu().view(m, n).numpy(), want.astype(INTS[name][0]))
        else:
            check(c[j, :m * n].cpu().view(m, n), left, right, c0[j, :m * n].view(m, n), name, k)
    if name in ("f16", "bf16", "f32"):
        d.flags, d.batches, d.m, d.k, d.n = _lib.GEMM_PTRS_ITEM_ORDER, 2, 64, 8192, 64
        assert lib.ntg_gemm_workspace_bytes(ctypes.byref(d)) > 0
        assert lib.ntg_gemm_ptrs_dev(ctypes.byref(d), tab.data_ptr(), tab.data_ptr() + 16, tab.data_ptr() + 32, st) == 1


def test_float64_items_that_are_split_alone_are_split_in_a_batch_too_large_for_it_to_matter():
    """128 items of an odd n are enough multiply-adds for padded copies, one is not and goes out in k ranges: the same bits."""
    lib = _lib.load()
    m, k, n, batch = 64, 4096, 257, 128
    gen = torch.Generator(device=DEV).manual_seed(3)
    a, b = (torch.randn(batch, *s, generator=gen, device=DEV, dtype=torch.float64) for s in ((m, k), (k, n)))
    together, alone = (torch.zeros(batch, m, n, device=DEV, dtype=torch.float64) for _ in range(2))
    strides = (m * k, k * n, m * n)
    product(lib, a, b, together, m, k, n, batch, strides, False, False, _lib.C_OVERWRITE)
    for i in (0, batch - 1):
        assert product(lib, a, b, alone, m, k, n, 1, strides, False, False, _lib.C_OVERWRITE, first=i) > 0
        assert torch.equal(together[i], alone[i])

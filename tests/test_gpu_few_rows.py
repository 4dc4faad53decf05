"""Products of up to 32 rows at the edges of their strips of columns, steps of k and lanes' vectors, on rows that start at any element.

Against the product in 64 bits: one rounding to the type (half a last place: 2^-11 Float16, 2^-8 BFloat16, 2^-24 Float32, relative) on a sum whose k
multiply-adds and eight partial sums each err by 2^-24 of sum |a||b| at most.  Whole numbers small enough for every sum to be exact check positions.
"""
import pytest
import torch

from neurotensor_amd import functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
UNIT = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}
# one element around a strip and a vector of columns, around 8 and 16 rows, around a step of k (16, 32) and whole rounds of steps over eight wavefronts
SIZES = [(1, 128, 1), (2, 129, 2), (3, 159, 3), (15, 160, 5), (16, 161, 7), (17, 255, 8), (31, 256, 9), (32, 257, 63), (5, 1024, 65), (9, 1031, 129),
         (16, 2049, 1030), (17, 1543, 4100), (1, 4097, 9001), (30, 640, 331)]


def matrix(rows, cols, dtype, gen, whole, offset):
    """rows x cols, contiguous, `offset` elements behind a 16-byte boundary"""
    buf = torch.empty(rows * cols + offset, dtype=dtype)
    v = buf[offset:].view(rows, cols)
    v.copy_(torch.randint(-3, 4, (rows, cols), generator=gen) if whole else torch.randn(rows, cols, generator=gen))
    return v, buf.to(DEV)[offset:].view(rows, cols)


@pytest.mark.parametrize("dtype", list(UNIT), ids=str)
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
def test_few_rows(dtype, ta, tb):
    gen = torch.Generator().manual_seed(3)
    for i, (m, k, n) in enumerate(SIZES):
        whole = i % 2 == 0
        a, da = matrix(*((k, m) if ta else (m, k)), dtype, gen, whole, i % 3)
        b, db = matrix(*((n, k) if tb else (k, n)), dtype, gen, whole, (i + 1) % 3)
        x, w = (a.t() if ta else a).double(), (b.t() if tb else b).double()
        c0, dc = matrix(m, n, dtype, gen, whole, 1)
        guard = torch.full((2, n), 77.0, dtype=dtype, device=DEV)
        room = torch.cat([guard[:1], dc, guard[1:]])
        acc = room[1:-1]
        bias = torch.randint(-3, 4, (n,), generator=gen).to(dtype)
        terms = x.abs() @ w.abs()
        got = {"c": (F.matmult(da, db, None, ta, tb), x @ w, terms), "add": (F.matmult(da, db, acc, ta, tb), x @ w + c0.double(), terms + c0.double().abs())}
        sums = x @ w + bias.double()
        got["bias"] = (F.linear(da, db, bias.to(DEV), ta, tb), sums, terms + bias.double().abs())
        got["relu"] = (F.linear_relu(da, db, bias.to(DEV), ta, tb), sums.clamp(min=0), terms + bias.double().abs())
        for what, (out, exact, size) in got.items():
            bound = UNIT[dtype] * exact.abs() + (k + 10) * 2.0 ** -24 * size + (2.0 ** -24 if dtype == torch.float16 else 0)
            if whole and dtype == torch.float32:
                bound = torch.zeros_like(bound)
            assert ((out.cpu().double() - exact).abs() <= bound).all(), (what, m, k, n)
        assert (room[0] == 77).all() and (room[-1] == 77).all()
        assert torch.equal(torch.relu(got["bias"][0]), got["relu"][0])


@pytest.mark.parametrize("dtype", list(UNIT), ids=str)
def test_infinities_of_the_last_column_and_k_stay_there(dtype):
    for tb in (False, True):
        a, b = torch.ones(5, 167, dtype=dtype), torch.ones(167, 71, dtype=dtype)
        b[166, 70] = float("inf")
        got = F.matmult(a.to(DEV), (b.t().contiguous() if tb else b).to(DEV), None, False, tb).cpu()
        assert torch.isinf(got[:, 70]).all() and (got[:, :70] == 167).all()

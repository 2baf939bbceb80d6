"""The order check that ``make_ranges`` runs on the device: a descent anywhere (first and last pair,
edges of stripes, either array, any row) sends the call to the host scan, row boundaries and equal
values do not; results equal the host builder's in every case."""
import pytest
import torch

from kernel_matmul_amd import _native
from kernel_matmul_amd.ranges import make_ranges

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")


def _flagged(x1, x2=None):
    flags = _native.sorted_flags(x1.to(DEVICE), None if x2 is None else x2.to(DEVICE))
    return any(flags.tolist())


@pytest.mark.parametrize("batch,n", [(1, 1), (1, 2), (3, 1), (3, 2), (2, 1025), (1, 131073), (2, 200_000)])
def test_flags(batch, n):
    x = torch.arange(n, dtype=torch.float32).div(3).floor().expand(batch, n).contiguous()  # equal neighbours
    assert not _flagged(x) and not _flagged(x, x) and not _flagged(x[:, :0], x)
    places = sorted({0, 1023, 1024, n // 2, 131071, n - 2} & set(range(n - 1)))
    for row in range(batch):
        for i in places:
            for value in (float("nan"), 1e9):
                y = x.clone()
                y[row, i] = value
                assert _flagged(y) and _flagged(x, y) and _flagged(y, x), (row, i, value)


@pytest.mark.parametrize("n1,n2", [(700, 5000), (5000, 129), (1, 300)])
@pytest.mark.parametrize("which", ["none", "first", "second"])
def test_patterns_agree_with_the_host(n1, n2, which):
    g = torch.Generator().manual_seed(n1 + n2)
    x1, x2 = (torch.sort(torch.rand(2, n, generator=g) * 50.0)[0] for n in (n1, n2))
    if which != "none":
        target = x1 if which == "first" else x2
        target[1] = target[1].flip(-1)
    for a, b in ((x1, x2), (x2, None)):
        got = make_ranges(3.0, a.to(DEVICE), None if b is None else b.to(DEVICE))
        for t, expected in zip(got, make_ranges(3.0, a, b)):
            assert t.is_cuda and torch.equal(t.cpu(), expected)

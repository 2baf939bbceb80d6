"""The order in which an XCD's workgroups take batch items: rotated from group to group, so that every batch item
of every row block is still computed once.  Each item's result is that of a call with this item alone; the
gradient is checked against the oracle.

Tolerance: 2^-19 of the sum of a range's |rhs|, whose entries are at most 1.2.  How many wavefronts share a range
depends on the number of items, and with it the order of the sums; each side is 2^-20 of that sum off at most (two
factors of 2^-22 and the exponentials' rounding, as in test_grid_form_gpu)."""
import pytest
import torch

from kernel_matmul_amd.compile import load_native
from kernel_matmul_amd.configurations import MatmulSingleConfiguration
from kernel_matmul_amd.ranges import make_ranges
from tests.test_grid_grad_gpu import _check as check_gradient

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")
BATCHES = [1, 2, 3, 4, 5, 6, 8, 10, 16, 24]


def _inputs(kt, batch, n, k):
    g = torch.Generator().manual_seed(batch)
    x = torch.sort(torch.rand(n, generator=g) * (n / 8.0))[0]
    ls = torch.linspace(2.0, 0.4, batch)
    rest = {"rbf": [1.2], "spectral": [0.3, 1.2], "locally_periodic": [0.8, 1.1, 0.9]}[kt]
    params = torch.stack([ls, *(torch.full((batch,), v) for v in rest)], dim=-1)
    start, end = make_ranges(10.0, x.to(DEVICE))
    return x, torch.randn(batch, n, k, generator=g), params, start.cpu(), end.cpu()


def _close(result, expected, rhs, start, end):
    sums = torch.cat([torch.zeros_like(rhs[:1]).double(), rhs.abs().double().cumsum(0)])
    bound = 2.0 ** -19 * 1.2 * float((sums[end.long()] - sums[start.long()]).max())
    assert float((result - expected).abs().max()) <= bound


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("kt,k,variant,rows,tail", [
    ("spectral", 5, "grid", 128, 0), ("spectral", 20, "grid", 128, None), ("rbf", 3, "grid", 128, 0),
    ("spectral", 5, "grid", 128, None), ("rbf", 3, "grid", 128, None), ("rbf", 3, "grid", 128, 4),
    ("locally_periodic", 5, "block", None, None), ("locally_periodic", 5, "mfma_f16_direct", 128, None),
    ("locally_periodic", 20, "mfma_f16_direct", 32, None),
])
def test_forward(kt, k, variant, rows, tail, batch):
    """tail (grid): how many row blocks of each XCD get a workgroup each; without the option all of a launch as
    small as this."""
    n = 2000  # sixteen row blocks: some XCDs get groups of their own, others share one
    x, rhs, params, start, end = (t.to(DEVICE) for t in _inputs(kt, batch, n, k))

    def call(*args):
        defines = dict(MatmulSingleConfiguration(kt).make_config(args))
        defines["MATMUL_VARIANT"] = variant
        if rows:
            defines["MATMUL_ROWS_PER_WAVE"] = rows
        if tail is not None:
            defines["MATMUL_GROUP_TAIL"] = tail
        return load_native("matmul", defines).call(*args)

    shared = [t.expand(batch, *t.shape) for t in (x, start, end)]
    result = call(shared[0], shared[0], rhs, params, shared[1], shared[2])
    for b in range(batch):
        _close(result[b], call(x, x, rhs[b], params[b], start, end), rhs[b], start, end)


@pytest.mark.parametrize("batch", [8, 10])
def test_large_launch(batch):
    """With row blocks of their own workgroup behind the groups."""
    n = 50_000
    x, rhs, params, start, end = (t.to(DEVICE) for t in _inputs("spectral", batch, n, 1))
    shared = [t.expand(batch, *t.shape) for t in (x, start, end)]
    args = (shared[0], shared[0], rhs, params, shared[1], shared[2])
    result = load_native("matmul", MatmulSingleConfiguration("spectral").make_config(args)).call(*args)
    for b in range(batch):
        one = (x, x, rhs[b], params[b], start, end)
        defines = dict(MatmulSingleConfiguration("spectral").make_config(one))
        defines["MATMUL_VARIANT"], defines["MATMUL_ROWS_PER_WAVE"] = "grid", 128
        _close(result[b], load_native("matmul", defines).call(*one), rhs[b], start, end)


@pytest.mark.parametrize("batch", [2, 3, 6, 16])
@pytest.mark.parametrize("kt,c", [("spectral", 4), ("rbf", 6)])
def test_gradient(kt, c, batch):
    n = 600
    x, left, params, start, end = _inputs(kt, batch, n, c)
    right = torch.randn(batch, n, c, generator=torch.Generator().manual_seed(1))
    shared = [t.expand(batch, *t.shape) for t in (x, start, end)]
    check_gradient(kt, shared[0], shared[0], left, right, params, shared[1], shared[2])


@pytest.mark.parametrize("k", [33, 64, 100])
@pytest.mark.parametrize("rows,tail", [(32, None), (64, None), (128, 0), (128, 4), (128, 37), (None, None)])
def test_halves_of_wide_rhs(k, rows, tail):
    """More than 32 spectral columns: an XCD's workgroups take one half of 64 columns and the other in turn, some 32 at a
    time.  The result is that of calls with 32 columns each."""
    n, batch = 20_000, 9
    x, rhs, params, start, end = (t.to(DEVICE) for t in _inputs("spectral", batch, n, k))
    shared = [t.expand(batch, *t.shape) for t in (x, start, end)]

    def call(part):
        args = (shared[0], shared[0], part, params, shared[1], shared[2])
        defines = dict(MatmulSingleConfiguration("spectral").make_config(args))
        if rows:
            defines["MATMUL_VARIANT"], defines["MATMUL_ROWS_PER_WAVE"] = "grid", rows
        if tail is not None:
            defines["MATMUL_GROUP_TAIL"] = tail
        return load_native("matmul", defines).call(*args)

    result = call(rhs)
    for first in range(0, k, 32):
        part = rhs[..., first:first + 32].contiguous()
        expected = call(part)
        for b in range(batch):
            _close(result[b, :, first:first + 32], expected[b], part[b], start, end)

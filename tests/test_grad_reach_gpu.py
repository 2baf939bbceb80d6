"""Hyper-parameter gradient pair by pair: the tiles that are left out because every entry of them is zero in fp32.

A batch that does not collapse to one dimension is evaluated without leaving anything out, in the same order
otherwise, so the sums are the same to the last bit: adding a zero changes none."""
import pytest
import torch

from kernel_matmul_amd.compile import load_native
from kernel_matmul_amd.configurations import BilinearDerivativeConfiguration

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")
N = 1500
# (twelve row blocks each: enough that rbf and spectral vectors of this width go pair by pair, and that a wavefront's
# share of a row block's columns is wide enough for the look at what is out of reach)
BATCH = (8, 16)
ITEMS = BATCH[0] * BATCH[1]


def _inputs(kt, c, lengthscale, density=1.0, periodic=0.8, seed=0):
    g = torch.Generator().manual_seed(seed)
    x1 = torch.sort(torch.rand(N, generator=g) * (N / density))[0]
    x2 = torch.sort(torch.rand(N, generator=g) * (N / density))[0]
    left = torch.randn(*BATCH, N, c, generator=g)
    right = torch.randn(*BATCH, N, c, generator=g)
    ls = lengthscale * torch.linspace(1.0, 2.0, ITEMS).reshape(BATCH)
    rest = {"rbf": [1.2], "spectral": [0.3, 1.2], "locally_periodic": [periodic, 1.1, 0.9]}[kt]
    params = torch.stack([ls, *(torch.full(BATCH, v) for v in rest)], dim=-1)
    mid = torch.arange(12) * 128 + 64
    start, end = (mid - 333).clamp(0, N).int(), (mid + 401).clamp(0, N).int()
    return [x1, x2, left, right, params, start, end]


def _call(kt, args):
    op = load_native("bilinear_derivative", BilinearDerivativeConfiguration(kt).make_config(args))
    return op.call(*args).cpu().reshape(ITEMS, -1)


def _check(kt, args):
    x1, x2, left, right, params, start, end = (t.to(DEVICE) for t in args)
    shared = [t.expand(*BATCH, *t.shape) for t in (x1, x2, start, end)]
    flat = [t.expand(ITEMS, *t.shape) for t in (x1, x2, start, end)]
    result = _call(kt, (flat[0], flat[1], left.flatten(0, 1), right.flatten(0, 1), params.flatten(0, 1), flat[2], flat[3]))
    # (a batch dimension stored the other way round)
    turned = params.transpose(0, 1).contiguous().transpose(0, 1)
    expected = _call(kt, (shared[0], shared[1], left, right, turned, shared[2], shared[3]))
    assert torch.equal(result.isnan(), expected.isnan())
    assert torch.equal(result.nan_to_num(), expected.nan_to_num())
    return result


CASES = [("rbf", 11), ("rbf", 16), ("spectral", 6), ("spectral", 8), ("spectral", 13), ("locally_periodic", 1), ("locally_periodic", 8),
         ("locally_periodic", 16)]


@pytest.mark.parametrize("kt,c", CASES)
@pytest.mark.parametrize("lengthscale", [0.02, 0.4, 1.1, 5.0, 60.0])
def test_lengthscales(kt, c, lengthscale):
    result = _check(kt, _inputs(kt, c, lengthscale))
    assert bool(result.isfinite().all())


@pytest.mark.parametrize("periodic", [-0.05, -1.0, 0.01, 0.0, float("nan")])
def test_second_lengthscales(periodic):
    """A negative one raises the entries by up to 2^(2 log2 e / |it|), a factor of 2^58 here."""
    _check("locally_periodic", _inputs("locally_periodic", 3, 0.7, periodic=periodic))


@pytest.mark.parametrize("kt,c", [("rbf", 12), ("spectral", 7), ("locally_periodic", 5)])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("what", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("at", [0, 700, 1499])
def test_values_that_are_not_finite(kt, c, value, what, at):
    args = _inputs(kt, c, 0.4)
    if what < 2:
        args[what][at] = value
    elif what < 4:
        args[what][1, 2, at, c - 1] = value
    else:
        args[4][1, 2, at % args[4].shape[-1]] = value
    _check(kt, args)


@pytest.mark.parametrize("kt,c", [("spectral", 8), ("locally_periodic", 4)])
def test_unsorted_coordinates(kt, c):
    args = _inputs(kt, c, 0.6)
    g = torch.Generator().manual_seed(3)
    args[0] = args[0][torch.randperm(N, generator=g)]
    args[1] = args[1][torch.randperm(N, generator=g)]
    _check(kt, args)


@pytest.mark.parametrize("ranges", [(0, 0), (0, 1), (1499, 1500), (700, 716), (0, 1500)])
def test_ranges(ranges):
    args = _inputs("spectral", 8, 0.5)
    args[5][:], args[6][:] = ranges
    _check("spectral", args)


@pytest.mark.parametrize("kt,c", [("locally_periodic", 8), ("rbf", 12), ("spectral", 7)])
@pytest.mark.parametrize("m", [2**30 + 300, 2**31 - 1 - 128])
def test_rows_at_the_largest_sizes(kt, c, m):
    """The gradient of the last rows of as many as the entry point takes (all others' ranges are empty) is that of
    these rows alone."""
    n, tail = 1000, m - (m - 1) // 128 * 128 + 256  # three row blocks
    blocks = (m + 127) // 128
    g = torch.Generator().manual_seed(5)
    x1 = torch.full((m,), -1e3, device=DEVICE)
    x1[m - tail:] = torch.sort(torch.rand(tail, generator=g) * 500.0)[0].to(DEVICE)
    x2 = torch.sort(torch.rand(n, generator=g) * 500.0)[0].to(DEVICE)
    left = torch.randn(1, c, generator=g).to(DEVICE).expand(m, c)
    right = torch.randn(n, c, generator=g).to(DEVICE)
    params = torch.tensor({"rbf": [0.8, 1.2], "spectral": [0.8, 0.3, 1.2], "locally_periodic": [0.8, 0.9, 1.1, 0.9]}[kt], device=DEVICE)
    start = torch.zeros(blocks, dtype=torch.int32, device=DEVICE)
    end = torch.zeros(blocks, dtype=torch.int32, device=DEVICE)
    end[-3:] = n
    op = load_native("bilinear_derivative", BilinearDerivativeConfiguration(kt).make_config((x1, x2, left, right, params, start, end)))
    result = op.call(x1, x2, left, right, params, start, end)
    expected = op.call(x1[m - tail:], x2, left[m - tail:], right, params, start[-3:], end[-3:])
    # (shorter shares of columns for fewer rows: other orders of fp32 sums, of which few terms are in reach)
    torch.testing.assert_close(result, expected, rtol=1e-4, atol=1e-4 * float(expected.abs().max()))


@pytest.mark.parametrize("what,value", [(1, 0.0), (1, float("nan")), (2, 0.0), (2, float("nan"))])
@pytest.mark.parametrize("c", [8, 16])
def test_parameters_that_make_entries_nan(c, what, value):
    """Where no column is in reach of a row as well (a second lengthscale of zero: entries a whole number of
    periods apart, here every fourth)."""
    args = _inputs("locally_periodic", c, 0.4)
    args[0] = torch.arange(N) * 0.25 + 3000.0
    args[1] = torch.arange(N) * 0.25
    args[4][1, 2, 2] = 1.0
    args[4][1, 2, what] = value
    result = _check("locally_periodic", args)
    item = BATCH[1] + 2
    assert bool(result[item].isnan().all())
    assert bool(result[:item].isfinite().all())

"""Locally periodic kernels: the tiles that are left out because every entry of them rounds to zero.

The results are those of the kernel that evaluates all tiles (fewer than 128 rows per wavefront): what is left
out adds exact zeros, and whatever is not finite is never left out.

Tolerance: 2^-21 of the sum of |rhs| over a range, whose entries are at most one: each side rounds its products to
2^-22 of their size (two fp16 halves a factor) and its sums to 2^-24 at each of some 25 additions that partial sums
of random signs grow through; the orders of the additions differ, and the workgroup-shared kernel forms the
coordinates' difference another way."""
import pytest
import torch

from kernel_matmul_amd.compile import load_native
from kernel_matmul_amd.configurations import MatmulSingleConfiguration

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")
N = 1500


def _inputs(k, lengthscale, periodic=0.8, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.sort(torch.rand(N, generator=g) * 150)[0]
    rhs = torch.randn(N, k, generator=g)
    params = torch.tensor([lengthscale, periodic, 1.1, 0.9])
    mid = torch.arange(12) * 128 + 64
    start, end = (mid - 400).clamp(0, N).int(), (mid + 401).clamp(0, N).int()
    return [x.clone(), x.clone(), rhs, params, start, end]


def _call(args, variant, rows):
    args = tuple(t.to(DEVICE) for t in args)
    defines = MatmulSingleConfiguration("locally_periodic").make_config(args)
    defines["MATMUL_VARIANT"] = variant
    if rows:
        defines["MATMUL_ROWS_PER_WAVE"] = rows
    return load_native("matmul", defines).call(*args).cpu()


def _check(args, k):
    expected = _call(args, "mfma_f16_direct", 64)
    sums = args[2].nan_to_num(0.0, 0.0, 0.0).abs().cumsum(0)
    atol = 2.0 ** -21 * float((sums[801:] - sums[:-801]).max()) * (8.0 if float(args[3][1]) < 0 else 1.0)
    torch.testing.assert_close(_call(args, "mfma_f16_direct", 128), expected, rtol=1e-5, atol=atol, equal_nan=True)
    block = _call(args, "block", None)
    # (a step that straddles a range's end hands a NaN to that range's rows too in the workgroup-shared kernel)
    assert bool((block.isnan() | ~expected.isnan()).all())
    both = ~block.isnan() & ~expected.isnan()
    torch.testing.assert_close(block[both], expected[both], rtol=1e-5, atol=atol)


@pytest.mark.parametrize("k", [1, 16, 20])
@pytest.mark.parametrize("lengthscale", [0.05, 0.4, 0.9, 1.4, 2.5, 30.0])
@pytest.mark.parametrize("periodic", [0.8, -1.0])  # (-1: entries of up to e^2)
def test_lengthscales(k, lengthscale, periodic):
    args = _inputs(k, lengthscale, periodic)
    _check(args, k)


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("what", ["rhs", "x1", "x2"])
@pytest.mark.parametrize("at", [0, 150, 700, 1499])
def test_values_that_are_not_finite(value, what, at):
    args = _inputs(3, 0.5)
    if what == "rhs":
        args[2][at, 1] = value
    else:
        args[0 if what == "x1" else 1][at] = value
    _check(args, 3)


def test_unsorted_coordinates():
    args = _inputs(5, 0.6)
    g = torch.Generator().manual_seed(3)
    args[0] = args[0][torch.randperm(N, generator=g)]
    args[1] = args[1][torch.randperm(N, generator=g)]
    _check(args, 5)


@pytest.mark.parametrize("what,value", [(0, float("nan")), (1, 0.0), (1, float("nan")), (2, 0.0), (2, float("nan"))])
@pytest.mark.parametrize("k", [1, 20])
@pytest.mark.parametrize("away", [0.0, 1000.0])
def test_parameters_that_make_entries_nan(what, value, k, away):
    """Where no column is in reach of a row as well (a second lengthscale of zero: entries a whole number of
    periods apart, here every fourth)."""
    args = _inputs(k, 0.5)
    args[3][2] = 1.0
    args[0] = torch.arange(N) * 0.25 + away
    args[1] = torch.arange(N) * 0.25
    args[3][what] = value
    _check(args, k)
    assert bool(_call(args, "mfma_f16_direct", 128).isnan().all())

"""The grid form of the hyper-parameter gradient at the places where it can go wrong: windows of
every size up to the largest and beyond (pairwise), vector widths on both sides of its groups and
passes, ranges and row blocks that are cut off, ranges on both sides of the least width and of a
column share, gaps, unsorted and equal points, strides, scales and values that are not finite.

Tolerance against float64, per parameter: 4e-6 sum |left| |right| times the size of the derivative's
terms.  An entry is a sum over grid points of products of two factors, each 1e-6 exact (exponent,
hardware exponential, split into two fp16 values, as in the forward), and the trapezoid rule at this
spacing adds 4e-8.  The terms' size: the envelope E for the output scale, (u^2 + 2) E for the
lengthscale (V V |p^2 - 1 / (4 ln 2)| averages to less) and (|d| + 2 l) E for the frequency.  What is
dropped below 2^-37 is covered by a floor of 2^-34 on E within the range."""
import numpy as np
import pytest
import torch

from kernel_matmul_amd.compile import load_native
from kernel_matmul_amd.configurations import BilinearDerivativeConfiguration
from kernel_matmul_amd.ranges import make_ranges
from oracle import kernels as oracle

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")


def _params(kt, lengthscale):
    ls = torch.as_tensor(lengthscale, dtype=torch.float32)
    f, s = torch.full_like(ls, 0.31), torch.full_like(ls, 1.3)
    return torch.stack([ls, f, s] if kt == "spectral" else [ls, s], dim=-1)


def _call(kt, *args):
    op = load_native("bilinear_derivative", BilinearDerivativeConfiguration(kt).make_config(args))
    result = op.call(*args)
    assert torch.equal(result, op.call(*args))  # sums in a fixed order
    return result.cpu().double().numpy()


def _check(kt, x1, x2, left, right, params, start, end, transform=lambda t: t.to(DEVICE)):
    result = _call(kt, *(transform(t) for t in (x1, x2, left, right, params, start, end)))
    a = [t.numpy() for t in (x1, x2, left, right, params, start, end)]
    expected = oracle.param_grad(kt, *a)
    mask = oracle.range_mask(a[5], a[6], a[0].shape[-1], a[1].shape[-1])
    d = a[0].astype(np.float64)[..., :, None] - a[1].astype(np.float64)[..., None, :]
    p = a[4].astype(np.float64)
    ls, sigma = (np.abs(p[..., i, None, None]) for i in (0, -1))
    env = (np.exp(-0.5 * (d / ls) ** 2) + 2.0 ** -34) * mask
    size = np.abs(a[2].astype(np.float64)) @ np.abs(np.swapaxes(a[3].astype(np.float64), -1, -2)) * env
    u2 = 0.5 * (d / ls) ** 2 / np.log(2.0)
    terms = [size * (u2 + 2.0) * sigma * 2.0 * np.log(2.0) / ls]
    if kt == "spectral":
        terms.append(size * (np.abs(d) + 2.0 * ls) * 2.0 * np.pi * sigma)
    terms.append(size)
    tol = 4e-6 * np.stack([t.sum((-2, -1)) for t in terms], axis=-1)
    tol = tol + 1e-6 * np.abs(expected) + 1e-30
    err = np.abs(result - expected)
    assert np.all(err <= tol), (float((err / tol).max()), result, expected)


def _points(n, extent, seed):
    return torch.sort(torch.rand(n, generator=torch.Generator().manual_seed(seed)) * extent)[0]


def _vectors(rows, c, seed, batch=()):
    return torch.randn(*batch, rows, c, generator=torch.Generator().manual_seed(seed))


def _ranges(m, n, width):
    rows = (m + 127) // 128
    g = torch.Generator().manual_seed(m + n + width)
    mid = (torch.arange(rows) * 128 + 64) * n // max(m, 1)
    lo = mid - width // 2 - torch.randint(0, 40, (rows,), generator=g)
    hi = mid + width // 2 + torch.randint(0, 40, (rows,), generator=g)
    return lo.clamp(0, n).int(), hi.clamp(0, n).int()


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
@pytest.mark.parametrize("c", [1, 4, 5, 8, 9, 16, 17, 33])
def test_vector_widths(kt, c):
    n = 1000
    x = _points(n, n / 10.0, 1).expand(2, n)
    start, end = (t.expand(2, -1) for t in _ranges(n, n, 500))
    right = _vectors(n, c, 2, (2,))
    _check(kt, x, x, 0.5 * right + 0.1 * _vectors(n, c, 3, (2,)), right, _params(kt, [1.0, -0.6]), start, end)


@pytest.mark.parametrize("kt,c", [("spectral", 3), ("spectral", 11), ("rbf", 6)])
@pytest.mark.parametrize("lengthscale", [0.1, 0.25, 0.3, 0.36, 0.4, 0.45, 0.6, 0.9, 2.0, 30.0, 1e4])
def test_window_sizes(kt, c, lengthscale):
    n = 1300
    x = _points(n, n / 10.0, 4)
    start, end = _ranges(n, n, 600)
    _check(kt, x, x, _vectors(n, c, 5), _vectors(n, c, 6), _params(kt, lengthscale), start, end)


@pytest.mark.parametrize("m,n", [(1, 400), (129, 97), (128, 96), (128, 95), (255, 511), (300, 1), (640, 257), (130, 2100)])
@pytest.mark.parametrize("c", [8, 12])
def test_cut_off_blocks_and_ranges(m, n, c):
    x1, x2 = _points(m, 20.0, 7), _points(n, 20.0, 8)
    blocks = (m + 127) // 128
    start = torch.zeros(blocks, dtype=torch.int32)
    end = torch.full((blocks,), n, dtype=torch.int32)
    end[-1] = min(n, 137) if blocks > 1 else n
    if blocks > 2:
        start[0] = end[0]
    _check("spectral", x1, x2, _vectors(m, c, 9), _vectors(n, c, 10), _params("spectral", 1.5), start, end)


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
@pytest.mark.parametrize("c", [6, 8, 11, 16, 17, 33])
@pytest.mark.parametrize("width", [1950, 2040, 2300])
def test_wide_vectors_and_long_ranges(kt, c, width):
    """Ranges on both sides of the width from which wide vectors take the form."""
    n = 3000
    x = _points(n, 50.0, 21)
    start, end = _ranges(n, n, width)
    _check(kt, x, x, _vectors(n, c, 22), _vectors(n, c, 23), _params(kt, 1.3), start, end)


@pytest.mark.parametrize("kind", ["gaps", "negative", "far", "unsorted", "equal"])
@pytest.mark.parametrize("kt,c", [("spectral", 4), ("spectral", 10), ("rbf", 2)])
def test_points(kt, c, kind):
    n = 900
    x = _points(n, 60.0, 11)
    if kind == "gaps":
        x = x + 9.0 * (torch.arange(n) // 100) + 2.5 * (torch.arange(n) % 100 > 53)
    elif kind == "negative":
        x = x - 30.0
    elif kind == "far":
        x = x + 3000.0
    elif kind == "equal":
        x = torch.sort((x / 4.0).round() * 4.0)[0]
    x2 = x[torch.randperm(n, generator=torch.Generator().manual_seed(12))] if kind == "unsorted" else x
    start, end = _ranges(n, n, 2 * n if kind == "unsorted" else 400)
    _check(kt, x, x2, _vectors(n, c, 13), _vectors(n, c, 14), _params(kt, 1.1), start, end)


@pytest.mark.parametrize("scale", [1e-30, 1e-12, 1e12])
def test_scales_and_strides(scale):
    """Vectors far from one and of very different columns, read with strides of three."""
    n, c = 700, 7
    x = _points(n, 60.0, 15)
    start, end = _ranges(n, n, 400)
    left, right = _vectors(n, c, 16), _vectors(n, c, 17) * scale
    right[:, 1:3] *= 1e-3

    def transform(t):
        t = t.to(DEVICE)
        wide = torch.zeros(*t.shape, 3, device=DEVICE, dtype=t.dtype)
        wide[..., 0] = t
        return wide[..., 0]

    _check("spectral", x, x, left, right, _params("spectral", 1.0), start, end, transform)


@pytest.mark.parametrize("which", ["left", "right"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_values_that_are_not_finite(which, value):
    n, c = 512, 4
    x = _points(n, 50.0, 18)
    start, end = _ranges(n, n, 400)
    vectors = {"left": _vectors(n, c, 19), "right": _vectors(n, c, 20)}
    vectors[which][200, 1] = value
    args = [t.to(DEVICE) for t in (x, x, vectors["left"], vectors["right"], _params("spectral", 1.0), start, end)]
    op = load_native("bilinear_derivative", BilinearDerivativeConfiguration("spectral").make_config(args))
    assert not torch.isfinite(op.call(*args)).any()


@pytest.mark.parametrize("gap", [1e2, 1e3, 1e4, 1e5, 1e6, 1e9])
@pytest.mark.parametrize("kt,c,count", [("spectral", 4, 1003), ("rbf", 6, 1003), ("spectral", 11, 2603)])
def test_columns_next_to_a_wide_gap(kt, c, count, gap):
    """Groups of 8 columns that lie on both sides of a gap of up to a billion lengthscales: a gradient that
    only the columns next to the gap and the rows near it make."""
    extent = count / 100.0
    x = torch.cat([_points(count, extent, 30), _points(500, 5.0, 31) + extent + gap])
    start, end = make_ranges(extent if c == 11 else 6.0, x)
    left, right = _vectors(len(x), c, 32), torch.zeros(len(x), c)
    right[count - 3:count] = _vectors(3, c, 33)
    _check(kt, x, x, left, right, _params(kt, 1.0), start, end)
    mirrored = -x.flip(0)
    _check(kt, mirrored, mirrored, left.flip(0), right.flip(0), _params(kt, 1.0),
           *make_ranges(extent if c == 11 else 6.0, mirrored))


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
@pytest.mark.parametrize("c", [1, 4, 8, 11, 20])
@pytest.mark.parametrize("i,j", [(207, 224), (64, 47)])
@pytest.mark.parametrize("spacing", [0.5, 0.6, 0.7])
def test_distant_entries_of_sparse_points(kt, c, i, j, spacing):
    """Row blocks evaluated pair by pair: an entry that fp32 can represent is not dropped, whatever its
    distance (here 2^-52, 2^-75 and 2^-102 of sigma, the only one of a coefficient that is not zero).
    The exponent is exact to three roundings of half an ulp: 0.7 * 102 * 3 * 2^-24."""
    n = 512
    x = torch.arange(n) * spacing
    start, end = torch.zeros(4, dtype=torch.int32), torch.full((4,), n, dtype=torch.int32)
    left, right = torch.zeros(n, c), torch.zeros(n, c)
    left[i], right[j] = 1e6, 1e9
    params = _params(kt, 1.0)
    result = _call(kt, *(t.to(DEVICE) for t in (x, x, left, right, params, start, end)))
    expected = oracle.param_grad(kt, *(t.numpy() for t in (x, x, left, right, params, start, end)))
    assert np.all(np.abs(result - expected) <= 2e-5 * np.abs(expected)), (result, expected)


@pytest.mark.parametrize("which", ["x2", "left", "right"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("kt,c,step,n", [("spectral", 4, 0.1, 640), ("spectral", 4, 0.7, 640), ("rbf", 6, 0.1, 640),
                                         ("rbf", 6, 0.7, 640), ("spectral", 11, 0.01, 2304), ("spectral", 11, 0.7, 640),
                                         ("rbf", 20, 0.01, 2304), ("rbf", 20, 0.7, 640)])
def test_values_out_of_reach_that_are_not_finite(kt, c, step, n, value, which):
    """Also a value that only meets entries which vanish: the gradient is not finite then (zero times a
    NaN or an infinity; an infinite coordinate of an rbf kernel makes the lengthscale's component so)."""
    near = torch.arange(n) * step
    x1 = torch.cat([near, near[-1] + 1000.0 + 0.01 * torch.arange(128)])
    x2 = torch.cat([-1000.0 + 0.01 * torch.arange(75), near])
    blocks = len(x1) // 128
    start, end = torch.zeros(blocks, dtype=torch.int32), torch.full((blocks,), len(x2), dtype=torch.int32)
    for place in (0, 40, 74) if which != "left" else (n, n + 100, n + 127):
        tensors = {"x1": x1, "x2": x2.clone(), "left": _vectors(len(x1), c, 50), "right": _vectors(len(x2), c, 51)}
        tensors[which][place] = value
        args = [t.to(DEVICE) for t in (*tensors.values(), _params(kt, 0.5), start, end)]
        result = _call_nan(kt, *args)
        if kt == "rbf" and which == "x2" and value == value:
            result = result[:1]
        assert not np.isfinite(result).any(), (place, result)


def _call_nan(kt, *args):
    return load_native("bilinear_derivative", BilinearDerivativeConfiguration(kt).make_config(args)).call(*args).cpu().numpy()


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
@pytest.mark.parametrize("c", [1, 4, 6, 8, 11, 20])
@pytest.mark.parametrize("left_scale,right_scale", [(1e-30, 1e33), (1e30, 1e-28), (1e-6, 1e37), (1e36, 1e-4)])
def test_scales_that_cancel(kt, c, left_scale, right_scale):
    """Vectors whose products are of ordinary size although they are not, as in a solve with a tiny or
    huge diagonal."""
    n = 2600
    x = _points(n, 26.0, 52)
    start, end = _ranges(n, n, 2 * n)
    left, right = _vectors(n, c, 53) * left_scale, _vectors(n, c, 54) * right_scale
    _check(kt, x, x, left, right, _params(kt, 1.3), start, end)


@pytest.mark.parametrize("kt,c", [("spectral", 3), ("spectral", 12), ("rbf", 5), ("rbf", 20)])
@pytest.mark.parametrize("width", [700, 4000])
def test_ranges_at_the_largest_sizes(kt, c, width):
    """The last columns of as many as the entry point takes (one point and one row, repeated), and empty
    ranges of the largest values: nothing past the largest int is formed."""
    n, m = 2**31 - 1 - 128, 300
    x1, one = _points(m, 3.0, 55), torch.ones(1)
    left, right = _vectors(m, c, 57), _vectors(1, c, 58)
    start = torch.tensor([n - width, 2**31 - 1, n], dtype=torch.int32)
    end = torch.tensor([n, 2**31 - 1, -2**31], dtype=torch.int32)
    params = _params(kt, 1.0)
    result = _call(kt, x1.to(DEVICE), one.to(DEVICE).expand(n), left.to(DEVICE), right.to(DEVICE).expand(n, c),
                   *(t.to(DEVICE) for t in (params, start, end)))
    first = np.array([0, 1, 1], np.int32), np.ones(3, np.int32)
    expected = width * oracle.param_grad(kt, *(t.numpy() for t in (x1, one, left, right, params)), *first)
    size = np.abs(left[:128].double().numpy()) @ np.abs(right.double().numpy().T)
    # (distances up to two lengthscales: the derivatives' factors are below 15)
    assert np.all(np.abs(result - expected) <= 4e-6 * 15.0 * width * size.sum()), (result, expected)


@pytest.mark.parametrize("kt,c", [("spectral", 4), ("spectral", 12), ("rbf", 6), ("rbf", 20)])
@pytest.mark.parametrize("small", [1e-27, 2.5e-26, 1e-20])
def test_vectors_that_grow_along_the_columns(kt, c, small):
    """Tiny values in front of ordinary ones (and behind them), whose sums follow the column's scale down."""
    n = 1200
    x = _points(n, n / 10.0, 61)
    right = _vectors(n, c, 62)
    right[:500] *= small
    right[800:] *= small
    left = _vectors(n, c, 63)
    start, end = _ranges(n, n, 700)
    _check(kt, x, x, left, right, _params(kt, 1.0), start, end)

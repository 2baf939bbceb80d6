"""The grid form of the forward operator (a Gaussian as a sum over an equidistant grid) at the places
where it can go wrong: windows of every size up to the largest and beyond, ranges that end anywhere,
row blocks and ranges that are cut off, gaps in the data, points next to the origin and unsorted
ones, every number of wavefronts per item, rhs widths on both sides of its groups.

Tolerance per element, against float64: 3e-6 (|envelope| @ |rhs|) + 2^-36 sigma sum |rhs|.  An entry is a
sum of products of two factors; each is rounded by its exponent (|exponent| < 16: two roundings of
half an fp32 ulp, 6.6e-7 together), the hardware exponential (1.2e-7) and its split into two fp16
values (2^-22), i.e. 1e-6 each; the trapezoid rule adds 6e-8 and phases 3e-8 revolutions each.  The
floor is what both factors drop below 2^-37."""
import numpy as np
import pytest
import torch

from kernel_matmul_amd.compile import load_native
from kernel_matmul_amd.configurations import MatmulSingleConfiguration
from kernel_matmul_amd.ranges import make_ranges
from oracle import kernels as oracle

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")


def _run(kt, x1, x2, rhs, params, start, end, rows=None, tail=None):
    args = tuple(t.to(DEVICE) for t in (x1, x2, rhs, params, start, end))
    defines = MatmulSingleConfiguration(kt).make_config(args)
    defines["MATMUL_VARIANT"] = "grid"
    if rows:
        defines["MATMUL_ROWS_PER_WAVE"] = rows
    if rows == 128 and tail is None:
        tail = 0  # (four row blocks a workgroup; launches as small as these have only the split tail otherwise)
    if tail is not None:
        defines["MATMUL_GROUP_TAIL"] = tail
    op = load_native("matmul", defines)
    out = op.call(*args)
    assert torch.equal(out, op.call(*args))  # sums in a fixed order
    return out.cpu().double().numpy()


def _check(kt, x1, x2, rhs, params, start, end, floor=1e-30, **launch):
    out = _run(kt, x1, x2, rhs, params, start, end, **launch)
    a = [t.numpy() for t in (x1, x2, rhs, params, start, end)]
    expected = oracle.matmul(kt, a[0], a[1], a[2], a[3], a[4], a[5])
    envelope = np.abs(oracle.dense("rbf", a[0], a[1], a[3][..., [0, -1]], a[4], a[5]))
    mask = oracle.range_mask(a[4], a[5], x1.shape[-1], x2.shape[-1]).astype(np.float64)
    size = np.abs(a[2].astype(np.float64))
    tol = 3e-6 * (envelope @ size) + 2.0 ** -36 * np.abs(a[3][..., -1, None, None]) * (mask @ size) + floor
    err = np.abs(out - expected)
    assert np.all(err <= tol), float((err / tol).max())


def _params(kt, lengthscale):
    ls = torch.as_tensor(lengthscale, dtype=torch.float32)
    f, s = torch.full_like(ls, 0.31), torch.full_like(ls, 1.3)
    return torch.stack([ls, f, s] if kt == "spectral" else [ls, s], dim=-1)


def _ranges(m, n, width, seed=0):
    """Ranges around the block's position that start and end anywhere."""
    g = torch.Generator().manual_seed(seed)
    rows = (m + 127) // 128
    mid = (torch.arange(rows) * 128 + 64) * n // max(m, 1)
    lo = mid - width // 2 - torch.randint(0, 40, (rows,), generator=g)
    hi = mid + width // 2 + torch.randint(0, 40, (rows,), generator=g)
    return lo.clamp(0, n).int(), hi.clamp(0, n).int()


def _points(n, extent, seed, batch=()):
    g = torch.Generator().manual_seed(seed)
    return torch.sort(torch.rand(*batch, n, generator=g) * extent, dim=-1)[0]


@pytest.mark.parametrize("rows", [16, 32, 64, 128])
@pytest.mark.parametrize("kt,k", [("spectral", 1), ("spectral", 16), ("spectral", 17), ("spectral", 33), ("spectral", 70),
                                  ("rbf", 3), ("rbf", 17), ("rbf", 64), ("rbf", 65)])
def test_rhs_widths_and_wavefronts(kt, k, rows):
    n = 1000
    x = _points(n, n / 10.0, 1).expand(2, n)
    rhs = torch.randn(2, n, k, generator=torch.Generator().manual_seed(2))
    start, end = (t.expand(2, -1) for t in _ranges(n, n, 500))
    _check(kt, x, x, rhs, _params(kt, [1.0, 0.6]), start, end, rows=rows)


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
@pytest.mark.parametrize("lengthscale", [0.1, 0.25, 0.3, 0.36, 0.45, 0.6, 0.9, 2.0, 30.0, 1e4])
def test_window_sizes(kt, lengthscale):
    """Ten points per unit: a 128-row block spans 12.8 / lengthscale lengthscales, windows of two to
    five tiles of the grid, and row blocks it does not fit (evaluated entry by entry), mixed."""
    n = 1300
    x = _points(n, n / 10.0, 3)
    rhs = torch.randn(n, 5, generator=torch.Generator().manual_seed(4))
    start, end = _ranges(n, n, 600)
    _check(kt, x, x, rhs, _params(kt, lengthscale), start, end)


@pytest.mark.parametrize("m,n", [(1, 400), (129, 161), (128, 159), (255, 160), (300, 1), (640, 257)])
@pytest.mark.parametrize("rows", [32, 128])
def test_cut_off_blocks_and_ranges(m, n, rows):
    """Rectangular matrices, last row blocks of one row, ranges on both sides of the width from
    which the form is taken (160), empty ranges and ranges beyond the matrix."""
    x1, x2 = _points(m, 20.0, 5), _points(n, 20.0, 6)
    blocks = (m + 127) // 128
    start = torch.zeros(blocks, dtype=torch.int32)
    end = torch.full((blocks,), n, dtype=torch.int32)
    end[-1] = min(n, 37) if blocks > 1 else n
    if blocks > 2:
        start[0] = end[0]
    rhs = torch.randn(n, 16, generator=torch.Generator().manual_seed(7))
    _check("spectral", x1, x2, rhs, _params("spectral", 1.5), start, end, rows=rows)


@pytest.mark.parametrize("kind", ["gaps", "origin", "negative", "far", "unsorted", "equal"])
@pytest.mark.parametrize("rows", [32, 128])
def test_coordinates(kind, rows):
    n = 900
    x = _points(n, 30.0, 8)
    if kind == "gaps":      # groups of neighbouring columns on both sides of gaps of every size
        x = x + torch.cumsum((torch.arange(n) % 97 == 5).float() * torch.linspace(0.5, 12.0, n), dim=0)
    elif kind == "origin":
        x = x * 0.3 - 2.0
    elif kind == "negative":
        x = x - 500.0
    elif kind == "far":
        x = x + 30000.0     # ulp 2^-9
    elif kind == "unsorted":
        x = x[torch.randperm(n, generator=torch.Generator().manual_seed(9))]
    else:
        x = torch.full((n,), 3.25)
    rhs = torch.randn(n, 4, generator=torch.Generator().manual_seed(10))
    start, end = _ranges(n, n, 700)
    for kt in ("spectral", "rbf"):
        _check(kt, x, x, rhs, _params(kt, 1.1), start, end, rows=rows)


@pytest.mark.parametrize("tail", [1, 3, 16])
def test_split_tail(tail):
    """The last items of every XCD split between four wavefronts, the rest one per wavefront."""
    n, batch = 128 * 24 + 5, 3
    x = _points(n, n / 10.0, 11).expand(batch, n)
    rhs = torch.randn(batch, n, 16, generator=torch.Generator().manual_seed(12))
    start, end = (t.expand(batch, -1) for t in _ranges(n, n, 400))
    _check("spectral", x, x, rhs, _params("spectral", [0.2, 0.8, 1.7]), start, end, rows=128, tail=tail)


@pytest.mark.parametrize("rows", [32, 128])
def test_values_that_are_not_finite(rows):
    """A NaN in rhs or in a row's coordinate: near rows, rows whose range does not hold it, other rows."""
    n = 1024
    x = _points(n, n / 10.0, 13)
    rhs = torch.randn(n, 2, generator=torch.Generator().manual_seed(14))
    start, end = _ranges(n, n, 400)
    params = _params("rbf", 1.0)
    clean = _run("rbf", x, x, rhs, params, start, end, rows=rows)
    bad = rhs.clone()
    bad[500, 1] = float("nan")
    out = _run_nan("rbf", x, x, bad, params, start, end, rows)
    near = (x - x[500]).abs() < 4.0
    assert np.all(np.isnan(out[near.numpy(), 1]))
    assert np.array_equal(out[:, 0], clean[:, 0]) or np.allclose(out[:, 0], clean[:, 0], rtol=1e-5, atol=1e-5)
    far = np.array([not (start[i // 128] <= 500 < end[i // 128]) for i in range(n)])
    assert np.all(np.isfinite(out[far]))
    moved = x.clone()
    moved[500] = float("nan")
    out = _run_nan("rbf", moved, x, rhs, params, start, end, rows)
    assert np.all(np.isnan(out[500])) and np.all(np.isfinite(np.delete(out, 500, axis=0)))


def _run_nan(kt, x1, x2, rhs, params, start, end, rows, tail=None):
    args = tuple(t.to(DEVICE) for t in (x1, x2, rhs, params, start, end))
    defines = MatmulSingleConfiguration(kt).make_config(args)
    defines["MATMUL_VARIANT"], defines["MATMUL_ROWS_PER_WAVE"] = "grid", rows
    if rows == 128 and tail is None:
        tail = 0
    if tail is not None:
        defines["MATMUL_GROUP_TAIL"] = tail
    return load_native("matmul", defines).call(*args).cpu().double().numpy()


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("kt,k", [("spectral", 2), ("spectral", 40), ("rbf", 3), ("rbf", 70)])
@pytest.mark.parametrize("rows,tail", [(16, None), (32, None), (64, None), (128, None), (128, 1)])
@pytest.mark.parametrize("layout", ["rows", "columns", "slice"])
def test_rhs_values_that_are_not_finite(kt, k, rows, tail, layout, value):
    """A value of rhs that is not finite reaches every row whose range holds its column, however far
    away, in its own rhs column and no other; everything else keeps its bits.  Columns near the rows
    and out of their reach, in the first, a middle and the last step of a range, with rhs dense across
    its rows, along its columns and neither."""
    n = 2048
    x = _points(n, n / 10.0, 40)
    rhs = torch.randn(n, k, generator=torch.Generator().manual_seed(41))
    start, end = _ranges(n, n, 900)
    params = _params(kt, 1.0)
    def laid_out(t):
        t = t.to(DEVICE)
        if layout == "columns":
            return t.T.contiguous().T
        return torch.cat([t, t], dim=1)[:, :k] if layout == "slice" else t

    clean = _run_nan(kt, x, x, laid_out(rhs), params, start, end, rows, tail)
    assert np.all(np.isfinite(clean))
    column = k - 1
    for j in (0, 700, 1024, int(end[5]) - 1, int(start[9]), n - 1):
        bad = rhs.clone()
        bad[j, column] = value
        out = _run_nan(kt, x, x, laid_out(bad), params, start, end, rows, tail)
        hit = np.array([bool(start[i // 128] <= j < end[i // 128]) for i in range(n)])
        assert hit.any() and not np.isfinite(out[hit, column]).any(), j
        assert np.array_equal(out[~hit], clean[~hit]), j
        assert np.array_equal(np.delete(out, column, 1), np.delete(clean, column, 1)), j


@pytest.mark.parametrize("kt,k", [("spectral", 1), ("spectral", 20), ("rbf", 5), ("rbf", 33)])
@pytest.mark.parametrize("rows", [32, 128])
@pytest.mark.parametrize("lengthscale", [1.0, 0.03])
def test_rhs_values_that_are_not_finite_in_a_long_range(kt, k, rows, lengthscale):
    """Ranges of more steps than are noted one by one, in the grid form and entry by entry."""
    n = 9000
    x = _points(n, n / 10.0, 48)
    rhs = torch.randn(n, k, generator=torch.Generator().manual_seed(49))
    blocks = (n + 127) // 128
    start, end = torch.zeros(blocks, dtype=torch.int32), torch.full((blocks,), n, dtype=torch.int32)
    clean = _run_nan(kt, x, x, rhs, _params(kt, lengthscale), start, end, rows)
    for j in (0, 2047, 2048, 5000, n - 1):
        bad = rhs.clone()
        bad[j, k - 1] = float("nan")
        out = _run_nan(kt, x, x, bad, _params(kt, lengthscale), start, end, rows)
        assert not np.isfinite(out[:, k - 1]).any(), j
        assert np.array_equal(out[:, :k - 1], clean[:, :k - 1]), j


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("kt,k", [("spectral", 2), ("spectral", 40), ("rbf", 3), ("rbf", 70)])
@pytest.mark.parametrize("rows,tail", [(16, None), (32, None), (64, None), (128, None), (128, 1)])
def test_column_coordinates_that_are_not_finite(kt, k, rows, tail, value):
    """A column's NaN reaches every row whose range holds it.  An infinite coordinate does where the
    kernel has an oscillating factor, and is out of reach of every row otherwise (exp(-inf) = 0).  The
    rows of such a range are evaluated entry by entry, within the form's bound of the clean result."""
    n = 2048
    x = _points(n, n / 10.0, 42)
    rhs = torch.randn(n, k, generator=torch.Generator().manual_seed(43))
    start, end = _ranges(n, n, 900)
    params = _params(kt, 1.0)
    for j in (0, 700, 1024, int(end[5]) - 1, n - 1):
        moved, without = x.clone(), rhs.clone()
        moved[j] = value
        without[j] = 0.0
        clean = _run_nan(kt, x, x, without, params, start, end, rows, tail)
        out = _run_nan(kt, x, moved, rhs, params, start, end, rows, tail)
        hit = np.array([bool(start[i // 128] <= j < end[i // 128]) for i in range(n)])
        if kt == "spectral" or value != value:
            assert not np.isfinite(out[hit]).any(), j
        else:
            size = np.abs(without.double().numpy())
            bound = 4e-6 * (np.abs(oracle.dense("rbf", x.numpy(), x.numpy(), params.numpy(), start.numpy(), end.numpy()))
                            @ size) + 2.0 ** -35 * size.sum(0)
            assert np.all(np.abs(out - clean)[hit] <= bound[hit]), j
        assert np.all(np.isfinite(out[~hit])), j


def test_variant_is_refused_for_other_kernels():
    x = _points(300, 30.0, 15).to(DEVICE)
    start, end = (t.to(DEVICE) for t in _ranges(300, 300, 200))
    args = (x, x, torch.randn(300, 2, device=DEVICE), torch.ones(4, device=DEVICE), start, end)
    defines = MatmulSingleConfiguration("locally_periodic").make_config(args)
    defines["MATMUL_VARIANT"] = "grid"
    with pytest.raises(RuntimeError, match="grid form"):
        load_native("matmul", defines).call(*args)


@pytest.mark.parametrize("gap", [1e2, 1e3, 1e4, 1e5, 1e6, 1e9])
@pytest.mark.parametrize("rows", [16, 32, 128])
def test_columns_next_to_a_wide_gap(gap, rows):
    """Groups of 8 columns that lie on both sides of a gap of up to a billion lengthscales, in the ranges
    of row blocks on either side of it: the near columns are as exact as any others, also where they are
    the only ones that are not zero, and where the rows go entry by entry (the second lengthscale)."""
    x = torch.cat([_points(1003, 10.03, 30), _points(500, 5.0, 31) + 10.03 + gap])
    rhs = torch.randn(len(x), 4, generator=torch.Generator().manual_seed(32))
    rhs[:1000, 2:] = 0.0
    rhs[1003:, 2:] = 0.0
    for kt, lengthscale in (("spectral", 1.0), ("rbf", 1.0), ("spectral", 0.03), ("rbf", 0.03)):
        _check(kt, x, x, rhs, _params(kt, lengthscale), *make_ranges(6.0, x), rows=rows)
        mirrored = -x.flip(0)
        _check(kt, mirrored, mirrored, rhs.flip(0), _params(kt, lengthscale), *make_ranges(6.0, mirrored), rows=rows)


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
@pytest.mark.parametrize("rows", [32, 128])
def test_block_around_the_origin(kt, rows):
    """Rows on both sides of the origin, whose distances to the block's middle row are half an ulp of 4
    (2.4e-7) off a representable value, against single columns two to four lengthscales away: without
    what the subtraction rounded off entries are 1.2e-6 to 2.3e-6 off.  The bound is the form's own: two
    factors, each of an exponent below 12 that is rounded twice (6.6e-7 at most together), averaged over
    the grid points that share neither rounding; measured 4.0e-7 in the 2-norm."""
    x1 = torch.cat([_points(64, 2.2, 33) - 6.3, torch.tensor([25000.49 * 2.0 ** -21]), _points(63, 2.2, 34) + 4.05])
    x2 = torch.linspace(-7.5, 7.5, 320)
    params = _params(kt, 0.42)
    if kt == "spectral":
        params[1] = 0.01
    start, end = torch.zeros(1, dtype=torch.int32), torch.full((1,), 320, dtype=torch.int32)
    relative = []
    for first in range(5):
        columns = torch.arange(16) * 20 + 4 * first
        rhs = torch.zeros(320, 16)
        rhs[columns, torch.arange(16)] = 1.0
        out = _run(kt, x1, x2, rhs, params, start, end, rows=rows)
        expected = oracle.matmul(kt, *(t.numpy() for t in (x1, x2, rhs, params, start, end)))
        d = np.abs(x1.double().numpy()[:, None] - x2[columns].double().numpy()) / 0.42
        relative.append((out / expected - 1.0)[(d > 2.0) & (d < 4.0)])
    error = np.sqrt(np.mean(np.concatenate(relative) ** 2))
    print(f"2-norm of the relative error: {error:.2e}")
    assert error < 8e-7


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
@pytest.mark.parametrize("rows", [16, 32, 64, 128])
@pytest.mark.parametrize("scale,sigma", [(4e36, 1e-3), (1e-28, 1.0), (1e-20, 1e15)])
def test_rhs_scales(kt, rows, scale, sigma):
    """rhs so large that its sums over a grid point's columns are not representable although the
    product is, and very small ones; columns of different scales beside them."""
    n = 1000
    x = _points(n, 10.0, 46)
    rhs = torch.rand(n, 3, generator=torch.Generator().manual_seed(47)) * scale
    rhs[:, 1] *= 1e-4
    params = _params(kt, 1.0)
    params[-1] = sigma
    if kt == "spectral":
        params[1] = 0.01
    start, end = _ranges(n, n, 700)
    _check(kt, x, x, rhs, params, start, end, rows=rows)


@pytest.mark.parametrize("kt,k", [("spectral", 3), ("spectral", 20), ("rbf", 3), ("rbf", 20), ("rbf", 40)])
@pytest.mark.parametrize("rows", [16, 32, 64, 128])
@pytest.mark.parametrize("scale", [1e-26, 1e-28, 1e-30])
def test_tiny_rhs(kt, k, rows, scale):
    """Full precision down to where the scale of rhs ends (2^100, of two fp16 halves of which the lower one takes
    steps of 2^-24), although the wavefronts' sums are exchanged at another scale."""
    n = 1400
    x = _points(n, n / 20.0, 63)
    rhs = torch.randn(n, k, generator=torch.Generator().manual_seed(64)) * scale
    start, end = _ranges(n, n, 700)
    _check(kt, x, x, rhs, _params(kt, 1.2), start, end, floor=0.0, rows=rows)


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("row", [0, 63, 64, 127, 192])
@pytest.mark.parametrize("rows", [16, 32, 128])
def test_a_row_coordinate_that_is_not_finite_stays_in_its_row(kt, value, row, rows):
    """Also for the block's middle row, the origin of its relative coordinates."""
    n = 300
    x = _points(n, 30.0, 44)
    rhs = torch.randn(n, 2, generator=torch.Generator().manual_seed(45))
    start, end = _ranges(n, n, 250)
    moved = x.clone()
    moved[row] = value
    out = _run_nan(kt, moved, x, rhs, _params(kt, 1.0), start, end, rows)
    clean = _run_nan(kt, x, x, rhs, _params(kt, 1.0), start, end, rows)
    if kt == "spectral" or value != value:
        assert not np.isfinite(out[row]).any()
    else:
        assert np.all(out[row] == 0.0)
    others = np.arange(n) != row
    assert np.allclose(out[others], clean[others], rtol=0.0, atol=2e-5)


@pytest.mark.parametrize("kt,k", [("spectral", 1), ("spectral", 20), ("rbf", 1), ("rbf", 40)])
@pytest.mark.parametrize("rows", [16, 32, 64, 128])
def test_ranges_at_the_largest_sizes(kt, k, rows):
    """The last columns of as many as the entry point takes (one point and one row, repeated), and empty
    ranges of the largest values: nothing past the largest int is formed."""
    n, m, width = 2**31 - 1 - 128, 300, 700
    x1, one = _points(m, 3.0, 55), torch.ones(1)
    rhs = torch.randn(1, k, generator=torch.Generator().manual_seed(56))
    start = torch.tensor([n - width, 2**31 - 1, n], dtype=torch.int32)
    end = torch.tensor([n, 2**31 - 1, -2**31], dtype=torch.int32)
    params = _params(kt, 1.0)
    args = [x1.to(DEVICE), one.to(DEVICE).expand(n), rhs.to(DEVICE).expand(n, k), params.to(DEVICE), start.to(DEVICE), end.to(DEVICE)]
    defines = MatmulSingleConfiguration(kt).make_config(args)
    defines["MATMUL_VARIANT"], defines["MATMUL_ROWS_PER_WAVE"] = "grid", rows
    if rows == 128:
        defines["MATMUL_GROUP_TAIL"] = 0
    out = load_native("matmul", defines).call(*args).cpu().double().numpy()
    column = oracle.matmul(kt, x1.numpy(), one.numpy(), rhs.numpy(), params.numpy(), np.zeros(3, np.int32), np.ones(3, np.int32))
    expected = width * column
    expected[128:] = 0.0
    envelope = np.abs(oracle.dense("rbf", x1.numpy(), one.numpy(), params[[0, -1]].numpy(), np.zeros(3, np.int32), np.ones(3, np.int32)))
    bound = 3e-6 * width * envelope @ np.abs(rhs.double().numpy())
    bound[128:] = 0.0
    assert np.all(np.abs(out - expected) <= bound)


@pytest.mark.parametrize("kt,k", [("spectral", 2), ("spectral", 20), ("spectral", 40), ("rbf", 3), ("rbf", 20), ("rbf", 50)])
@pytest.mark.parametrize("rows", [16, 32, 64, 128])
@pytest.mark.parametrize("lengthscale", [1.0, 0.03])
@pytest.mark.parametrize("small", [1e-27, 2.5e-26, 1e-20])
def test_rhs_that_grows_along_the_columns(kt, k, rows, lengthscale, small):
    """Tiny values in front of ordinary ones (and behind them), whose sums follow the column's scale down."""
    n = 1400
    x = _points(n, n / 10.0, 59)
    rhs = torch.randn(n, k, generator=torch.Generator().manual_seed(60))
    rhs[:500] *= small
    rhs[900:] *= small
    start, end = _ranges(n, n, 900)
    _check(kt, x, x, rhs, _params(kt, lengthscale), start, end, rows=rows)

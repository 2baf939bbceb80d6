"""The grid form's workgroups that take several row blocks together (128 rows per wavefront): ranges that
overlap in every way, groups cut off by the matrix, columns shared by all ranges on both sides of what one
wavefront takes, windows up to what fits the workgroup's memory, batch dimensions that do not collapse.

Tolerance as in test_grid_form_gpu."""
import pytest
import torch

from kernel_matmul_amd.compile import load_native
from kernel_matmul_amd.configurations import MatmulSingleConfiguration
from kernel_matmul_amd.ranges import make_ranges
from tests.test_grid_form_gpu import DEVICE, _check, _params, _points

pytestmark = pytest.mark.gpu


def _rhs(*shape, seed=3):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


def _group_check(kt, x1, x2, rhs, params, start, end):
    _check(kt, x1, x2, rhs, params, start.int(), end.int(), rows=128)


@pytest.mark.parametrize("n", [161, 300, 512, 513, 640, 1000, 1152])
@pytest.mark.parametrize("kt,k", [("spectral", 3), ("spectral", 17), ("spectral", 40), ("rbf", 5), ("rbf", 20), ("rbf", 50)])
def test_symmetric_pattern(kt, k, n):
    """One to nine row blocks with the pattern that make_ranges builds."""
    x = _points(n, n / 10.0, n)
    start, end = make_ranges(9.0, x.to(DEVICE))
    _group_check(kt, x, x, _rhs(n, k), _params(kt, 1.5), start.cpu(), end.cpu())


# Columns that all four ranges share: none, fewer than a step, one wavefront's, just below and above what is
# shared out, many.
@pytest.mark.parametrize("width", [300, 385, 400, 512, 639, 641, 672, 900, 2500])
@pytest.mark.parametrize("lengthscale", [0.4, 1.5])
def test_shared_columns(width, lengthscale):
    n = 2700
    x = _points(n, n / 20.0, width)
    mid = torch.arange(22) * 128 + 64
    start, end = (mid - width // 2).clamp(0, n), (mid + (width + 1) // 2).clamp(0, n)
    _group_check("spectral", x, x, _rhs(n, 4), _params("spectral", lengthscale), start, end)


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
@pytest.mark.parametrize("ranges", [
    [(0, 1000), (0, 1000), (0, 1000), (0, 1000)],      # equal
    [(0, 1000), (1000, 1000), (300, 299), (0, 200)],   # empty and backward ones among them
    [(600, 900), (400, 700), (200, 500), (0, 300)],    # descending
    [(0, 170), (200, 380), (500, 700), (800, 1000)],   # apart, with gaps
    [(0, 1000), (400, 600), (450, 550), (490, 510)],   # nested
    [(0, 5), (3, 8), (100, 101), (990, 1000)],         # too short
    [(-5, 400), (90, 2000), (-9, -3), (999, 5000)],    # beyond the columns
    [(31, 997), (1, 966), (33, 999), (2, 67)],         # odd
])
def test_ranges_that_overlap_in_every_way(kt, ranges):
    n, m = 1000, 512
    x1, x2 = _points(m, 20.0, 1), _points(n, 20.0, 2)
    start, end = torch.tensor(ranges, dtype=torch.int32).T.contiguous()
    lo = start.clamp(0, n)
    # (the oracle takes ranges within the columns)
    args = (kt, x1, x2, _rhs(n, 3), _params(kt, 1.2))
    if torch.equal(lo, start) and bool((end <= n).all()) and bool((end >= start).all()):
        _group_check(*args, start, end)
        return
    from tests.test_grid_form_gpu import _run
    hi = torch.maximum(end.clamp(0, n), lo)
    assert (_run(*args, start, end, rows=128) == _run(*args, torch.minimum(lo, hi), hi, rows=128)).all()


@pytest.mark.parametrize("lengthscale", [0.5, 0.55, 0.6, 0.65, 0.7, 0.8, 1.0])
@pytest.mark.parametrize("k", [16, 32])
def test_windows_up_to_the_largest(lengthscale, k):
    n = 1100
    x = torch.arange(n) / 10.0
    start, end = make_ranges(4.0, x.to(DEVICE))
    _group_check("spectral", x, x, _rhs(n, k), _params("spectral", lengthscale), start.cpu(), end.cpu())


@pytest.mark.parametrize("swap", [(0, 1), (5, 130), (128, 300), (255, 256), (383, 700)])
@pytest.mark.parametrize("what", ["rows", "columns"])
def test_single_coordinates_out_of_order(swap, what):
    n = 768
    x1, x2 = _points(n, 60.0, 5), _points(n, 60.0, 5)
    x = x1 if what == "rows" else x2
    x[[swap[0], swap[1]]] = x[[swap[1], swap[0]]]
    mid = torch.arange(6) * 128 + 64
    _group_check("spectral", x1, x2, _rhs(n, 2), _params("spectral", 1.1), (mid - 250).clamp(0, n), (mid + 250).clamp(0, n))


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
def test_batch_dimensions_that_do_not_collapse(kt):
    n = 700
    x = _points(n, 70.0, 7).expand(2, 3, n)
    params = _params(kt, [0.9, 1.4, 2.0])[None].expand(2, 3, -1)
    rhs = _rhs(2, 1, n, 6).expand(2, 3, n, 6)
    start, end = (t.cpu().expand(2, 3, -1) for t in make_ranges(8.0, x[0, 0].to(DEVICE)))
    _group_check(kt, x, x, rhs, params, start, end)


@pytest.mark.parametrize("core", [257, 259, 260, 272, 287, 288, 383, 384])
@pytest.mark.parametrize("kt,k", [("spectral", 4), ("rbf", 20)])
@pytest.mark.parametrize("ends", ["apart", "equal", "last"])
def test_shared_columns_that_are_no_whole_steps(core, kt, k, ends):
    """Four shares of the core in whole steps are more than it has; behind its end the ranges go on, stop
    together, or stop at the last column."""
    m, n = 512, 384 + core + (0 if ends == "last" else 384)
    x1, x2 = _points(m, 40.0, core), _points(n, 40.0, core + 1)
    row = torch.arange(4)
    start = row * 128
    end = 384 + core + (row * 128 if ends == "apart" else 0 * row)
    _group_check(kt, x1, x2, _rhs(n, k), _params(kt, 3.0), start, end)


@pytest.mark.parametrize("density,cutoff", [(22.0, 12.0), (25.0, 25.0), (10.0, 40.0)])
def test_rectangular_pattern(density, cutoff):
    """make_ranges for two sets of points: ranges that start and end anywhere."""
    m, n = 2600, 2500
    x1, x2 = _points(m, m / density, 1), _points(n, m / density, 2)
    start, end = make_ranges(cutoff, x1.to(DEVICE), x2.to(DEVICE))
    _group_check("spectral", x1, x2, _rhs(n, 4), _params("spectral", 2.0), start.cpu(), end.cpu())


@pytest.mark.parametrize("border", [128, 256, 300, 384])
@pytest.mark.parametrize("kt,k", [("spectral", 4), ("rbf", 20)])
def test_ascending_runs_out_of_order(kt, k, border):
    """Columns in two ascending runs, the upper one first: the pieces of a shared core reach further than its
    first and last coordinate say."""
    n = 512
    x = _points(n, 10.0, border)
    order = torch.cat([torch.arange(border, n), torch.arange(border)])
    start, end = torch.zeros(4), torch.full((4,), float(n))
    _group_check(kt, x, x[order], _rhs(n, k), _params(kt, 0.8), start, end)


@pytest.mark.parametrize("kt", ["spectral", "rbf"])
@pytest.mark.parametrize("m", [2**31 - 512 + 5, 2**31 - 1 - 128])
@pytest.mark.parametrize("tail", [0, 4])
def test_rows_at_the_largest_sizes(kt, m, tail):
    """The last rows of as many as the entry point takes (all others' ranges are empty) are those of these rows
    alone: the last group's wavefronts without a row block stay within the rows."""
    n, last = 1000, m - (m - 1) // 512 * 512
    x1 = torch.full((m,), -1e3, device=DEVICE)
    x1[m - last:] = _points(last, 50.0, 1).to(DEVICE)
    x2, rhs = _points(n, 50.0, 2).to(DEVICE), _rhs(n, 1).to(DEVICE)
    params = _params(kt, 1.1).to(DEVICE)
    blocks, own = (m + 127) // 128, (last + 127) // 128
    start = torch.zeros(blocks, dtype=torch.int32, device=DEVICE)
    end = torch.zeros(blocks, dtype=torch.int32, device=DEVICE)
    end[blocks - own:] = n

    def call(*args):
        defines = MatmulSingleConfiguration(kt).make_config(args)
        defines["MATMUL_VARIANT"], defines["MATMUL_ROWS_PER_WAVE"], defines["MATMUL_GROUP_TAIL"] = "grid", 128, tail
        return load_native("matmul", defines).call(*args)

    result = call(x1, x2, rhs, params, start, end)
    alone = call(x1[m - last:], x2, rhs, params, start[blocks - own:], end[blocks - own:])
    assert torch.equal(result[m - last:], alone)
    assert not result[:m - last].any()

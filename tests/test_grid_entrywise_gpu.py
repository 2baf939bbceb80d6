"""The grid form's row blocks that go entry by entry because their points are sparse against the lengthscale, with
as many rows at a time as one, two, four or eight wavefronts per row block take: row blocks that end in each group of
16 rows, ranges on both sides of what is tabulated at a time.

Tolerance as in test_grid_form_gpu."""
import pytest
import torch

from kernel_matmul_amd.ranges import make_ranges
from tests.test_grid_form_gpu import DEVICE, _check, _params, _points

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [128, 64, 32, 16])
@pytest.mark.parametrize("kt,k", [("spectral", 3), ("spectral", 20), ("spectral", 40), ("rbf", 5), ("rbf", 20), ("rbf", 50)])
@pytest.mark.parametrize("n", [145, 192, 383, 700])
def test_sparse_points(kt, k, n, rows):
    x = _points(n, float(n), n)
    rhs = torch.randn(n, k, generator=torch.Generator().manual_seed(3))
    start, end = make_ranges(60.0, x.to(DEVICE))
    _check(kt, x, x, rhs, _params(kt, 0.6), start.cpu().int(), end.cpu().int(), rows=rows)

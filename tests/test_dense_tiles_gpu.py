"""Dense matrices and their gradient at the edges of what a wavefront writes and reads: whole and ragged groups of four
columns, shares and row groups, ranges that end inside of them, weights in any layout.

The matrix against float64 closed forms: an exponent u^2 of up to 95 (lengthscales from 0.7 on, distances up to 8) and a phase
of up to 14 turns, two roundings (2^-24 of either) each.  The gradient: the same for each term, relative to the largest, of
which roundings of random signs add up."""
import math

import numpy as np
import pytest
import torch

from kernel_matmul_amd import _native
from oracle import kernels as oracle

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")
RELATIVE = 2.0 ** -23 * (95 * math.log(2) + 2 * math.pi * 14)
COLUMNS = {"rbf": 2, "spectral": 3, "locally_periodic": 4}


def _inputs(kernel, batch, m, n, seed=0):
    g = torch.Generator().manual_seed(seed)
    x1 = torch.sort(torch.rand(batch, m, generator=g) * 8)[0]
    x2 = torch.sort(torch.rand(batch, n, generator=g) * 8)[0]
    params = 0.7 + torch.rand(batch, COLUMNS[kernel], generator=g)
    blocks = -(-m // 128)
    start = (torch.arange(batch * blocks).view(batch, blocks) * 37 % max(n // 2, 1)).int()
    end = (start + n // 3 + 1 + 5 * torch.arange(blocks)).clamp(max=n).int()
    end[:, -1] = n
    if blocks > 2:
        end[:, 1] = start[:, 1]
    return x1, x2, params, start, end


@pytest.mark.parametrize("kernel", ["rbf", "spectral", "locally_periodic"])
@pytest.mark.parametrize("batch,m,n", [
    (1, 1, 1), (1, 15, 4), (2, 16, 5), (1, 17, 252), (3, 31, 255), (1, 33, 256), (2, 127, 257), (1, 129, 260), (1, 300, 515),
    (1, 385, 1028), (9, 130, 64), (40, 260, 68),
])
def test_tiles(kernel, batch, m, n):
    args = _inputs(kernel, batch, m, n)
    on = [t.to(DEVICE) for t in args]
    dense = _native.dense(kernel, *on).cpu().double().numpy()
    mine = np.stack([oracle.dense(kernel, *(t[b].numpy() for t in args)) for b in range(batch)])
    assert ((dense == 0) >= (mine == 0)).all()
    np.testing.assert_allclose(dense, mine, rtol=RELATIVE, atol=2 * RELATIVE)
    g = torch.Generator().manual_seed(5)
    weights = torch.randn(batch, m, n, generator=g)
    gapped = torch.full((batch, 2 * m, 3 * n), float("nan"))
    gapped[:, ::2, ::3] = weights
    grads = [_native.dense_bwd(kernel, *on, w) for w in (
        weights.to(DEVICE), weights.mT.contiguous().to(DEVICE).mT, gapped.to(DEVICE)[:, ::2, ::3])]
    assert torch.equal(grads[0], grads[1]) and torch.equal(grads[0], grads[2])
    for b in range(batch):
        x1, x2, p, start, end = (t[b].numpy() for t in args)
        terms = oracle.kernel_matrix_grad(kernel, x1, x2, p) * oracle.range_mask(start, end, m, n) * weights[b].double().numpy()
        size = abs(terms).max(axis=(1, 2)) * np.count_nonzero(terms, axis=(1, 2)) ** 0.5  # (of a sum of random signs)
        difference = abs(grads[0][b].cpu().double().numpy() - terms.sum(axis=(1, 2)))
        assert (difference <= RELATIVE * size + 1e-12).all()


@pytest.mark.parametrize("n", [2 ** 31 - 132, 2 ** 31 - 129, 2 ** 31 - 256])
def test_columns_up_to_the_largest_number(n):
    """The columns behind the last ones of a matrix lie past the largest int.  Points in one place: every entry is one."""
    x1, x2 = torch.zeros(1, device=DEVICE), torch.zeros(1, device=DEVICE).expand(n)
    start, end = torch.tensor([5], dtype=torch.int32, device=DEVICE), torch.tensor([n - 3], dtype=torch.int32, device=DEVICE)
    dense = _native.dense("rbf", x1, x2, torch.ones(2, device=DEVICE), start, end)[0]
    assert not dense[:5].any() and not dense[-3:].any()
    assert int((dense == 1).sum()) == n - 8


def test_gradient_of_ranges_up_to_the_largest_number_of_columns():
    """Shares of a short range that begin behind it lie past the largest int.  Points in one place: an entry's derivative
    by the output scale is one, by the lengthscale zero."""
    n = 2 ** 31 - 129
    x1, x2 = torch.zeros(1, device=DEVICE), torch.zeros(1, device=DEVICE).expand(n)
    weights = torch.ones(1, 1, device=DEVICE).expand(1, n)
    for first in (n - 100, n - 1000, n - 2 ** 20):
        start, end = (torch.tensor([i], dtype=torch.int32, device=DEVICE) for i in (first, n))
        grad = _native.dense_bwd("rbf", x1, x2, torch.ones(2, device=DEVICE), start, end, weights)
        # (whole numbers: exact)
        assert grad.tolist() == [0.0, n - first]


def test_gradient_of_more_row_blocks_than_a_launch_takes():
    """Eight wavefronts each for 2^23 row blocks and more are more threads than a launch may have.  Points in one place."""
    m = 2 ** 30 + 1024
    x1, x2 = torch.zeros(1, device=DEVICE).expand(m), torch.zeros(1, device=DEVICE)
    start, end = (torch.full((1,), i, dtype=torch.int32, device=DEVICE).expand(m // 128) for i in (0, 1))
    grad = _native.dense_bwd("rbf", x1, x2, torch.ones(2, device=DEVICE), start, end, torch.ones(1, 1, device=DEVICE).expand(m, 1))
    assert grad.tolist() == [0.0, m]  # (whole numbers: exact)

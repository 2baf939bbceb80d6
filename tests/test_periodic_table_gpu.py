"""Locally periodic forward from tabulated phases: every decomposition of its launch table, at its edges, against
float64, and against the kernel that evaluates each entry directly over the forms that both accept.

Tolerance of an entry K rhs, relative: its factors 2^-21 together (two fp16 halves each) and the sums as much; the exponent
u^2 + cl sin^2 of its power of two four roundings (2^-24 of it each) and, tabulated, cosines times cl / 2 (2^-22 each, four
of them); the phase, formed as a product where entries are evaluated directly, two roundings (2^-24) of its turns, of
which the exponent feels pi cl times as much.  Entries below 2^-39 of the output scale are left out."""
import pytest
import torch

from kernel_matmul_amd.compile import load_native
from kernel_matmul_amd.configurations import MatmulSingleConfiguration

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")


def _inputs(m, n, k, batch, density=12.0, offset=3.0, seed=0):
    g = torch.Generator().manual_seed(seed)

    def u(lo, hi):
        return lo + (hi - lo) * torch.rand(batch, generator=g)

    x2 = torch.sort(torch.rand(n, generator=g) * (n / density))[0] + offset
    x1 = x2[:m].clone() if m <= n else torch.sort(torch.rand(m, generator=g) * (n / density))[0] + offset
    params = torch.stack([u(0.4, 2.5), u(0.4, 2.0), u(0.4, 2.0), u(-1.0, 2.0)], dim=-1)
    rhs = torch.randn(n, k, generator=g)
    blocks = -(-m // 128)
    start = (torch.arange(blocks) * 61 % max(n - 200, 1)).int()
    end = (start + 200 + 37 * torch.arange(blocks) % 300).clamp(max=n).int()
    t = [x1, x2, rhs, params, start, end]
    return [t[0].expand(batch, m), t[1].expand(batch, n), t[2].expand(batch, n, k), t[3], t[4].expand(batch, -1),
            t[5].expand(batch, -1)]


def _operator(args, variant=None, rows=None):
    defines = MatmulSingleConfiguration("locally_periodic").make_config(args)
    if variant:
        defines["MATMUL_VARIANT"] = variant
    if rows:
        defines["MATMUL_ROWS_PER_WAVE"] = rows
    return load_native("matmul", defines)


def _exact(args, items):
    """(result, tolerance) of some batch items in float64."""
    out, tolerance = [], []
    for b in items:
        x1, x2, rhs, p, start, end = (t[b].cpu().double() for t in args)
        d = x1[:, None] - x2[None, :]
        u2, cl, turns = d ** 2 / p[0] ** 2 * 0.7213475, 2.885390 / p[1], d / p[2]
        K = p[3] * torch.exp2(-(d / p[0]) ** 2 * 0.72134752044448170368 - 2.8853900817779268147 / p[1] * torch.sin(torch.pi * turns) ** 2)
        column = torch.arange(x2.shape[0])[None, :]
        block = torch.arange(x1.shape[0]) // 128
        inside = (column >= start[block][:, None]) & (column < end[block][:, None])
        K = K * inside
        out.append(K @ rhs)
        relative = 2.0 ** -20 + 2.0 ** -22 * (u2 + cl.abs()) + 2.0 ** -22 * 3.2 * cl.abs() * turns.abs()
        tolerance.append((K.abs() * relative + inside * p[3].abs() * 2.0 ** -38) @ rhs.abs())
    return torch.stack(out), torch.stack(tolerance)


def _check(args, name=None):
    args = [t.to(DEVICE) for t in args]
    op = _operator(args)
    if name:
        assert name in op.describe(*args)
    out = op.call(*args)
    items = sorted({0, args[3].shape[0] // 2, args[3].shape[0] - 1})
    exact, tolerance = _exact(args, items)
    assert float(((out[items].cpu().double() - exact).abs() / (tolerance + 1e-30)).max()) <= 1.0
    direct = _operator(args, "mfma_f16_direct", 64).call(*args)
    torch.testing.assert_close(out, direct, rtol=1e-5, atol=2 * float(tolerance.max()))


@pytest.mark.parametrize("k,batch,name", [
    (16, 16, "G=1, R=2, W=8"), (1, 30, "G=1, R=2, W=8"), (16, 31, "G=1, R=4, W=8"), (3, 225, "G=1, R=4, W=8"),
    (16, 226, "G=1, R=8, W=4"), (15, 999, "G=1, R=8, W=4"), (16, 1000, "G=1, R=8, W=2"), (2, 2499, "G=1, R=8, W=2"),
    (16, 2500, "G=1, R=8, W=1"), (17, 16, "G=2, R=4, W=8"), (32, 55, "G=2, R=4, W=8"), (32, 56, "G=2, R=8, W=8"),
    (31, 100, "G=2, R=8, W=8"), (32, 101, "G=2, R=8, W=4"), (20, 1000, "G=2, R=8, W=2"), (32, 2500, "G=2, R=8, W=1"),
    (33, 16, "G=4, R=2, W=8"), (64, 31, "G=4, R=4, W=8"), (64, 55, "G=4, R=4, W=8"), (40, 56, "G=4, R=4, W=4"),
    (64, 500, "G=4, R=4, W=2"), (63, 1250, "G=4, R=4, W=1"), (65, 25, "G=4, R=4, W=8"),
])
def test_decompositions(k, batch, name):
    _check(_inputs(131, 700, k, batch), name)


@pytest.mark.parametrize("m,n", [(128, 33), (255, 64), (257, 1), (640, 1031), (4000, 4000)])
@pytest.mark.parametrize("density", [0.7, 6.0, 300.0])
@pytest.mark.parametrize("offset", [0.0, -2.0, 5000.0])
def test_shapes_and_spacings(m, n, density, offset):
    """Steps with and without gaps (0.7 points per unit: all entries directly), next to the origin and far from it."""
    args = _inputs(m, n, 5, 40, density, offset)
    if offset > 100:  # coordinates are multiples of 2^-11 there; their differences stay exact
        args[0], args[1] = ((t * 1024).round() / 1024 for t in args[:2])
    _check(args)
    args[3] = args[3].clone()
    args[3][:, 1] = 0.2
    _check(args)


@pytest.mark.parametrize("column,value", [(1, 0.361), (1, 0.36), (1, 0.05), (1, 0.002), (1, 50.0), (1, -1.5), (0, 0.02), (0, 40.0), (2, 0.05),
                                          (2, 1e4), (3, 0.0), (0, -0.8)])
def test_parameters(column, value):
    """On both sides of the second lengthscale up to which the squared sine is taken; signs and extremes."""
    args = _inputs(260, 900, 4, 40)
    args[3][:, column] = value
    if value < 0 and column == 1:  # (entries of up to e^(4/3): within fp16's range at these scales)
        args[3][:, 3] = 0.5
    _check(args)


@pytest.mark.parametrize("what", ["rhs", "x1", "x2"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("at", [0, 130, 333, 699])
@pytest.mark.parametrize("batch", [16, 226, 2500])
def test_values_that_are_not_finite(what, value, at, batch):
    """Within reach of a row block or not: NaN where the direct kernel has it."""
    args = _inputs(512, 700, 3, batch // 4 + 1)
    args[3][:, 0] = 0.4
    args = [t.clone() for t in args]
    if what == "rhs":
        args[2][:, at, 1] = value
    else:
        args[0 if what == "x1" else 1][:, min(at, 511 if what == "x1" else 699)] = value
    args = [t.to(DEVICE) for t in args]
    out, direct = _operator(args).call(*args), _operator(args, "mfma_f16_direct", 64).call(*args)
    torch.testing.assert_close(out, direct, rtol=1e-4, atol=1e-4, equal_nan=True)


@pytest.mark.parametrize("what,value", [(0, float("nan")), (1, 0.0), (1, float("nan")), (2, 0.0), (2, float("nan"))])
def test_parameters_that_make_entries_nan(what, value):
    args = _inputs(300, 600, 2, 16)
    args[3][:, what] = value
    args = [t.to(DEVICE) for t in args]
    out, direct = _operator(args).call(*args), _operator(args, "mfma_f16_direct", 64).call(*args)
    torch.testing.assert_close(out, direct, rtol=1e-4, atol=1e-4, equal_nan=True)


@pytest.mark.parametrize("batch", [16, 300, 2500])
def test_strides_empty_ranges_and_scales(batch):
    """Transposed, gapped and reversed-range inputs; rhs columns over 24 decades, zeros, tiny and huge ones."""
    args = [t.clone() for t in _inputs(256, 500, 6, batch)]
    args[4][:, 1] = 400
    args[5][:, 1] = 400
    args[2] *= torch.tensor([1e-12, 1e-3, 0.0, 1.0, 1e6, 1e12])
    wide = torch.full((batch, 6, 1000), float("nan"))
    wide[:, :, ::2] = args[2].transpose(1, 2)
    x2 = torch.full((batch, 1500), float("nan"))
    x2[:, ::3] = args[1]
    plain = [t.to(DEVICE) for t in args]
    strided = list(plain)
    strided[1], strided[2] = x2.to(DEVICE)[:, ::3], wide.to(DEVICE)[:, :, ::2].transpose(1, 2)
    out = _operator(plain).call(*plain)
    assert bool((out[:, 128:] == 0).all()) and bool((out[:, :, 2] == 0).all())
    assert torch.equal(out, _operator(strided).call(*strided))
    exact, tolerance = _exact(plain, [0])
    assert bool(((out[0].cpu().double() - exact[0]).abs() <= tolerance[0] + 1e-25).all())


def test_unsorted_coordinates():
    args = [t.clone() for t in _inputs(512, 700, 5, 40)]
    g = torch.Generator().manual_seed(2)
    args[0], args[1] = args[0][:, torch.randperm(512, generator=g)], args[1][:, torch.randperm(700, generator=g)]
    _check(args)

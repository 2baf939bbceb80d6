"""fp32 contraction through the grid and by entries: every decomposition of its launch table, at its edges, against float64,
and against the kernel that evaluates each entry directly where values are not finite.

Tolerance of an entry K rhs against float64, relative to the entry without an oscillating factor: sums of at most `columns`
products, added one after another (2^-24 each), twice that of 60 grid points; the exponent u^2 + cl sin^2 of its power of two
four roundings (2^-24 of it each); what the grid's spacing and the end of its windows leave out (2^-21); cosines and sines
2^-22 each, four of them, and where the phase is tabulated, times cl / 2.  Entries below 2^-126 are left out."""
import pytest
import torch

from kernel_matmul_amd.compile import load_native
from kernel_matmul_amd.configurations import MatmulSingleConfiguration

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")
KERNELS = ["rbf", "spectral", "locally_periodic"]


def _inputs(kernel, m, n, k, batch, density=12.0, form="sorted", seed=0):
    g = torch.Generator().manual_seed(seed)

    def u(lo, hi):
        return lo + (hi - lo) * torch.rand(batch, generator=g)

    x2 = torch.sort(torch.rand(n, generator=g) * (n / density))[0] + 200.0
    if form == "gaps":
        x2 = x2 + torch.where(torch.arange(n) > n // 3, 60.0, 0.0) + torch.where(torch.arange(n) > n // 2 + 3, 4.0, 0.0)
    x1 = x2[:m].clone() if m <= n else torch.sort(torch.rand(m, generator=g) * (n / density))[0] + 200.0
    if form == "reversed":
        x2 = x2.flip(0)
    elif form == "shuffled":
        x2 = x2[torch.randperm(n, generator=g)]
    elif form == "far":
        x2 = x2 + 14.0 / 0.85 * 0.9
    columns = {"rbf": [u(0.5, 2.0), u(-1.0, 2.0)], "spectral": [u(0.5, 2.0), u(0.1, 2.0), u(-1.0, 2.0)],
               "locally_periodic": [u(0.5, 2.0), u(0.3, 2.0), u(0.4, 2.0), u(-1.0, 2.0)]}[kernel]
    rhs = torch.randn(n, k, generator=g)
    blocks = -(-m // 128)
    start = (torch.arange(blocks) * 61 % max(n - 200, 1)).int()
    end = (start + 157 + 37 * torch.arange(blocks) % 300).clamp(max=n).int()
    end[-1] = n
    t = [x1, x2, rhs, torch.stack(columns, dim=-1), start, end]
    return [t[0].expand(batch, m), t[1].expand(batch, n), t[2].expand(batch, n, k), t[3], t[4].expand(batch, -1), t[5].expand(batch, -1)]


def _operator(kernel, args, variant="mfma_f32"):
    defines = MatmulSingleConfiguration(kernel).make_config(args)
    defines["MATMUL_VARIANT"] = variant
    return load_native("matmul", defines)


def _exact(kernel, args, items):
    out, tolerance = [], []
    for b in items:
        x1, x2, rhs, p, start, end = (t[b].cpu().double() for t in args)
        d = x1[:, None] - x2[None, :]
        exponent = 0.72134752044448170368 * (d / p[0]) ** 2
        phase = torch.zeros_like(d)
        cosine = torch.ones_like(d)
        if kernel == "spectral":
            cosine = torch.cos(2 * torch.pi * p[1] * d)
            phase += 2.0 ** -20
        elif kernel == "locally_periodic":
            cl = 2.8853900817779268147 / p[1]
            exponent = exponent + cl * torch.sin(torch.pi * d / p[2]) ** 2
            phase += 2.0 ** -20 * cl
        column = torch.arange(x2.shape[0])[None, :]
        block = torch.arange(x1.shape[0]) // 128
        inside = (column >= start[block][:, None]) & (column < end[block][:, None])
        K = p[-1] * torch.exp2(-exponent) * inside
        out.append((K * cosine) @ rhs)
        count = (end - start)[block][:, None] + 60
        relative = 2.0 ** -24 * (count + 4 * exponent + 8) + 2.0 ** -21 + phase
        tolerance.append((K.abs() * relative + inside * p[-1].abs() * 2.0 ** -126) @ rhs.abs())
    return torch.stack(out), torch.stack(tolerance)


def _on_device(args):
    return [t.contiguous().to(DEVICE) if t.shape[0] < 2 else t[:1].contiguous().to(DEVICE).expand(t.shape) if t.stride(0) == 0
            else t.to(DEVICE) for t in args]


def _check(kernel, args, text, below=0.0):
    args = _on_device(args)
    op = _operator(kernel, args)
    assert text in op.describe(*args), op.describe(*args)
    result = op.call(*args)
    result = (result[0] if isinstance(result, (tuple, list)) else result).cpu().double()
    batch = args[0].shape[0]
    items = sorted({0, 1, batch // 2, batch - 1})
    exact, tolerance = _exact(kernel, args, items)
    tolerance += below  # a result's own rounding there
    assert ((result[items] - exact).abs() <= tolerance).all(), float(((result[items] - exact).abs() / tolerance).max())


# items 130 / 390 / 2100 / 5100: eight, four, two and one wavefronts a row block (spectral with more than 16 columns four from
# 400, two from 513 and one from 741 on)
@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("batch,k", [(44, 16), (130, 1), (700, 16), (1700, 15), (140, 17), (250, 32), (24, 70)])
def test_every_decomposition_against_float64(kernel, batch, k):
    items = 3 * batch * -(-k // 32)
    four = kernel == "spectral" and k > 16
    if four and items < 400:
        w = None
    elif four:
        w = 4 if items < 700 else 1
    elif kernel == "locally_periodic":
        w = 8 if items < 250 else (4 if items < 5000 else 2)
    else:
        w = 8 if items < 250 else (4 if items < 2000 else (2 if items < 5000 else 1))
    text = "fwd_grid_f32<%s, G=%d, W=%d>" % (kernel, 1 if k <= 16 else 2, w) if w else "f32"
    _check(kernel, _inputs(kernel, 300, 700, k, batch, seed=batch), text)


@pytest.mark.parametrize("m,batch,k,w", [(384, 170, 17, 4), (300, 171, 32, 2), (384, 123, 40, 2), (300, 247, 20, 1)])
def test_wavefronts_of_four_operand_groups(m, batch, k, w):
    _check("spectral", _inputs("spectral", m, 700, k, batch, seed=batch), "fwd_grid_f32<spectral, G=2, W=%d>" % w)


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("form,density", [("sorted", 0.2), ("sorted", 2.0), ("sorted", 300.0), ("gaps", 12.0), ("reversed", 12.0),
                                          ("shuffled", 12.0), ("far", 40.0)])
def test_forms_of_coordinates_against_float64(kernel, form, density):
    _check(kernel, _inputs(kernel, 257, 650, 16, 44, density, form), "fwd_grid_f32")


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("m,n", [(1, 1), (128, 95), (128, 96), (128, 159), (129, 161), (385, 32)])
def test_ragged_and_short_ranges(kernel, m, n):
    batch = 130 // -(-m // 128) + 1
    args = _inputs(kernel, m, n, 5, batch)
    args[4], args[5] = torch.zeros_like(args[4]), torch.full_like(args[5], n)
    _check(kernel, args, "fwd_grid_f32")


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("value", [1e38, 1e31, 1e25, 1e-30, 1e-37])
def test_values_of_rhs_at_the_ends_of_the_range(kernel, value):
    # one column of rhs with a value that others cannot make up for, one all of whose values are of that size
    args = [t.clone() for t in _inputs(kernel, 256, 650, 16, 64)]
    args[3][:, -1] = args[3][:, -1].abs().clamp(max=1.0) * 0.5
    args[2][:, 100, 3] = value
    args[2][:, :, 7] *= min(value, 1e34)
    _check(kernel, args, "fwd_grid_f32", below=2.0 ** -148)


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("what", ["rhs inf", "rhs nan", "rhs far nan", "x2 nan", "x2 inf", "x1 nan", "lengthscale zero", "lengthscale inf"])
def test_values_that_are_not_finite(kernel, what):
    args = [t.clone() for t in _inputs(kernel, 256, 650, 16, 64)]
    value = float(what.split()[-1]) if what.split()[-1] in ("inf", "nan") else 0.0
    if what.startswith("rhs far"):
        args[5][...] = 650
        args[2][1, 640, 3] = value
    elif what.startswith("rhs"):
        args[2][1, 100, 3] = value
    elif what.startswith("x2"):
        args[1][1, 90] = value
    elif what.startswith("x1"):
        args[0][1, 130] = value
    else:
        args[3][1, 0] = 0.0 if "zero" in what else float("inf")
    args = [t.to(DEVICE) for t in args]
    got, want = (_operator(kernel, args, v).call(*args) for v in ("mfma_f32", "mfma_f32_direct"))
    got, want = (r[0] if isinstance(r, (tuple, list)) else r for r in (got, want))
    # (an infinity times an entry is NaN where the entry is zero in fp32, which the two round differently about 2^-126)
    finite = want.isfinite()
    assert torch.equal(got.isfinite(), finite)
    assert torch.allclose(got[finite], want[finite], rtol=1e-3, atol=1e-4 * float(want[finite].abs().median()) + 1e-30)

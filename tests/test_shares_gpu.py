"""Few rows against many points: ranges in shares of several workgroups, and the steps of a range shared by a workgroup's
wavefronts entry by entry, against float64; values that are not finite against one workgroup for each range.

Tolerance of an entry K rhs against float64, relative to the entry without an oscillating factor: its two factors 2^-21
together (two fp16 halves each), twice that through the grid, and the sums as much; the exponent u^2 + cl sin^2 of its power
of two four roundings (2^-24 of it each); cosines 2^-22, four of them, and where they stand in the exponent, times cl / 2.
Entries below 2^-37 of the output scale are left out (2^-38: each half of the bound)."""
import ctypes

import pytest
import torch

from kernel_matmul_amd import _native
from kernel_matmul_amd.compile import load_native
from kernel_matmul_amd.configurations import MatmulSingleConfiguration
from kernel_matmul_amd.ranges import make_ranges

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")
KERNELS = ["rbf", "spectral", "locally_periodic"]


def _inputs(kernel, m, n, k, batch, density=10.0, cutoff=12.0, local=False, seed=0):
    g = torch.Generator().manual_seed(seed)

    def u(lo, hi):
        return lo + (hi - lo) * torch.rand(batch, generator=g)

    extent = n / density
    x2 = torch.sort(torch.rand(n, generator=g) * extent)[0]
    x1 = torch.sort(torch.rand(m, generator=g) * (min(extent, 30.0) if local else extent))[0]
    columns = {"rbf": [u(0.5, 2.0), u(-1.0, 2.0)], "spectral": [u(0.5, 2.0), u(0.1, 2.0), u(-1.0, 2.0)],
               "locally_periodic": [u(0.5, 2.0), u(0.3, 2.0), u(0.4, 2.0), u(-1.0, 2.0)]}[kernel]
    x1, x2 = x1.to(DEVICE), x2.to(DEVICE)
    start, end = make_ranges(cutoff, x1, x2)
    rhs = torch.randn(n, k, generator=g).to(DEVICE)
    return [x1.expand(batch, m), x2.expand(batch, n), rhs.expand(batch, n, k), torch.stack(columns, dim=-1).to(DEVICE),
            start.expand(batch, -1), end.expand(batch, -1)]


def _operator(kernel, args, variant=None):
    defines = MatmulSingleConfiguration(kernel).make_config(args)
    if variant:
        defines["MATMUL_VARIANT"] = variant
    return load_native("matmul", defines)


def _call(op, args):
    result = op.call(*args)
    return result[0] if isinstance(result, (tuple, list)) else result


def _exact(kernel, args, b):
    x1, x2, rhs, p, start, end = (t[b].double() for t in args)
    out, tolerance = [], []
    for i in range(0, x1.shape[0], 128):
        lo, hi = int(start[i // 128]), int(end[i // 128])
        d = x1[i:i + 128, None] - x2[None, lo:hi]
        exponent = 0.72134752044448170368 * (d / p[0]) ** 2
        phase, cosine = torch.zeros_like(d), torch.ones_like(d)
        if kernel == "spectral":
            cosine = torch.cos(2 * torch.pi * p[1] * d)
            phase += 2.0 ** -20
        elif kernel == "locally_periodic":
            cl, turns = 2.8853900817779268147 / p[1], d / p[2]
            exponent = exponent + cl * torch.sin(torch.pi * turns) ** 2
            phase += 2.0 ** -20 * cl + 2.0 ** -22 * 3.2 * cl * turns.abs()
        K = p[-1] * torch.exp2(-exponent)
        out.append((K * cosine) @ rhs[lo:hi])
        relative = 2.0 ** -19 + 2.0 ** -22 * exponent + phase
        tolerance.append((K.abs() * relative + p[-1].abs() * 2.0 ** -37) @ rhs[lo:hi].abs())
    return torch.cat(out), torch.cat(tolerance)


def _check(kernel, args, text):
    op = _operator(kernel, args)
    assert text in op.describe(*args), op.describe(*args)
    result = _call(op, args).double()
    for b in sorted({0, args[0].shape[0] - 1}):
        exact, tolerance = _exact(kernel, args, b)
        assert ((result[b] - exact).abs() <= tolerance).all(), float(((result[b] - exact).abs() / tolerance).max())


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("m,n,k,batch,density,local", [(1, 2048, 1, 1, 10.0, False), (100, 5001, 3, 1, 10.0, False), (128, 70000, 16, 1, 10.0, False),
                                                       (129, 20000, 17, 2, 10.0, False), (300, 30000, 40, 1, 10.0, False),
                                                       (100, 40000, 8, 1, 700.0, True), (1000, 60000, 2, 8, 3.0, False),
                                                       (200, 9000, 5, 3, 0.5, True)])
def test_shares_against_float64(kernel, m, n, k, batch, density, local):
    _check(kernel, _inputs(kernel, m, n, k, batch, density, local=local), "_shares<" + kernel)


# 800 / 300 / 100 row blocks: two, four, eight wavefronts each
@pytest.mark.parametrize("kernel", ["rbf", "spectral"])
@pytest.mark.parametrize("batch,w", [(40, 2), (15, 4), (5, 8)])
@pytest.mark.parametrize("columns", [300, 700])
def test_rows_far_apart_against_float64(kernel, batch, w, columns):
    _check(kernel, _inputs(kernel, 20 * 128 - 3, 20 * columns, 5, batch), "fwd_grid<%s, G=1, W=%d>" % (kernel, w))


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("what", ["nothing", "rhs inf", "rhs nan", "x2 nan", "x2 inf", "x1 nan", "empty", "reversed"])
def test_values_that_are_not_finite(kernel, what):
    args = [t.clone() for t in _inputs(kernel, 300, 12000, 4, 2)]
    value = float(what.split()[-1]) if what.split()[-1] in ("inf", "nan") else 0.0
    if what.startswith("rhs"):
        args[2][1, 7000, 2] = value
    elif what.startswith("x2"):
        args[1][1, 7000] = value
    elif what.startswith("x1"):
        args[0][1, 130] = value
    elif what == "empty":
        args[5][1, 1] = args[4][1, 1]
    elif what == "reversed":
        args[1], args[2] = args[1].flip(1), args[2].flip(1)
        args[4], args[5] = torch.zeros_like(args[4]), torch.full_like(args[5], 12000)
    op = _operator(kernel, args)
    assert "_shares<" in op.describe(*args)
    got = _call(op, args)
    want = _call(_operator(kernel, args, "mfma_f16_direct" if kernel == "locally_periodic" else "grid"), args)
    assert torch.equal(got.isfinite(), want.isfinite())
    finite = want.isfinite()
    assert torch.allclose(got[finite], want[finite], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("kernel", KERNELS)
def test_without_scratch_and_under_capture(kernel):
    args = _inputs(kernel, 300, 30000, 8, 2)
    op = _operator(kernel, args)
    want = _call(op, args)
    lib = _native.load_library()
    assert lib.km_matmul_workspace_size(_native._kernel_id(kernel), 1, _native._i64((2,)), 300, 30000, 8, None) % (2 * 300 * 8 * 4) == 0
    plain = torch.empty_like(want)
    status = lib.km_matmul(_native._kernel_id(kernel), 1, _native._i64((2,)), 300, 30000, 8, *_native._tensors_args(*args), plain.data_ptr(), None,
                           ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert status == 0
    assert torch.allclose(plain, want, rtol=1e-4, atol=1e-4)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        _call(op, args)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = _call(op, args)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, want)
        torch.randn(100000, device=DEVICE).sum().item()


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("columns", [0, 1, 31, 511, 512, 513, 1024, 5000])
def test_short_ranges_are_one_share(kernel, columns):
    """A range of up to 512 columns is written by one workgroup, and the scratch memory left alone; a longer one is not.
    (Entries below 2^-24 of the output scale: their high half is within fp16's smallest step, 2^-24, their low half within
    2^-11 of that, which shows where a range has hardly any columns.)"""
    args = [t.clone() for t in _inputs(kernel, 200, 20000, 5, 2, local=True)]
    args[4][:], args[5][:] = 37, 37 + columns
    args[4][1, 1], args[5][1, 1] = 100, 300
    lib, head = _native.load_library(), (_native._kernel_id(kernel), 1, _native._i64((2,)), 200, 20000, 5)
    need = lib.km_matmul_workspace_size(*head, None)
    assert need > 0
    scratch = torch.full((need // 4,), float("nan"), device=DEVICE)
    out = torch.full((2, 200, 5), float("nan"), device=DEVICE)
    assert lib.km_matmul_with_workspace(*head, *_native._tensors_args(*args), out.data_ptr(), None, scratch.data_ptr(), need,
                                        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    touched = ~scratch.isnan().view(-1, 2, 200, 5)
    assert not touched[:, 1, 128:].any()
    assert touched[:, 0].any() == (columns > 512) and touched[:, 1, :128].any() == (columns > 512)
    for b in range(2):
        exact, tolerance = _exact(kernel, args, b)
        largest = args[2][b, 37:max(37 + columns, 300)].abs().sum(0).double()
        assert ((out[b].double() - exact).abs() <= tolerance + 2.0 ** -35 * args[3][b, -1].abs() * largest).all()

"""The native calls on tensors against the autograd functions that they stand for: the same launches, so the same bits,
over the forms that both take, and what autograd asks of a node."""
import threading

import pytest
import torch
from torch.utils.checkpoint import checkpoint

from kernel_matmul_amd import _native
from kernel_matmul_amd import linear_operator as lo
from kernel_matmul_amd.linear_operator import KernelMatmulLinearOperator
from kernel_matmul_amd.ranges import make_ranges

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")
COLUMNS = {"rbf": 2, "spectral": 3, "locally_periodic": 4}


def _operator(kernel="spectral", batch=(2,), n=300, m=None, requires_grad=True, seed=0):
    g = torch.Generator().manual_seed(seed)
    x2 = torch.sort(torch.rand(n, generator=g) * 20)[0].to(DEVICE)
    x1 = x2 if m is None else torch.sort(torch.rand(m, generator=g) * 20)[0].to(DEVICE)
    params = (0.5 + torch.rand(*batch, COLUMNS[kernel], generator=g)).to(DEVICE).requires_grad_(requires_grad)
    start, end = make_ranges(4.0, x1, align=True) if m is None else make_ranges(4.0, x1, x2, align=True)
    K = KernelMatmulLinearOperator(x1[:, None], x2[:, None], params, start, end, kernel_type=kernel, symmetric=m is None)
    return K, params, g


def _general(K, rhs):
    """The product through the autograd function."""
    batch = torch.broadcast_shapes(K.shape[:-2], rhs.shape[:-2])
    x1, x2, params, start, end = K._get_args_for_native(batch)
    return lo._MatmulOperator.apply(x1, x2, rhs.expand(*batch, *rhs.shape[-2:]), params, start, end, K._native_matmul,
                                    K._native_matmul_bwd, K._symmetric, K._transposed_ranges)


@pytest.mark.parametrize("kernel", ["rbf", "spectral", "locally_periodic"])
@pytest.mark.parametrize("batch", [(), (1,), (3,), (2, 3)])
@pytest.mark.parametrize("m", [None, 131])
@pytest.mark.parametrize("form", ["dense", "shared", "transposed", "gaps", "more batch"])
def test_products_and_their_gradients(kernel, batch, m, form):
    K, params, g = _operator(kernel, batch, m=m)
    n, k = K.shape[-1], 5
    if form == "more batch":
        rhs = torch.randn(4, *batch, n, k, generator=g)
    elif form == "shared":
        rhs = torch.randn(n, k, generator=g)
    elif form == "transposed":
        rhs = torch.randn(*batch, k, n, generator=g).transpose(-1, -2)
    elif form == "gaps":
        rhs = torch.randn(*batch, 2 * n, 3 * k, generator=g)[..., ::2, ::3]
    else:
        rhs = torch.randn(*batch, n, k, generator=g)
    rhs = rhs.to(DEVICE).requires_grad_()
    out = K @ rhs
    general = _general(_operator(kernel, batch, m=m)[0], rhs)
    assert torch.equal(out, general)
    weights = torch.randn(out.shape, generator=g).to(DEVICE)
    for w in (weights, torch.ones((), device=DEVICE).expand(out.shape), weights.mT.contiguous().mT):
        got = torch.autograd.grad(out, (params, rhs), w, retain_graph=True)
        reference = _operator(kernel, batch, m=m)
        expected = torch.autograd.grad(_general(reference[0], rhs), (reference[1], rhs), w)
        assert all(torch.equal(a, b) for a, b in zip(got, expected))
        (alone,) = torch.autograd.grad(out, (params,), w, retain_graph=True)
        assert torch.equal(alone, got[0])
    with torch.no_grad():
        plain = K @ rhs
    assert torch.equal(plain, out) and not plain.requires_grad


@pytest.mark.parametrize("kernel", ["rbf", "spectral", "locally_periodic"])
@pytest.mark.parametrize("batch", [(), (2, 3)])
def test_matrices_entries_and_bilinear_forms(kernel, batch):
    K, params, g = _operator(kernel, batch, n=150)
    other, other_params, _ = _operator(kernel, batch, n=150)
    call = other._get_args_for_native(other.batch_shape)
    dense = K.to_dense()
    expected = lo._DenseOperator.apply(*call, other._native_dense, other._native_dense_bwd)
    w = torch.randn(dense.shape, generator=g).to(DEVICE)
    assert torch.equal(dense, expected)
    assert torch.equal(*(torch.autograd.grad(d, (p,), w)[0] for d, p in ((dense, params), (expected, other_params))))
    row, col = (torch.randint(150, (40,), generator=g).to(DEVICE) for _ in range(2))
    index = [torch.randint(s, (40,), generator=g).to(DEVICE) for s in batch]
    for got, r, c, b in ((K._get_indices(row, col, *index), row, col, index), (K.diagonal(), None, None, None)):
        if r is None:
            assert torch.equal(got, torch.diagonal(dense, dim1=-2, dim2=-1))
            r = c = torch.arange(150, device=DEVICE).expand(got.shape)
            b = [torch.arange(s, device=DEVICE).view([-1 if i == d else 1 for i in range(got.dim())]).expand(got.shape)
                 for d, s in enumerate(batch)]
        expected = lo._IndexOperator.apply(*call, other._native_index, other._native_index_bwd, r.int(), c.int(), *(t.int() for t in b))
        assert torch.equal(got, expected)
        w = torch.randn(got.shape, generator=g).to(DEVICE)
        assert torch.equal(*(torch.autograd.grad(e, (p,), w)[0] for e, p in ((got, params), (expected, other_params))))
    left, right = (torch.randn(*batch, 150, 3, generator=g).to(DEVICE) for _ in range(2))
    grad = K._bilinear_derivative(left, right)[2]
    x1, x2, p, start, end = call
    assert torch.equal(grad, other._native_bilinear_derivative(x1, x2, left, right, p, start, end))


def test_what_autograd_asks_of_a_node():
    K, params, g = _operator()
    rhs = torch.randn(2, 300, 4, generator=g).to(DEVICE).requires_grad_()
    expected = torch.autograd.grad((K @ rhs).square().sum(), (params, rhs))
    # saved tensors go through the hooks
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.shape), t.cpu())[1], lambda t: t.to(DEVICE)):
        out = (K @ rhs).square().sum()
    assert torch.Size((2, 300, 4)) in seen and len(seen) >= 6
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(out, (params, rhs)), expected))
    again = checkpoint(lambda p, v: (K @ v).square().sum(), params, rhs, use_reentrant=False)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(again, (params, rhs)), expected))
    # a graph that is used up, and inputs that changed
    out = (K @ rhs).sum()
    out.backward()
    with pytest.raises(RuntimeError, match="second time"):
        out.backward()
    out = K @ rhs
    with torch.no_grad():
        rhs.mul_(2.0)
    with pytest.raises(RuntimeError, match="inplace"):
        out.sum().backward()
    # a gradient that is a negated view
    z = torch.complex(torch.zeros_like(K @ rhs), K @ rhs)
    (grad,) = torch.autograd.grad(z.conj().imag.sum(), (params,))
    (positive,) = torch.autograd.grad((K @ rhs).sum(), (params,))
    torch.testing.assert_close(grad, -positive)
    with torch.inference_mode():
        assert (K @ rhs).is_inference()


def test_an_operators_own_native_function_is_called():
    K, params, g = _operator(requires_grad=False)
    rhs = torch.randn(2, 300, 4, generator=g).to(DEVICE)
    expected = K @ rhs
    function, calls = K._native_matmul, []
    K._native_matmul = lambda *args: (calls.append(1), function(*args))[1]
    assert torch.equal(K @ rhs, expected) and calls == [1]


def test_streams_and_threads():
    K, params, g = _operator()
    rhs = torch.randn(2, 300, 4, generator=g).to(DEVICE).requires_grad_()
    expected = [K @ rhs, *torch.autograd.grad((K @ rhs).sum(), (params, rhs))]
    torch.cuda.synchronize()
    results = {}

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                out = K @ rhs
                grads = torch.autograd.grad(out.sum(), (params, rhs))
            stream.synchronize()
            results[i] = [out, *grads]

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(results) == 4 and all(torch.equal(a, b) for r in results.values() for a, b in zip(r, expected))


@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("batch", [(), (3,), (2, 2)])
@pytest.mark.parametrize("kind", ["plain", "unsorted", "strided", "nan", "double"])
@pytest.mark.parametrize("align", [False, True])
def test_ranges(two, batch, kind, align):
    g = torch.Generator().manual_seed(4)
    x1, x2 = (torch.sort(torch.rand(*batch, n, generator=g) * 30)[0] for n in (500, 700))
    if kind == "unsorted":
        x1[..., 3] = 1000.0
    elif kind == "nan":
        x1[..., 499] = float("nan")
    elif kind == "double":
        x1, x2 = x1.double(), x2.double()
    expected = make_ranges(2.0, x1.float(), x2.float() if two else None, align=align)
    if kind == "strided":
        x1 = x1.repeat_interleave(2, -1)[..., ::2]
    if kind == "double":
        with pytest.raises(RuntimeError, match="expected scalar type Float"):
            make_ranges(2.0, x1.to(DEVICE), x2.to(DEVICE) if two else None, align=align)
        return
    for cutoff in (2.0, 2):
        got = make_ranges(cutoff, x1.to(DEVICE), x2.to(DEVICE) if two else None, align=align)
        assert all(torch.equal(a.cpu(), b) and a.is_cuda for a, b in zip(got, expected))


def test_refused_ranges_leave_no_launch_behind():
    """The order check writes to host memory that goes back to its pool: a builder that refuses the block size behind it
    waits for it."""
    x = torch.arange(200.0, device=DEVICE)
    make_ranges(2.0, x)
    torch.cuda._sleep(200_000_000)
    with pytest.raises(RuntimeError, match="sizes out of range"):
        make_ranges(2.0, x, block_size=2 ** 31 - 1)
    assert torch.cuda.current_stream().query()


@pytest.mark.parametrize("k", [5, 16, 31, 32, 33, 48, 63, 64, 65, 80])
@pytest.mark.parametrize("offset", [0, 1, 16])
def test_results_are_written_where_they_are_asked_for(k, offset):
    """The way of the stores depends on the width of the rows and on where the result begins."""
    K, _, g = _operator("rbf", (3,), n=3000, requires_grad=False)
    x1, x2, params, start, end = K._get_args_for_native((3,))
    args = (x1, x2, torch.randn(3, 3000, k, generator=g).to(DEVICE), params, start, end)
    assert "fwd_grid" in _native.describe_matmul("rbf", 3, 3000, 3000, k)
    memory = torch.full((offset + 3 * 3000 * k + 64,), float("nan"), device=DEVICE)
    out = _native.matmul("rbf", *args, out=memory[offset:offset + 3 * 3000 * k].view(3, 3000, k))
    assert torch.equal(out, _native.matmul("rbf", *args))
    assert memory[:offset].isnan().all() and memory[offset + 3 * 3000 * k:].isnan().all()
    exact = torch.stack([_native.dense("rbf", *(t[b] for t in (x1, x2, params, start, end))).double() @ args[2][b].double() for b in range(3)])
    assert float((out.double() - exact).norm() / exact.norm()) < 4e-6  # (two fp16 halves of either factor, and the entries' own)

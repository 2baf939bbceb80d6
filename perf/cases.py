"""The work that users of the framework have it do, as cases that can be timed and compared.

A case is a dict of plain values.  Coordinates are sorted points on a line, ``density`` of them per
unit on average (``grid``: "uniform" draws, or "gaps" for cumulative sums of exponential gaps, which
is what irregular sampling in time looks like); hyper-parameters are those of the benchmark
configurations (lengthscales of half a unit to two units, frequencies below half a revolution per
unit, output scales around one), one set per batch item; the sparsity pattern is the one that
``make_ranges`` builds for a cutoff of ``cutoff`` times the largest lengthscale.

``op`` says what one pass is:

forward    ``K @ rhs`` on a ``KernelMatmulLinearOperator`` (square, symmetric pattern): one product of
           a conjugate-gradient solve.  ``shared``: all batch items (hyper-parameter sets) get the
           same right-hand side; otherwise each has its own.  ``contraction`` "mfma_f32" is the
           option to have every product of the contraction in fp32, through ``NativeFunction``'s
           module.
predict    ``K(test, train) @ weights`` at new points: pattern, operator and product; rectangular, and
           the ends of the pattern fall anywhere.
train      forward and backward through autograd: the gradients with respect to the
           hyper-parameters and to the right-hand side, a fresh operator in each pass as in a fit.
bilinear   ``_bilinear_derivative``: the hyper-parameter gradient of a likelihood from solves and
           probe vectors.
dense      ``to_dense()``, its backward, and ``diagonal()``: what predictive variances are made of.
"""
from __future__ import annotations

import math

import torch

from kernel_matmul_amd.compile import load_native
from kernel_matmul_amd.configurations import MatmulSingleConfiguration
from kernel_matmul_amd.linear_operator import KernelMatmulLinearOperator
from kernel_matmul_amd.ranges import make_ranges

_BLOCK = 128


def _case(name, op, kernel, n, k, batch, density, cutoff, m=0, grid="uniform", shared=False, contraction="auto"):
    case = dict(op=op, kernel=kernel, n=n, k=k, batch=batch, density=density, cutoff=cutoff, m=m, grid=grid,
                shared=shared, contraction=contraction)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # The smallest call of a solver: one right-hand side, a few thousand points (the sizes and
        # density of the first benchmark configuration); launches and latency are what it costs.
        _case("small_solve", "forward", "rbf", 4096, 1, 0, 41.0, 8.0),
        # A solve for a handful of hyper-parameter sets at medium size, every set with right-hand
        # sides of its own (the second configuration).
        _case("medium_solve", "forward", "spectral", 20_000, 16, 4, 10.0, 6.0),
        # The headline: one product with 16 columns for eight hyper-parameter sets.
        _case("headline", "forward", "spectral", 100_000, 16, 8, 10.0, 6.0, shared=True),
        # The same size with every product of the contraction in fp32, an option of the operator.
        _case("headline_fp32", "forward", "spectral", 100_000, 16, 8, 10.0, 6.0, shared=True, contraction="mfma_f32"),
        # A million points, 32 columns, eight sets: the largest call (the fifth configuration).
        _case("million", "forward", "spectral", 1_000_000, 32, 8, 10.0, 5.0, shared=True),
        # The recipe of the reference's own benchmark: one rbf matrix, 64 columns, wide windows.
        _case("wide_rhs", "forward", "rbf", 65_536, 64, 1, 24.0, 10.0),
        # Quasi-periodic signals: the third kernel function, at a ragged size.
        _case("periodic", "forward", "locally_periodic", 50_021, 16, 8, 10.0, 6.0),
        # A training step on irregularly sampled data: both gradients (the third configuration).
        _case("train_irregular", "train", "spectral", 50_000, 8, 2, 1.0, 6.0, grid="gaps"),
        # The likelihood's gradient for 16 sets from 4 vectors (the fourth configuration).
        _case("likelihood_grad", "bilinear", "spectral", 100_000, 4, 16, 10.0, 6.0, shared=True),
        # The fit of the reference's example: 7200 dense points, a likelihood gradient from the
        # targets and ten probe vectors.
        _case("fit_grad", "bilinear", "spectral", 7200, 11, 0, 720.0, 3.9),
        # Predictions at new points: a rectangular product of odd sizes with few columns, and all
        # that a call with new points brings with it.
        _case("predict", "predict", "rbf", 50_000, 3, 4, 10.0, 5.0, m=9973),
        # Dense columns of a small matrix and the gradient through them.
        _case("dense_columns", "dense", "spectral", 7200, 0, 0, 20.0, 4.0),
    ]


# The largest drawn case costs no more than the largest listed one.
_MOST_WORK = 1_000_000 * 8 * 200 * (16 + 32)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        op = rng.choice(["forward", "forward", "forward", "predict", "train", "bilinear", "dense"])
        kernel = rng.choice(["rbf", "spectral", "spectral", "locally_periodic"])
        density = round(math.exp(rng.uniform(math.log(1.0), math.log(720.0))), 2)
        cutoff = round(rng.uniform(3.5, 10.0), 2)
        grid = rng.choice(["uniform", "uniform", "gaps"])
        batch = rng.choice([0, 1, 2, 3, 4, 6, 8, 16])
        n = _log_int(rng, 1000, 1_000_000)
        k, m, shared, contraction = 0, 0, False, "auto"
        if op == "forward":
            k = rng.choice([1, 2, 5, 8, 11, 16, 16, 24, 32, 40, 64])
            shared = rng.random() < 0.3
            contraction = "mfma_f32" if rng.random() < 0.15 else "auto"
        elif op == "predict":
            k, m = rng.choice([1, 1, 3, 7]), _log_int(rng, 100, n)
        elif op == "train":
            k = rng.choice([1, 4, 8, 11, 16])
        elif op == "bilinear":
            k, shared = rng.choice([1, 4, 5, 8, 11, 16, 20]), rng.random() < 0.5
        elif op == "dense":
            n, batch = _log_int(rng, 500, 12_000), min(batch, 2)
        case = _case("", op, kernel, n, k, batch, density, cutoff, m, grid, shared, contraction)
        # train runs three products' worth of work, gradients touch two vectors per entry
        passes = {"train": 3, "bilinear": 2}.get(op, 1)
        # (entries in the pattern, right-hand side and result values)
        if passes * _pairs(case, whole_blocks=True) * (16 + k) > _MOST_WORK:
            continue
        if max(batch, 1) * n * max(k, 1) > 100_000_000:
            continue
        return case


def _cutoff(case):
    return case["cutoff"] * (1.0 if case["batch"] < 2 else 2.0)  # distance: times the largest lengthscale


def _pairs(case, whole_blocks=False):
    """Entries of the matrix within the cutoff; whole_blocks: as many as the block-wise pattern has."""
    rows = case["m"] or case["n"]
    width = 2 * _cutoff(case) * case["density"] + (2 * _BLOCK if whole_blocks else 0)
    return max(case["batch"], 1) * rows * min(width, case["n"])


_PARAMS = {"rbf": 2, "spectral": 3, "locally_periodic": 4}


def _points(case, count, extent, u):
    if case["grid"] == "gaps":
        x = torch.cumsum(-torch.log1p(-u[:count].double()), dim=0)
        return (x * (extent / max(float(x[-1]), 1e-9))).float()
    return torch.sort(u[:count] * extent)[0]


def prepare(case, seed):
    g = torch.Generator().manual_seed(seed)
    n, k, batch, m = case["n"], case["k"], case["batch"], case["m"]
    bshape = (batch,) if batch else ()
    extent = n / case["density"]
    device = torch.device("cuda")
    x_host = _points(case, n, extent, torch.rand(n, generator=g))
    x = x_host.to(device)

    def u(lo, hi):
        return lo + (hi - lo) * torch.rand(bshape, generator=g)

    # One set (no batch): lengthscale one, so that the cutoff is what the case says; several:
    # spread over half a unit to two units, the largest two.
    if batch >= 2:
        lengthscale = u(0.5, 2.0)
        lengthscale[0] = 2.0
    else:
        lengthscale = torch.ones(bshape)
    columns = {
        "rbf": lambda: [lengthscale, u(0.5, 2.0)],
        "spectral": lambda: [lengthscale, u(0.05, 0.5), u(0.5, 2.0)],
        "locally_periodic": lambda: [lengthscale, u(0.5, 2.0), u(0.5, 2.0), u(0.5, 2.0)],
    }[case["kernel"]]()
    params = torch.stack(columns, dim=-1).to(device)
    state = {"case": case, "params": params, "x": x[:, None]}
    gd = torch.Generator(device=device).manual_seed(seed)

    def vectors(rows, columns_, shared):
        shape = (rows, columns_) if shared else (*bshape, rows, columns_)
        return torch.randn(shape, generator=gd, device=device)

    op = case["op"]
    if op == "predict":
        x1 = _points(case, m, extent, torch.rand(max(m, 1), generator=g)).to(device)
        state["x1"], state["rhs"] = x1[:, None], vectors(n, k, False)
        return state

    start, end = make_ranges(_cutoff(case), x)
    state["start"], state["end"] = start, end
    if op == "train":
        state["params"].requires_grad_(True)
        # The loss's gradient correlates with the vectors that the product was taken of.
        rhs = vectors(n, k, False)
        state["grad_out"] = 0.5 * rhs + 0.1 * vectors(n, k, False)
        state["rhs"] = rhs.requires_grad_(True)
        return state
    if op == "dense":
        state["params"].requires_grad_(True)
        state["grad_out"] = torch.randn(*bshape, n, n, generator=gd, device=device)
    state["K"] = KernelMatmulLinearOperator(x[:, None], x[:, None], state["params"], start, end,
                                            kernel_type=case["kernel"], symmetric=True)
    if op == "forward":
        state["rhs"] = vectors(n, k, case["shared"])
        if case["contraction"] != "auto":
            # The module of a define set, called on stride-0 views of the batch shape.
            rhs = state["rhs"].expand(*bshape, n, k)
            args = (x.expand(*bshape, n), x.expand(*bshape, n), rhs, params, start.expand(*bshape, -1),
                    end.expand(*bshape, -1))
            defines = dict(MatmulSingleConfiguration(case["kernel"]).make_config(args))
            defines["MATMUL_VARIANT"] = case["contraction"]
            state["native"], state["args"] = load_native("matmul", defines), args
    elif op == "bilinear":
        # The vectors of a likelihood's gradient: one term alpha^T dK alpha of the solve for the
        # targets with itself, and probe vectors z with their solves A^-1 z; the solves are the
        # vectors damped, so the two sides correlate as they do in a fit.
        probes = vectors(n, k, case["shared"])
        solves = 0.5 * probes + 0.1 * vectors(n, k, case["shared"])
        state["left"], state["right"] = solves, probes
    return state


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "forward":
        if "native" in state:
            return state["native"].call(*state["args"])
        return state["K"] @ state["rhs"]
    if op == "predict":
        start, end = make_ranges(_cutoff(case), state["x1"][:, 0], state["x"][:, 0])
        K = KernelMatmulLinearOperator(state["x1"], state["x"], state["params"], start, end,
                                       kernel_type=case["kernel"], symmetric=False)
        return K @ state["rhs"]
    if op == "train":
        params, rhs = state["params"], state["rhs"]
        K = KernelMatmulLinearOperator(state["x"], state["x"], params, state["start"], state["end"],
                                       kernel_type=case["kernel"], symmetric=True)
        out = K @ rhs
        grad_params, grad_rhs = torch.autograd.grad(out, (params, rhs), state["grad_out"])
        return out.detach(), grad_params, grad_rhs
    if op == "bilinear":
        return state["K"]._bilinear_derivative(state["left"], state["right"])[2]
    # dense
    dense = state["K"].to_dense()
    (grad_params,) = torch.autograd.grad(dense, (state["params"],), state["grad_out"])
    return dense.detach(), grad_params, state["K"].diagonal().detach()


def work(case):
    """Bytes: every input read once, every result written once.  Flops: the product's (or the
    coefficients') multiply-adds of the entries within the cutoff."""
    n, k, m, items = case["n"], case["k"], case["m"] or case["n"], max(case["batch"], 1)
    blocks = -(-m // _BLOCK)
    params = items * _PARAMS[case["kernel"]]
    inputs = n + params + 2 * blocks
    vectors = items * n * k
    op = case["op"]
    if op == "forward":
        values, flops = inputs + (n * k if case["shared"] else vectors) + vectors, 2 * _pairs(case) * k
    elif op == "predict":
        values, flops = inputs + m + vectors + items * m * k, 2 * _pairs(case) * k
    elif op == "train":
        values, flops = inputs + 4 * vectors + params, 6 * _pairs(case) * k
    elif op == "bilinear":
        values, flops = inputs + 2 * (n * k if case["shared"] else vectors) + params, 2 * _pairs(case) * k
    else:
        # the whole matrix is written; of the gradient the entries within the cutoff are read
        values, flops = inputs + items * n * n + _pairs(case) + items * n + params, 0
    return {"bytes": 4 * int(values), "flops": int(flops)}


def tolerance(case):
    """Four times the largest distance from a float64 evaluation over the listed and ninety drawn
    cases (2-norm of a whole result; largest element over the result's root mean square)."""
    if case["op"] == "bilinear":
        return {"rel": 2e-6, "max": 5e-5}
    if case["op"] == "dense":  # random weights: the gradient's terms cancel
        return {"rel": 1e-5, "max": 5e-5}
    return {"rel": 4e-6, "max": 5e-5}

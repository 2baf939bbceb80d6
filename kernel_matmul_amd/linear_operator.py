"""LinearOperator over the on-the-fly kernel matrix and the autograd wiring of the native ops.

Mirrors kernel_matmul/linear_operator.py:22-289 of the reference: same constructor, same
batch broadcasting (stride-0 ``expand`` views, no copies), same hooks
(``_matmul``, ``_size``, ``_transpose_nonbatch``, ``to_dense``, ``_expand_batch``, ``to``,
``type``, ``_bilinear_derivative``, ``_get_indices``).

The ``linear_operator`` package is optional.  When it is installed the class derives from
``linear_operator.LinearOperator`` and plugs into GPyTorch's solvers; when it is not, a small
stand-in base supplies ``shape``/``size``/``matmul``/``@``/``transpose``/``diagonal`` so that
the operator remains usable (and testable) on its own.

Two additions over the reference: the backward of ``matmul`` also returns the gradient with
respect to ``rhs`` (``K^T @ grad`` through the same forward kernel on the transposed
pattern), and ``_IndexOperator.backward`` unpacks its saved tensors correctly for batched
operators (the reference slices ``[:8]`` into 7 names, linear_operator.py:71).
"""
from __future__ import annotations

import multiprocessing.pool
from typing import List, Tuple

import torch
import torch.autograd.forward_ad as forward_ad
from torch import Size, Tensor, dtype

from kernel_matmul_amd import _native, ranges
from kernel_matmul_amd.configurations import (
    BilinearDerivativeConfiguration,
    DenseBwdConfiguration,
    DenseConfiguration,
    IndexBwdConfiguration,
    IndexConfiguration,
    MatmulAutotuneConfiguration,
    MatmulBwdConfiguration,
)
from kernel_matmul_amd.native_function import NativeFunction

try:  # pragma: no cover - depends on the environment
    from linear_operator import LinearOperator
    from linear_operator.utils.generic import _to_helper

    HAVE_LINEAR_OPERATOR = True
except ImportError:
    HAVE_LINEAR_OPERATOR = False

    class LinearOperator:  # type: ignore[no-redef]
        """Minimal stand-in used when the ``linear_operator`` package is absent."""

        def __init__(self, *args, **kwargs):
            self._args = args
            self._kwargs = kwargs

        @property
        def shape(self) -> Size:
            return self._size()

        def size(self, dim: int | None = None):
            return self.shape if dim is None else self.shape[dim]

        def dim(self) -> int:
            return len(self.shape)

        @property
        def batch_shape(self) -> Size:
            return self.shape[:-2]

        @property
        def device(self):
            return self._args[0].device

        @property
        def dtype(self):
            return self._args[0].dtype

        def matmul(self, other: Tensor) -> Tensor:
            if other.dim() == 1:
                return self._matmul(other.unsqueeze(-1)).squeeze(-1)
            return self._matmul(other)

        __matmul__ = matmul

        def transpose(self, dim1: int, dim2: int):
            ndim = self.dim()
            if {dim1 % ndim, dim2 % ndim} != {ndim - 2, ndim - 1}:
                raise NotImplementedError("only the two matrix dimensions can be transposed")
            return self._transpose_nonbatch()

        @property
        def mT(self):
            return self._transpose_nonbatch()

        def expand(self, *sizes):
            if len(sizes) == 1 and not isinstance(sizes[0], int):
                sizes = tuple(sizes[0])
            return self._expand_batch(Size(sizes[:-2]))

        def diagonal(self) -> Tensor:
            if hasattr(self, "_diagonal"):
                return self._diagonal()
            n = min(self.shape[-2], self.shape[-1])
            index = torch.arange(n, device=self.device)
            batch = torch.meshgrid(
                *(torch.arange(s, device=self.device) for s in self.batch_shape), index, indexing="ij"
            )
            return self._get_indices(batch[-1], batch[-1], *batch[:-1])

        def to(self, *args, **kwargs):
            return self

        def type(self, dtype):
            return self

    def _to_helper(*args, **kwargs):
        device = kwargs.get("device")
        dtype_ = kwargs.get("dtype")
        for arg in args:
            if isinstance(arg, torch.dtype):
                dtype_ = arg
            elif isinstance(arg, (str, torch.device)):
                device = torch.device(arg)
        return device, dtype_


def _recorded(differentiable: tuple) -> bool:
    if torch.is_grad_enabled():
        for t in differentiable:
            if t.requires_grad:
                return True
    return False


def _transformed() -> bool:
    return not (
        forward_ad._current_level < 0  # (no dual tensors)
        and not torch._C._are_functorch_transforms_active()
        and torch._C._get_tracing_state() is None
        and not torch.compiler.is_compiling()
    )


def _plain(differentiable: tuple) -> bool:
    """Whether nothing records or transforms a call on these tensors, so that the native function can be called
    itself.  A call that is recorded but not transformed has a native node (csrc/km_torch.cpp); every other one goes
    through the autograd functions below."""
    return not _recorded(differentiable) and not _transformed()


class _MatmulOperator(torch.autograd.Function):
    """K @ rhs with gradients for the hyper-parameters (matmul_bwd) and for rhs (K^T @ grad)."""

    @staticmethod
    def forward(ctx, x1, x2, rhs, params, start, end, native_matmul, native_matmul_bwd, symmetric=False,
                transposed_ranges=None):
        ctx.save_for_backward(x1, x2, rhs, params, start, end)
        ctx.native_matmul = native_matmul
        ctx.native_matmul_bwd = native_matmul_bwd
        ctx.symmetric = symmetric
        ctx.transposed_ranges = transposed_ranges  # callable returning (start_t, end_t), or None
        return native_matmul(x1, x2, rhs, params, start, end)

    @staticmethod
    def backward(ctx, grad_output):
        x1, x2, rhs, params, start, end = ctx.saved_tensors
        grad_params = None
        grad_rhs = None
        if ctx.needs_input_grad[3]:
            grad_params = ctx.native_matmul_bwd(x1, x2, rhs, params, start, end, grad_output)
        if ctx.needs_input_grad[2]:
            if ctx.symmetric:
                start_t, end_t = start, end
            else:
                try:
                    if ctx.transposed_ranges is not None:
                        start_t, end_t = ctx.transposed_ranges(start.shape[:-1])
                    else:
                        start_t, end_t = ranges.transpose_ranges(start, end, x1.shape[-1], x2.shape[-1])
                except ValueError as error:
                    raise RuntimeError(
                        "the gradient with respect to rhs needs the transposed sparsity pattern; "
                        "build the ranges with align=True"
                    ) from error
            grad_rhs = ctx.native_matmul(x2, x1, grad_output, params, start_t, end_t)
        return None, None, grad_rhs, grad_params, None, None, None, None, None, None


class _DenseOperator(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x1, x2, params, start, end, native_dense, native_dense_bwd):
        ctx.save_for_backward(x1, x2, params, start, end)
        ctx.native_dense_bwd = native_dense_bwd
        return native_dense(x1, x2, params, start, end)

    @staticmethod
    def backward(ctx, grad_output):
        x1, x2, params, start, end = ctx.saved_tensors
        grad = ctx.native_dense_bwd(x1, x2, params, start, end, grad_output)
        return None, None, grad, None, None, None, None


class _IndexOperator(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x1, x2, params, start, end, native_index, native_index_bwd, row_index,
                col_index, *batch_indices):
        ctx.save_for_backward(x1, x2, params, start, end, row_index, col_index, *batch_indices)
        ctx.native_index_bwd = native_index_bwd
        return native_index(x1, x2, params, start, end, batch_indices, row_index, col_index)

    @staticmethod
    def backward(ctx, grad_output):
        x1, x2, params, start, end, row_index, col_index = ctx.saved_tensors[:7]
        batch_indices = ctx.saved_tensors[7:]
        grad = ctx.native_index_bwd(
            x1, x2, params, start, end, batch_indices, row_index, col_index, grad_output
        )
        return (None, None, grad, None, None, None, None, None, None, *[None for _ in batch_indices])


def _widen(t: Tensor, batch_shape: Size, trailing: int) -> Tensor:
    """``t`` as a stride-0 view of the batch shape (itself where it has it)."""
    if t.shape[:-trailing] == batch_shape:
        return t
    return t.expand(*batch_shape, *t.shape[-trailing:])


class _Native:
    """A native function of the operator's kernel type, made when it is first used (a fit makes an operator for
    every set of hyper-parameters and uses one or two)."""

    def __init__(self, op: str, configuration, autotuned: bool = False):
        self._op = op
        self._configuration = configuration
        self._autotuned = autotuned

    def __set_name__(self, owner, name):
        self._name = name

    def __get__(self, operator, owner=None):
        if operator is None:
            return self
        pool = {"compile_pool": operator._compile_pool} if self._autotuned else {}
        function = NativeFunction(self._op, self._configuration(operator._kernel_type), **pool)
        operator.__dict__[self._name] = operator._made[self._name] = function
        return function


class KernelMatmulLinearOperator(LinearOperator):
    """The (masked) kernel matrix K(x1, x2) of shape (..., M, N), never materialised.

    Args:
        x1: inputs of shape (..., M, 1), sorted along M.
        x2: inputs of shape (..., N, 1), sorted along N.
        params: kernel hyper-parameters of shape (..., P).
        start, end: sparsity pattern of shape (..., ceil(M / 128)), see ``ranges.make_ranges``.
        kernel_type: "rbf", "spectral" or "locally_periodic" (required).
        symmetric: whether K equals its transpose; determined from ``x1 == x2`` if omitted.
        compile_pool: accepted for compatibility; nothing is compiled at run time.
    """

    _native_matmul = _Native("matmul", MatmulAutotuneConfiguration, autotuned=True)
    _native_matmul_bwd = _Native("matmul_bwd", MatmulBwdConfiguration)
    _native_bilinear_derivative = _Native("bilinear_derivative", BilinearDerivativeConfiguration)
    _native_index = _Native("index", IndexConfiguration)
    _native_index_bwd = _Native("index_bwd", IndexBwdConfiguration)
    _native_dense = _Native("dense", DenseConfiguration)
    _native_dense_bwd = _Native("dense_bwd", DenseBwdConfiguration)

    def __init__(
        self,
        x1: Tensor,
        x2: Tensor,
        params: Tensor,
        start: Tensor,
        end: Tensor,
        kernel_type: str | None = None,
        symmetric: bool | None = None,
        compile_pool: multiprocessing.pool.Pool | None = None,
    ):
        super().__init__(
            x1, x2, params, start, end,
            kernel_type=kernel_type, symmetric=symmetric, compile_pool=compile_pool,
        )
        if kernel_type is None:
            raise ValueError("kernel_type must be specified")
        if x1.dim() < 2 or x2.dim() < 2 or x1.size(-1) != 1 or x2.size(-1) != 1:
            raise ValueError("x1 and x2 must have shapes (..., M, 1) and (..., N, 1), respectively")
        if symmetric is None:
            symmetric = torch.equal(x1, x2)

        self._given = (x1, x2, params, start, end)
        shapes = (x1.shape[:-2], x2.shape[:-2], params.shape[:-1], start.shape[:-1], end.shape[:-1])
        distinct = set(shapes) - {Size(())}
        if len(distinct) > 1:
            batch_shape = torch.broadcast_shapes(*shapes)
        else:  # (the usual case, at a tenth of the time)
            batch_shape = distinct.pop() if distinct else Size(())
        self._kernel_type = kernel_type
        self._kernel_number = _native.KERNEL_TYPES.get(kernel_type)
        self._compile_pool = compile_pool
        self._batch_shape = batch_shape
        self._symmetric = symmetric
        self._ranges_t = None  # pattern of the transpose, built on first use
        self._diagonal_indices = None  # index tensors of the diagonal, built on first use
        self._native_args = None  # (batch shape, widened constructor tensors) of the last call
        self._made = {}  # the native functions made so far (_Native)

    # -- helpers -------------------------------------------------------------------------
    # The constructor tensors as stride-0 views of the batch shape.
    _x1 = property(lambda self: _widen(self._given[0], self._batch_shape, 2))
    _x2 = property(lambda self: _widen(self._given[1], self._batch_shape, 2))
    _params = property(lambda self: _widen(self._given[2], self._batch_shape, 1))
    _start = property(lambda self: _widen(self._given[3], self._batch_shape, 1))
    _end = property(lambda self: _widen(self._given[4], self._batch_shape, 1))

    def _calls(self, *functions: str):
        """The native module of calls on tensors, if nothing asks for the native functions of these names: they are
        the operator's own and nobody has taken them in hand, and their modules would watch no call."""
        for name in functions:
            if (self.__dict__.get(name, self) is not self._made.get(name, self)
                    or getattr(type(self), name) is not KernelMatmulLinearOperator.__dict__[name]):
                return None
        calls = _native.torch_calls()
        return None if calls.watched() else calls

    def _get_args_for_native(self, batch_shape) -> tuple[Tensor, Tensor, Tensor, Tensor, Tensor]:
        """The constructor tensors as stride-0 views of ``batch_shape``.  The views of the tensors
        that carry no gradient (coordinates and pattern) are kept for the last shape asked for:
        solvers call with the same one over and over.  ``params`` is widened on every call, so
        the view belongs to the autograd mode of that call (a view made under ``no_grad`` or
        ``inference_mode`` would cut later calls off from the hyper-parameters' gradient)."""
        batch_shape = Size(batch_shape)
        if self._native_args is None or self._native_args[0] != batch_shape:
            x1, x2, _, start, end = self._given
            self._native_args = (batch_shape, _native.torch_calls().views(x1, x2, start, end, tuple(batch_shape)))
        x1, x2, start, end = self._native_args[1]
        return x1, x2, _widen(self._given[2], batch_shape, 1), start, end

    def _transposed_ranges(self, batch_shape=None) -> tuple[Tensor, Tensor]:
        """Pattern of K^T, computed once per operator (the check that the pattern is block
        aligned and the host pass both synchronise with the device); optionally widened to
        ``batch_shape`` as stride-0 views."""
        if self._ranges_t is None:
            self._ranges_t = ranges.transpose_ranges(
                self._start, self._end, self._x1.size(-2), self._x2.size(-2)
            )
        start_t, end_t = self._ranges_t
        if batch_shape is not None:
            start_t = start_t.expand(*batch_shape, start_t.shape[-1])
            end_t = end_t.expand(*batch_shape, end_t.shape[-1])
        return start_t, end_t

    # -- LinearOperator hooks ------------------------------------------------------------
    def _matmul(self, rhs: Tensor) -> Tensor:
        columns = self._given[1].size(-2)
        if rhs.shape[:-2] == self._batch_shape and rhs.size(-2) == columns:
            batch_shape, rhs_ = self._batch_shape, rhs  # nothing to broadcast
        else:
            expected = Size((*self._batch_shape, columns, rhs.size(-1)))
            broadcast = torch.broadcast_shapes(expected, rhs.shape)
            batch_shape = broadcast[:-2]
            rhs_ = rhs.expand(*broadcast)
        x1, x2, params, start, end = self._get_args_for_native(batch_shape)
        call = (x1, x2, rhs_, params, start, end)
        recorded, transformed = _recorded((rhs_, params)), _transformed()
        # (the transposed pattern of one that is not symmetric is the autograd function's to find)
        if not transformed and (not recorded or self._symmetric or not rhs_.requires_grad):
            calls = self._calls("_native_matmul", "_native_matmul_bwd")
            if calls is not None:
                out = calls.matmul_recorded(self._kernel_number, *call)
                if out is not None:
                    return out
        native = self._native_matmul
        if not recorded and not transformed:
            return native(*call)
        return _MatmulOperator.apply(*call, native, self._native_matmul_bwd, self._symmetric, self._transposed_ranges)

    def _size(self) -> Size:
        return Size((*self._batch_shape, self._given[0].size(-2), self._given[1].size(-2)))

    def _transpose_nonbatch(self) -> "KernelMatmulLinearOperator":
        if self._symmetric:
            return self
        start_t, end_t = self._transposed_ranges()
        return KernelMatmulLinearOperator(
            self._x2, self._x1, self._params, start_t, end_t, kernel_type=self._kernel_type
        )

    def to_dense(self) -> Tensor:
        call = self._get_args_for_native(self._batch_shape)
        if not _transformed():
            calls = self._calls("_native_dense", "_native_dense_bwd")
            if calls is not None:
                out = calls.dense_recorded(self._kernel_number, *call)
                if out is not None:
                    return out
        if _plain((call[2],)):
            return self._native_dense(*call)
        return _DenseOperator.apply(*call, self._native_dense, self._native_dense_bwd)

    def _expand_batch(self, batch_shape: Size | List[int]) -> "KernelMatmulLinearOperator":
        return KernelMatmulLinearOperator(
            self._x1.expand(*batch_shape, *self._x1.shape[-2:]),
            self._x2.expand(*batch_shape, *self._x2.shape[-2:]),
            self._params.expand(*batch_shape, self._params.shape[-1]),
            self._start.expand(*batch_shape, self._start.shape[-1]),
            self._end.expand(*batch_shape, self._end.shape[-1]),
            kernel_type=self._kernel_type,
        )

    def to(self, *args, **kwargs):
        device, dtype_ = _to_helper(*args, **kwargs)
        if (device is not None and device.type != "cuda") or (
            dtype_ is not None and dtype_ != torch.float32
        ):
            raise NotImplementedError("KernelMatmulLinearOperator only supports CUDA and float32")
        return super().to(*args, **kwargs)

    def type(self, dtype: dtype):
        if dtype != torch.float32:
            raise NotImplementedError("KernelMatmulLinearOperator only supports CUDA and float32")
        return super().type(dtype)

    def _bilinear_derivative(self, left_vecs: Tensor, right_vecs: Tensor) -> Tuple[Tensor | None, ...]:
        batch_shape = self._batch_shape
        if not left_vecs.shape[:-2] == right_vecs.shape[:-2] == batch_shape:
            batch_shape = torch.broadcast_shapes(
                left_vecs.shape[:-2], right_vecs.shape[:-2], batch_shape
            )
        left_vecs = _widen(left_vecs, batch_shape, 2)
        right_vecs = _widen(right_vecs, batch_shape, 2)
        x1, x2, params, start, end = self._get_args_for_native(batch_shape)
        call = (x1, x2, left_vecs, right_vecs, params, start, end)
        calls = self._calls("_native_bilinear_derivative")
        grad = calls.param_grad(self._kernel_number, *call, None) if calls is not None else None
        if grad is None:
            grad = self._native_bilinear_derivative(*call)
        # one entry per constructor tensor: x1, x2, params, start, end
        return None, None, grad, None, None

    def _diagonal(self) -> Tensor:
        """The diagonal through the index operator, with its index tensors (int32 views that
        repeat one arange per dimension, no copies) built once per operator instead of by the
        base class's ``arange`` / ``meshgrid`` / dtype conversion on every call."""
        if self._diagonal_indices is None:
            n = min(self._x1.shape[-2], self._x2.shape[-2])
            batch_shape = tuple(self._batch_shape)
            device = self._x1.device
            row = torch.arange(n, dtype=torch.int32, device=device).expand(*batch_shape, n)
            batch = []
            for d, size in enumerate(batch_shape):
                view = [1] * (len(batch_shape) + 1)
                view[d] = size
                batch.append(torch.arange(size, dtype=torch.int32, device=device).view(view).expand(*batch_shape, n))
            self._diagonal_indices = (row, tuple(batch))
        row, batch = self._diagonal_indices
        return self._entries(batch, row, row)

    def _entries(self, batch: tuple, row: Tensor, col: Tensor) -> Tensor:
        call = self._get_args_for_native(self._batch_shape)
        if not _transformed():
            calls = self._calls("_native_index", "_native_index_bwd")
            if calls is not None:
                out = calls.index_recorded(self._kernel_number, *call, row, col, batch)
                if out is not None:
                    return out
        if _plain((call[2],)):
            return self._native_index(*call, batch, row, col)
        return _IndexOperator.apply(*call, self._native_index, self._native_index_bwd, row, col, *batch)

    def _get_indices(self, row_index: Tensor, col_index: Tensor, *batch_indices: Tensor) -> Tensor:
        device = self._given[0].device
        shape = torch.broadcast_shapes(
            row_index.shape, col_index.shape, *(b.shape for b in batch_indices)
        )

        def prepare(index: Tensor) -> Tensor:
            return index.expand(*shape).to(device=device, dtype=torch.int32)

        return self._entries(tuple(prepare(b) for b in batch_indices), prepare(row_index), prepare(col_index))

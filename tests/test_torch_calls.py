"""What the native calls on tensors hand back to the general path, which refuses it."""
import pytest
import torch

from kernel_matmul_amd import _native
from kernel_matmul_amd.linear_operator import KernelMatmulLinearOperator


def _args(k=2):
    x = torch.arange(200.0)
    return [x, x, torch.ones(200, k), torch.ones(3), torch.zeros(2).int(), torch.full((2,), 200).int()]


def test_host_tensors_and_other_objects_are_handed_back():
    calls = _native.torch_calls()
    x1, x2, rhs, params, start, end = _args()
    assert calls.matmul(1, x1, x2, rhs, params, start, end, None, None) is None
    assert calls.matmul(None, x1, x2, rhs, params, start, end, None, None) is None
    assert calls.matmul(1, x1, x2, None, params, start, end, None, None) is None
    assert calls.matmul(1, x1, x2) is None
    assert calls.matmul_recorded(1, x1, x2, rhs, params, start, end) is None
    assert calls.param_grad(1, x1, x2, rhs, rhs, params, start, end, None) is None
    assert calls.dense(1, x1, x2, params, start, end) is None and calls.dense_recorded(1, x1, x2, params, start, end) is None
    assert calls.dense_bwd(1, x1, x2, params, start, end, rhs) is None
    assert calls.index(1, x1, x2, params, start, end, start, start, ()) is None
    assert calls.index_bwd(1, x1, x2, params, start, end, start, start, x1, ()) is None
    assert calls.make_ranges(1.0, x1, None, 128, False) is None and calls.make_ranges(1, x1, None, 128, False) is None
    with pytest.raises(RuntimeError, match="x must be a CUDA tensor"):
        _native.matmul("spectral", *_args())
    with pytest.raises(ValueError, match="Unknown kernel type"):
        _native.matmul("square", *_args())


def test_watched_calls_and_own_functions_take_the_general_path(monkeypatch):
    x = torch.zeros(200, 1)
    make = lambda cls=KernelMatmulLinearOperator: cls(x, x, torch.ones(3), torch.zeros(2), torch.zeros(2), kernel_type="spectral",
                                                      symmetric=True)
    K = make()
    assert K._calls("_native_matmul") is not None
    for name in ("KERNEL_MATMUL_COMPILE_DEBUG", "KERNEL_MATMUL_COMPILE_PRINT_SIZE"):
        monkeypatch.setenv(name, "true")
        assert _native.torch_calls().watched() and K._calls("_native_matmul") is None
        monkeypatch.setenv(name, "false")
        assert K._calls("_native_matmul") is not None
    K._native_matmul_bwd = None
    assert K._calls("_native_matmul") is not None and K._calls("_native_matmul", "_native_matmul_bwd") is None

    class Own(KernelMatmulLinearOperator):
        _native_dense = None

    assert make(Own)._calls("_native_dense") is None and make(Own)._calls("_native_matmul") is not None


@pytest.mark.parametrize("number", [-1, 3, 2 ** 32 + 1, 2 ** 70, -2 ** 70])
def test_numbers_that_are_no_kernels_are_handed_back(number):
    calls = _native.torch_calls()
    x1, x2, rhs, params, start, end = _args()
    matrix = (number, x1, x2, params, start, end)
    assert calls.matmul(number, x1, x2, rhs, params, start, end, None, None) is None
    assert calls.matmul_recorded(number, x1, x2, rhs, params, start, end) is None
    assert calls.param_grad(number, x1, x2, rhs, rhs, params, start, end, None) is None
    assert calls.dense(*matrix) is None and calls.dense_recorded(*matrix) is None and calls.dense_bwd(*matrix, rhs) is None
    assert calls.index(*matrix, start, start, ()) is None and calls.index_recorded(*matrix, start, start, ()) is None
    assert calls.index_bwd(*matrix, start, start, x1, ()) is None


@pytest.mark.parametrize("block_size", [0, -1, 2 ** 31, 2 ** 70, -2 ** 70])
def test_block_sizes_that_are_none_are_handed_back(block_size):
    x = torch.arange(200.0)
    assert _native.torch_calls().make_ranges(1.0, x, None, block_size, False) is None
    assert _native.torch_calls().make_ranges(1.0, x, x, block_size, True) is None


def test_native_functions_that_the_operator_made_itself_are_its_own():
    x = torch.zeros(200, 1)
    K = KernelMatmulLinearOperator(x, x, torch.ones(3), torch.zeros(2), torch.zeros(2), kernel_type="spectral", symmetric=True)
    function = K._native_matmul
    assert K._native_matmul is function and K._calls("_native_matmul", "_native_matmul_bwd") is not None
    K._native_matmul = lambda *args: function(*args)
    assert K._calls("_native_matmul") is None
    K._native_matmul = function
    assert K._calls("_native_matmul") is not None

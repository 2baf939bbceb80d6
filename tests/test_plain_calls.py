"""When an operator calls its native function itself: only where nothing records or transforms the call.  Every
other call goes through the autograd function, which records it or refuses it."""
import pytest
import torch
import torch.autograd.forward_ad as forward_ad

from kernel_matmul_amd.linear_operator import KernelMatmulLinearOperator, _plain
from kernel_matmul_amd.native_function import NativeFunction


def test_what_is_plain():
    t, p = torch.ones(3), torch.ones(3, requires_grad=True)
    assert _plain((t, t))
    assert not _plain((t, p)) and not _plain((p, t))
    with torch.no_grad():
        assert _plain((t, p))
    with torch.inference_mode():
        assert _plain((t, p))
    with forward_ad.dual_level():
        assert not _plain((t, t))
        with torch.no_grad():
            assert not _plain((t, p))
    seen = []
    torch.func.vmap(lambda v: (seen.append(_plain((t,))), v)[1])(torch.ones(2, 3))
    torch.func.grad(lambda v: (seen.append(_plain((t,))), v.sum())[1])(t)
    torch.jit.trace(lambda v: (seen.append(_plain((t,))), v + 1)[1], (t,), check_trace=False)
    assert seen == [False, False, False]


@pytest.mark.parametrize("shapes", [
    [(), (), (), (), ()], [(2,), (), (2,), (), ()], [(1,), (), (), (), ()], [(2, 1), (3,), (), (1, 3), ()],
])
def test_batch_shapes_of_the_constructor(shapes):
    b = torch.broadcast_shapes(*shapes)
    x1, x2, params, start, end = (torch.zeros(*s, *t) for s, t in zip(shapes, ((200, 1), (300, 1), (3,), (2,), (2,))))
    K = KernelMatmulLinearOperator(x1, x2, params, start.int(), end.int(), kernel_type="spectral", symmetric=False)
    assert K.shape == (*b, 200, 300)
    assert [tuple(t.shape) for t in K._get_args_for_native(b)] == [(*b, 200), (*b, 300), (*b, 3), (*b, 2), (*b, 2)]
    assert [tuple(t.shape) for t in K._get_args_for_native((4, *b))][2] == (4, *b, 3)


def test_native_functions_are_made_once_per_operator():
    x = torch.zeros(200, 1)
    make = lambda: KernelMatmulLinearOperator(x, x, torch.ones(3), torch.zeros(2), torch.zeros(2), kernel_type="spectral",
                                              symmetric=True)
    K, other = make(), make()
    assert isinstance(K._native_matmul, NativeFunction) and K._native_matmul is K._native_matmul
    assert K._native_matmul is not other._native_matmul and K._native_matmul is not K._native_matmul_bwd
    assert K._native_index.name == "index" and K._native_dense_bwd.name == "dense_bwd"

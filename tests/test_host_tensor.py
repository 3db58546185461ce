"""Host-side tensor construction from numpy arrays (no GPU): the shape, dtype
and values match what the reference's constructor produces from
``data.tolist()`` (src/nanotorch/core.py:79-84), including 0-d arrays,
non-contiguous arrays and a dtype override."""

from __future__ import annotations

import numpy as np
import pytest

import nanotorch_amd as nt


@pytest.mark.parametrize("arr", [
    np.float32(2.5),
    np.full((), 7, np.int64),
    np.arange(5, dtype=np.float64),
    np.arange(12, dtype=np.int32).reshape(3, 4),
    np.arange(24, dtype=np.float32).reshape(2, 3, 4)[:, ::2, 1:].transpose(2, 0, 1),
    np.array([[True, False], [False, True]]),
])
def test_from_numpy_matches_tolist(arr):
    a = np.asarray(arr)
    t = nt.Tensor(a)
    ref = nt.tensor(a.tolist())
    assert t.shape == a.shape == ref.shape
    assert t.numpy().dtype == a.dtype
    assert t.cpu().tolist() == a.tolist()


def test_from_numpy_with_dtype_override():
    a = np.arange(6, dtype=np.int32).reshape(2, 3)
    t = nt.Tensor(a, dtype=nt.float32)
    assert t.dtype == nt.float32 and t.shape == (2, 3)
    assert t.cpu().tolist() == [[0.0, 1.0, 2.0], [3.0, 4.0, 5.0]]


def test_reshape_view_refuses_another_size():
    """The ops' reshape of a gradient, like Tensor.reshape: not a prefix of a
    larger one."""
    from nanotorch_amd.core import reshape_view

    x = nt.Tensor(np.arange(12, dtype=np.float32))
    assert reshape_view(x, (3, 4)).cpu().tolist() == np.arange(12.0).reshape(3, 4).tolist()
    for dims in ((2, 4), (5,), (), (0,), (13,)):
        with pytest.raises(ValueError):
            reshape_view(x, dims)


def test_sizeof_refuses_an_unknown_dtype():
    from nanotorch_amd._data_type import Dtype, sizeof

    assert [sizeof(d) for d in Dtype] == [sizeof(int(d)) for d in Dtype] == [1, 4, 8, 4, 8]
    for bad in (17, "float32", None, []):
        with pytest.raises(ValueError):
            sizeof(bad)


def test_any_true_requires_grad_gets_its_gradient():
    """requires_grad is taken by its truth (the constructor keeps what it was
    given), in the fused backward as everywhere else."""
    from nanotorch_amd.autograd.function import Function
    from nanotorch_amd.core import _run_backward

    class Twice(Function):
        def fused_ok(self):
            return True

        def _backward_into(self, g, needs, targets):
            return [nt.Tensor([2 * v for v in g.tolist()]) if n else None for n in needs]

    for flag in (True, 1, 2, "yes"):
        x = nt.Tensor([1.0], requires_grad=flag)
        _run_backward(Twice(), nt.Tensor([3.0]), (x,))
        assert x.grad is not None and x.grad.tolist() == [6.0], flag
    x = nt.Tensor([1.0])
    _run_backward(Twice(), nt.Tensor([3.0]), (x,))
    assert x.grad is None

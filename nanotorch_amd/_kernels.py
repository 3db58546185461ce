"""Device operations on tensor views: the call surface of the reference's
``_C`` kernels (src/nanotorch/_C.pyi:63-136), implemented over libnt.

Every function takes ``Tensor`` views, checks that they live on the device,
builds ``nt_view`` descriptors and calls one C ABI entry point.  Outputs are
fresh contiguous buffers in the view's logical row-major order, as in the
reference (src/cpp/ops/unary_ops.cu:9-16, binary_ops.cu:10-19).
"""

from __future__ import annotations

import ctypes
import math

from . import _lib
from ._data_type import Dtype
from ._indexing import row_major_strides
from ._storage import Storage
from .cuda import Device


def require_device(*tensors) -> None:
    """Device ops run on the GPU only; host tensors are staging buffers."""
    for t in tensors:
        if t._storage._device != Device.Cuda:
            raise RuntimeError(
                "nanotorch_amd computes on the GPU: move tensors to "
                "device='cuda' (host tensors only hold and transfer data)."
            )


def _check_same_device(*tensors) -> None:
    devs = {t.device for t in tensors}
    if len(devs) > 1:
        raise RuntimeError("Expected all tensors on the same device.")


def view_of(t) -> _lib.NtView:
    s = t._storage
    return _lib.make_view(s.data_ptr(), t._offset, int(s.dtype), t._shape, t._strides)


def flat_view(storage: Storage, shape, offset: int = 0) -> _lib.NtView:
    return _lib.make_view(
        storage.data_ptr(), offset, int(storage.dtype), tuple(shape), row_major_strides(shape)
    )


def _packed(t) -> bytes:
    """view_of as bytes, for _lib.call_packed."""
    s = t._storage
    return _lib.pack_view(s._ptr, t._offset, s._dtype, t._shape, t._strides)


def _packed_flat(storage: Storage, shape) -> bytes:
    """flat_view as bytes, for _lib.call_packed."""
    return _lib.pack_view(storage._ptr, 0, storage._dtype, shape, row_major_strides(shape))


def _numel(shape) -> int:
    return math.prod(shape)


# ------------------------------------------------------------- factories


def fill(n: int, value, dtype: Dtype, device: Device) -> Storage:
    if Device(device) == Device.Cpu:
        return Storage.from_iterable([value] * n, dtype, Device.Cpu)
    out = Storage.allocate(n, dtype, Device.Cuda)
    if n:
        _lib.call("nt_fill", out.data_ptr(), int(dtype), n, float(value))
    return out


# ------------------------------------------------------------ elementwise


def unary(op: int, x, scalar: float = 0.0) -> Storage:
    require_device(x)
    out = Storage.allocate(_numel(x._shape), x.dtype, Device.Cuda)
    vx = _packed(x)
    vo = _packed_flat(out, x._shape)
    _lib.call_packed("nt_unary", op, vx, float(scalar), vo)
    return out


def binary(op: int, x1, x2) -> Storage:
    require_device(x1, x2)
    if x1._shape != x2._shape:
        raise RuntimeError("_dispatch_binary: Expected two views of the same shape.")
    out_dtype = Dtype.Bool if op in (_lib.EQ, _lib.GT, _lib.GE) else x1.dtype
    out = Storage.allocate(_numel(x1._shape), out_dtype, Device.Cuda)
    v1, v2 = _packed(x1), _packed(x2)
    vo = _packed_flat(out, x1._shape)
    _lib.call_packed("nt_binary", op, v1, v2, vo)
    return out


def sgd_step(p, g, lr32: float) -> None:
    """p = p - (g * lr32) in one pass, in place (the two roundings of the
    reference's `p -= p.grad * lr`, nn/optimizers.py:45-51); float32
    device tensors of one shape, lr32 already a float32 value."""
    require_device(p, g)
    vp, vg = _packed(p), _packed(g)
    _lib.call_packed("nt_sgd_step", vp, vg, lr32)
    p._storage.bump_version()


def inplace(op: int, out, other) -> None:
    """out = out (op) other, in place (reference: inplace_ops.cu:39-79)."""
    require_device(out, other)
    vo, v2 = _packed(out), _packed(other)
    _lib.call_packed("nt_inplace", op, vo, v2)
    out._storage.bump_version()


def copy_view(src, out) -> None:
    """out[...] = src, both strided views of one shape (copy_ops.cu:187-203)."""
    _check_same_device(src, out)
    if out.device == Device.Cpu:
        _host_copy(src, out)
        return
    vs, vo = _packed(src), _packed(out)
    _lib.call_packed("nt_copy", vs, vo)


def clone_contiguous(x) -> Storage:
    """Contiguous copy of a view (copy_ops.cu:205-217)."""
    out = Storage.allocate(_numel(x._shape), x.dtype, x.device)
    if x.device == Device.Cpu:
        vals = host_values(x)
        if vals:
            out.host_array()[: len(vals)] = vals
        return out
    if _numel(x._shape):
        vs = _packed(x)
        vo = _packed_flat(out, x._shape)
        _lib.call_packed("nt_copy", vs, vo)
    return out


def cast(storage: Storage, dtype: Dtype) -> Storage:
    """Whole-buffer dtype conversion; on the device, no host round trip
    (the reference's CUDA cast copies to the host and back,
    src/cpp/storage.cpp:50-51)."""
    if dtype == storage.dtype:
        return storage
    n = storage.size
    if storage.device == Device.Cpu:
        src = storage.host_array()[:n]
        return Storage.from_iterable(src, dtype, Device.Cpu)
    out = Storage.allocate(n, dtype, Device.Cuda)
    if n:
        vs = _packed_flat(storage, (n,))
        vo = _packed_flat(out, (n,))
        _lib.call_packed("nt_copy", vs, vo)
    return out


def equals(x1, x2) -> bool:
    _check_same_device(x1, x2)
    if x1.device == Device.Cpu:
        return host_values(x1) == host_values(x2)
    v1, v2 = _packed(x1), _packed(x2)
    res = ctypes.c_int32(0)
    _lib.call_packed("nt_equals", v1, v2, ctypes.byref(res))
    return bool(res.value)


# ---------------------------------------------------------------- backward


def unary_bwd(op: int, g, saved, scalar: float, gx_target) -> "Storage | None":
    """Fused unary backward.  gx_target is an existing gradient tensor to
    accumulate into (in place) or None; returns the new storage when None."""
    require_device(g)
    vg = _packed(g)
    vs = _packed(saved) if saved is not None else None
    if gx_target is None:
        out = Storage.allocate(_numel(g._shape), g.dtype, Device.Cuda)
        vo = _packed_flat(out, g._shape)
        _lib.call_packed("nt_unary_bwd", op, vg, vs, float(scalar), vo, 0)
        return out
    vo = _packed(gx_target)
    _lib.call_packed("nt_unary_bwd", op, vg, vs, float(scalar), vo, 1)
    gx_target._storage.bump_version()
    return None


def binary_bwd(op: int, g, a, b, need_a: bool, target_a, need_b: bool, target_b):
    """Fused binary backward; returns (new_storage_a | None, new_storage_b | None)."""
    require_device(g)
    vg = _packed(g)
    va = _packed(a) if a is not None else None
    vb = _packed(b) if b is not None else None
    outs = []
    views = []
    for need, target in ((need_a, target_a), (need_b, target_b)):
        if not need:
            outs.append(None)
            views.append((None, 0))
        elif target is None:
            st = Storage.allocate(_numel(g._shape), g.dtype, Device.Cuda)
            outs.append(st)
            views.append((_packed_flat(st, g._shape), 0))
        else:
            outs.append(None)
            views.append((_packed(target), 1))
    (vga, acc_a), (vgb, acc_b) = views
    _lib.call_packed(
        "nt_binary_bwd",
        op,
        vg,
        va,
        vb,
        vga,
        acc_a,
        vgb,
        acc_b,
    )
    for need, target in ((need_a, target_a), (need_b, target_b)):
        if need and target is not None:
            target._storage.bump_version()
    return outs[0], outs[1]


# -------------------------------------------------------------- reductions


def reduce(op: int, x, axes, out_dtype: Dtype, want_aux: bool = False):
    """Reduction over `axes` (tuple order); returns Storage or
    (Storage, idx Storage, count Storage) when want_aux (max/min)."""
    require_device(x)
    keep = [s for i, s in enumerate(x._shape) if i not in axes]
    k = _numel(keep)
    out = Storage.allocate(k, out_dtype, Device.Cuda)
    vx = _packed(x)
    vo = _packed_flat(out, (k,))
    idx = cnt = None
    vi = vc = None
    if want_aux:
        idx = Storage.allocate(k, Dtype.Int64, Device.Cuda)
        cnt = Storage.allocate(k, Dtype.Int32, Device.Cuda)
        vi = _packed_flat(idx, (k,))
        vc = _packed_flat(cnt, (k,))
    arr = _lib.axes_array(axes)
    _lib.call_packed("nt_reduce", op, vx, arr, len(axes), vo, vi, vc)
    if want_aux:
        return out, idx, cnt
    return out


def mean(x, axes, out_dtype: Dtype) -> Storage:
    """Mean over `axes`: the sum in out_dtype divided by the element count,
    in one call (nt_mean)."""
    require_device(x)
    k = _numel([s for i, s in enumerate(x._shape) if i not in axes])
    out = Storage.allocate(k, out_dtype, Device.Cuda)
    vx = _packed(x)
    vo = _packed_flat(out, (k,))
    _lib.call_packed("nt_mean", vx, _lib.axes_array(axes), len(axes), vo)
    return out


def reduce_bwd(op: int, g, scale: float, idx, cnt, axes, shape, target):
    """Backward of a reduction into a tensor of `shape`.  g holds one value
    per kept index (any shape, made contiguous here); accumulates into
    `target` when given, else returns a new contiguous Storage."""
    require_device(g)
    g = g._to_contiguous()
    k = g.numel
    vg = _lib.pack_view(g._storage._ptr, g._offset, g._storage._dtype, (k,), (1,))
    vi = _packed_flat(idx, (k,)) if idx is not None else None
    vc = _packed_flat(cnt, (k,)) if cnt is not None else None
    arr = _lib.axes_array(axes)
    if target is None:
        out = Storage.allocate(_numel(shape), g.dtype, Device.Cuda)
        vo = _packed_flat(out, shape)
        acc = 0
    else:
        out = None
        vo = _packed(target)
        acc = 1
    _lib.call_packed(
        "nt_reduce_bwd",
        op,
        vg,
        float(scale),
        vi,
        vc,
        arr,
        len(axes),
        vo,
        acc,
    )
    if target is not None:
        target._storage.bump_version()
    return out


# ------------------------------------------------------------------ matmul


def matmul(x1, x2, out_shape) -> Storage:
    """Batched matmul of same-rank views (batch dims already expanded)."""
    require_device(x1, x2)
    if x1.dtype != x2.dtype:
        raise RuntimeError("matmul: dtype mismatch")
    out = Storage.allocate(_numel(out_shape), x1.dtype, Device.Cuda)
    v1, v2 = _packed(x1), _packed(x2)
    vo = _packed_flat(out, out_shape)
    _lib.call_packed("nt_matmul", v1, v2, vo, 0)
    return out


def matmul_bias(x1, x2, bias, out_shape) -> Storage:
    """x1 @ x2 + bias (2-D float32 views, bias 1-D over the columns) in one
    product whose epilogue adds the bias: the same two fp32 roundings as the
    product followed by a broadcast add."""
    require_device(x1, x2, bias)
    out = Storage.allocate(_numel(out_shape), x1.dtype, Device.Cuda)
    v1, v2, vb = _packed(x1), _packed(x2), _packed(bias)
    vo = _packed_flat(out, out_shape)
    _lib.call_packed("nt_matmul_bias", v1, v2, vb, vo)
    return out


def linear(x, w, bias, out_shape) -> Storage:
    """matmul_bias on the fp32 kernels at every size: a layer's forward."""
    require_device(x, w, bias)
    out = Storage.allocate(_numel(out_shape), x.dtype, Device.Cuda)
    _lib.call_packed("nt_linear", _packed(x), _packed(w), _packed(bias),
                     _packed_flat(out, out_shape))
    return out


def matmul_into(x1, x2, target, accumulate: bool) -> None:
    require_device(x1, x2, target)
    v1, v2, vo = _packed(x1), _packed(x2), _packed(target)
    _lib.call_packed("nt_matmul", v1, v2, vo, int(accumulate))
    target._storage.bump_version()


# ------------------------------------------------------------- host helpers


def host_values(x) -> list:
    """Values of a host view in logical row-major order."""
    arr = x._storage.host_array()
    shape, strides, off = x._shape, x._strides, x._offset
    n = _numel(shape)
    if n == 0:
        return []
    out = []

    def rec(d: int, base: int) -> None:
        if d == len(shape):
            out.append(arr[base])
            return
        st = strides[d]
        for i in range(shape[d]):
            rec(d + 1, base + i * st)

    rec(0, off)
    return out


def _host_copy(src, out) -> None:
    vals = host_values(src)
    if src.dtype != out.dtype:
        from ._storage import _convert

        vals = [_convert(v, out.dtype) for v in vals]
    arr = out._storage.host_array()
    shape, strides = out._shape, out._strides
    it = iter(vals)

    def rec(d: int, base: int) -> None:
        if d == len(shape):
            arr[base] = next(it)
            return
        for i in range(shape[d]):
            rec(d + 1, base + i * strides[d])

    if _numel(shape):
        rec(0, out._offset)

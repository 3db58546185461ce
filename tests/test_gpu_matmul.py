"""MatMulOp forward and both gradients on the GPU (fp32 MFMA) against the
oracle's sequential dot products.

Bar: |gpu - ref| <= 1e-4 * (|A|.|B|)_ij per element (a different fp32
accumulation order), plus a normwise check, on every output element; the
config shapes against the oracle's OpenMP product (bit-identical to its
sequential k loop).
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from helpers import assert_bitexact, assert_rel, dev, dev_T, host, rng, seed_of

import nanotorch_amd as nt
from nanotorch_amd import _kernels as K

pytestmark = pytest.mark.gpu


def _mm(x1, x2):
    out_shape = tuple(x1.shape[:-2]) + (x1.shape[-2], x2.shape[-1])
    return host(nt.Tensor._new_contiguous(K.matmul(x1, x2, out_shape), out_shape))


def _check(got, a, b, what):
    want = O.matmul(np.ascontiguousarray(a), np.ascontiguousarray(b), parallel=True)
    scale = O.matmul(np.abs(a).astype(np.float64), np.abs(b).astype(np.float64), parallel=True)
    assert_rel(got, want, 1e-4, what, scale=scale)
    nrm = np.linalg.norm(got.astype(np.float64) - want) / max(np.linalg.norm(want), 1e-30)
    assert nrm < 1e-5, (what, nrm)


SHAPES = [(1, 1, 1), (2, 3, 4), (5, 7, 3), (32, 32, 32), (128, 128, 128), (129, 33, 130),
          (257, 100, 63), (64, 1000, 96), (300, 257, 511), (1024, 512, 768),
          # K % 32 == 0 with ragged M / N (multiples of 4): the direct-to-LDS
          # kernel's clamped edge tiles, every layout pair
          (132, 96, 260), (36, 64, 100), (1000, 256, 1004), (4, 32, 4)]


@pytest.mark.parametrize("layout", ["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("M,K_,N", SHAPES)
def test_matmul_layouts(gpu, M, K_, N, layout):
    r = rng(seed_of(M, K_, N, layout))
    a = r.standard_normal((M, K_)).astype(np.float32)
    b = (r.standard_normal((K_, N)) / np.sqrt(K_)).astype(np.float32)
    xa = dev_T(a) if layout[0] == "T" else dev(a)
    xb = dev_T(b) if layout[1] == "T" else dev(b)
    _check(_mm(xa, xb), a, b, f"{layout} {M}x{K_}x{N}")


def test_matmul_generic_strides_and_batch(gpu):
    r = rng(1)
    a = r.standard_normal((3, 4 * 2)).astype(np.float32)
    b = np.ones((4, 2), dtype=np.float32)
    got = _mm(dev(np.arange(12, dtype=np.float32).reshape(3, 4))[:, ::2], dev(np.ones((2, 2), np.float32)))
    assert_bitexact(got, np.array([[2, 2], [10, 10], [18, 18]], np.float32), "strided ::2")
    # batched with a broadcast (stride-0) batch operand
    a = r.standard_normal((4, 3, 37, 19)).astype(np.float32)
    b = r.standard_normal((19, 23)).astype(np.float32)
    xb = dev(b).expand(4, 3, 19, 23)
    got = _mm(dev(a), xb)
    _check(got, a, np.broadcast_to(b, (4, 3, 19, 23)), "batched+bcast")
    # batched, vector layouts, K % 32 == 0 (direct-to-LDS kernel)
    a = r.standard_normal((2, 3, 68, 64)).astype(np.float32)
    b = r.standard_normal((2, 3, 64, 132)).astype(np.float32)
    _check(_mm(dev(a), dev(b)), a, b, "batched direct")
    del b


def test_matmul_other_dtypes_exact(gpu):
    """fp64 / int paths accumulate in k order like the reference: exact."""
    r = rng(2)
    for dt in (np.float64, np.int64, np.int32):
        a = (r.standard_normal((33, 45)) * 10).astype(dt)
        b = (r.standard_normal((45, 27)) * 10).astype(dt)
        got = _mm(dev(a), dev_T(b))
        assert_bitexact(got, O.matmul(a, b), f"{dt}")


def test_matmul_accumulate(gpu):
    r = rng(3)
    a = r.standard_normal((200, 150)).astype(np.float32)
    b = r.standard_normal((150, 170)).astype(np.float32)
    old = r.standard_normal((200, 170)).astype(np.float32)
    tgt = dev(old)
    K.matmul_into(dev(a), dev(b), tgt, accumulate=True)
    want = O.matmul(a, b) + old
    scale = O.matmul(np.abs(a).astype(np.float64), np.abs(b).astype(np.float64)) + np.abs(old)
    assert_rel(host(tgt), want, 1e-4, "accumulate", scale=scale)


def _full_check(got, want, scale, what):
    """Every output: |gpu - ref| <= 1e-4 * (|A|.|B|)_ij, and normwise."""
    assert_rel(got, want, 1e-4, what, scale=scale)
    nrm = np.linalg.norm(got.astype(np.float64) - want) / max(np.linalg.norm(want), 1e-30)
    assert nrm < 1e-5, (what, nrm)


@pytest.mark.parametrize("M,K_,N", [(4096, 4096, 4096), (8192, 1024, 4096)])
def test_config4_full_size(gpu, M, K_, N):
    """Config 4 at its shapes: forward, dA = dG.B^T and dB = A^T.dG through
    autograd (MatmulOp), with A contiguous and as a transposed view.  Every
    output element is compared with the oracle's sequential fp32 dot product
    (the reference's k loop) within 1e-4 * (|A|.|B|)_ij."""
    r = rng(seed_of("c4", M, K_, N))
    A = r.standard_normal((M, K_)).astype(np.float32)
    B = (r.standard_normal((K_, N)) / np.sqrt(K_)).astype(np.float32)
    G = r.standard_normal((M, N)).astype(np.float32)
    At, Bt = np.ascontiguousarray(A.T), np.ascontiguousarray(B.T)
    aA, aB, aG = (np.abs(v).astype(np.float64) for v in (A, B, G))
    ref = {"fwd": (O.matmul(A, B, parallel=True), aA @ aB),
           "dA": (O.matmul(G, Bt, parallel=True), aG @ aB.T),
           "dB": (O.matmul(At, G, parallel=True), aA.T @ aG)}
    del aA, aB, aG
    for a_layout in ("contig", "transposed"):
        xa = dev(A) if a_layout == "contig" else dev_T(A)
        xa.enable_grad()
        xb = dev(B, requires_grad=True)
        y = xa @ xb
        _full_check(host(y), *ref["fwd"], f"fwd {a_layout} {M}x{K_}x{N}")
        # backward with upstream G: loss = sum(y * G) has dL/dy = G
        loss = (y * dev(G)).sum()
        loss.backward()
        _full_check(host(xa.grad), *ref["dA"], f"dA {a_layout} {M}x{K_}x{N}")
        _full_check(host(xb.grad), *ref["dB"], f"dB {a_layout} {M}x{K_}x{N}")
        del xa, xb, y, loss


def _batched_T(a):
    """Batched device operand equal to `a`, stored with its last two axes
    swapped (a transposed view per batch)."""
    return dev(np.ascontiguousarray(np.swapaxes(a, -1, -2))).transpose(-2, -1)


@pytest.mark.parametrize("layout", ["NN", "TN", "NT", "TT"])
def test_wide_tile_kernel_full_check(gpu, layout):
    """16 x [1024, 128] @ [128, 1024]: M and N multiples of 256, K of 64,
    and 256 tiles of 256x256 -- the wide-tile kernel's conditions -- with
    every output compared, once written and once accumulated into C."""
    r = rng(seed_of("wide", layout))
    Bt, M, K_, N = 16, 1024, 128, 1024
    a = r.standard_normal((Bt, M, K_)).astype(np.float32)
    b = (r.standard_normal((Bt, K_, N)) / np.sqrt(K_)).astype(np.float32)
    xa = _batched_T(a) if layout[0] == "T" else dev(a)
    xb = _batched_T(b) if layout[1] == "T" else dev(b)
    _check(_mm(xa, xb), a, b, f"wide {layout}")
    old = r.standard_normal((Bt, M, N)).astype(np.float32)
    tgt = dev(old)
    K.matmul_into(xa, xb, tgt, accumulate=True)
    want = O.matmul(a, b, parallel=True) + old
    scale = O.matmul(np.abs(a).astype(np.float64), np.abs(b).astype(np.float64),
                     parallel=True) + np.abs(old)
    assert_rel(host(tgt), want, 1e-4, f"wide accumulate {layout}", scale=scale)


@pytest.mark.parametrize("layout", ["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("accumulate", [False, True])
def test_wide_tile_split_k_full_check(gpu, accumulate, layout):
    """[1024, 8192] @ [8192, 2048]: 32 tiles of 256x256, so the wide kernel
    splits K into 8 slices (one tile per CU) and sums them in slice order;
    every operand layout (TN is the dB = A^T.dG of autograd); every output
    compared with an fp64 product (the bound covers fp32 accumulation in any
    order)."""
    r = rng(seed_of("splitk", accumulate, layout))
    M, K_, N = 1024, 8192, 2048
    a = r.standard_normal((M, K_)).astype(np.float32)
    b = (r.standard_normal((K_, N)) / np.sqrt(K_)).astype(np.float32)
    old = r.standard_normal((M, N)).astype(np.float32)
    tgt = dev(old)
    xa = dev_T(a) if layout[0] == "T" else dev(a)
    xb = dev_T(b) if layout[1] == "T" else dev(b)
    K.matmul_into(xa, xb, tgt, accumulate=accumulate)
    want = a.astype(np.float64) @ b.astype(np.float64) + (old if accumulate else 0.0)
    scale = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64) + (
        np.abs(old) if accumulate else 0.0)
    assert_rel(host(tgt), want, 1e-4, f"split-K accumulate={accumulate}", scale=scale)


# ----------------------------------------------------- bias in the epilogue

BIAS_SHAPES = [(7, 5, 3), (129, 33, 130), (300, 257, 512),  # generic / edge tiles
               (1024, 512, 768),                            # 128x128 MFMA kernels
               (4096, 1024, 4096),                          # bf16 planes, one slice
               (1024, 8192, 4100),                          # bf16 planes, split K
               (4096, 64, 4096),                            # wide kernel, one pass
               (1024, 8192, 256),                           # tile kernels, split K
               (64, 0, 96)]                                  # K = 0: C = bias


@pytest.mark.parametrize("layout", ["NN", "TN"])
@pytest.mark.parametrize("M,K_,N", BIAS_SHAPES)
def test_matmul_bias_equals_product_then_add(gpu, M, K_, N, layout):
    """nt_matmul_bias (the bias added in the product's epilogue) against the
    same product from nt_matmul followed by the broadcast add kernel, bit for
    bit: the fused form keeps the two fp32 roundings of the reference's
    MatmulOp then AddOp."""
    r = rng(seed_of("mmbias", M, K_, N, layout))
    a = r.standard_normal((M, K_)).astype(np.float32)
    b = (r.standard_normal((K_, N)) / np.sqrt(max(K_, 1))).astype(np.float32)
    bias = r.standard_normal(N).astype(np.float32)
    ta = dev(a) if layout == "NN" else dev_T(a)
    tb, tbias = dev(b), dev(bias)
    fused = host(nt.Tensor._new_contiguous(K.matmul_bias(ta, tb, tbias, (M, N)), (M, N)))
    prod = nt.Tensor._new_contiguous(K.matmul(ta, tb, (M, N)), (M, N))
    want = host(prod + tbias)
    assert_bitexact(fused, want, f"bias {M}x{K_}x{N} {layout}")


def test_matmul_bias_rejects_bad_operands(gpu):
    a, b = dev(np.ones((4, 3), np.float32)), dev(np.ones((3, 5), np.float32))
    with pytest.raises(RuntimeError):
        K.matmul_bias(a, b, dev(np.ones(4, np.float32)), (4, 5))  # wrong length
    with pytest.raises(ValueError):
        K.matmul_bias(dev(np.ones((4, 3))), dev(np.ones((3, 5))), dev(np.ones(5)), (4, 5))


def test_linear_fused_forward_and_backward_match_the_composition(gpu):
    """nn.Linear on float32 device tensors (LinearOp: product + bias in one
    kernel) against the reference's composition x @ W + b through the
    Tensor API, bit for bit: output, dx, dW, db, first-write and
    accumulated."""
    from nanotorch_amd import nn
    r = rng(seed_of("linear-fused"))
    x = r.standard_normal((512, 256)).astype(np.float32)
    g = r.standard_normal((512, 384)).astype(np.float32)
    lin = nn.Linear(256, 384)
    W0 = host(lin._W)
    lin._b = dev(r.standard_normal(384).astype(np.float32), requires_grad=True)
    b0 = host(lin._b)
    results = []
    for fused in (True, False):
        W = dev(W0, requires_grad=True)
        b = dev(b0, requires_grad=True)
        X = dev(x, requires_grad=True)
        G = dev(g)
        for _ in range(2):  # the second pass accumulates into the grads
            if fused:
                lin._W, lin._b = W, b
                z = lin(X)
                assert type(z.grad_fn).__name__ == "LinearOp"
            else:
                z = X @ W + b
            (z * G).sum().backward()
        results.append([host(z), host(X.grad), host(W.grad), host(b.grad)])
    for name, f, c in zip(("z", "dx", "dW", "db"), *results):
        assert_bitexact(f, c, name)


@pytest.mark.parametrize("x_T", [False, True])
@pytest.mark.parametrize("x_grad,W_grad,b_grad", [(True, True, True), (False, True, True),
                                                  (True, False, False), (False, False, True)])
def test_linear_fused_grad_subsets_and_views(gpu, x_T, x_grad, W_grad, b_grad):
    """LinearOp against x @ W + b with the input read through a `.T` view
    and with each subset of x, W and b requiring a gradient (a frozen
    layer, the first layer's input): every gradient that exists matches
    the composition's bit for bit, the others stay None, and under no_grad
    neither form records a graph."""
    from nanotorch_amd import nn
    r = rng(seed_of("linear-subsets", x_T, x_grad, W_grad, b_grad))
    x = r.standard_normal((300, 130)).astype(np.float32)
    g = r.standard_normal((300, 96)).astype(np.float32)
    W0 = (r.standard_normal((130, 96)) / np.sqrt(130)).astype(np.float32)
    b0 = r.standard_normal(96).astype(np.float32)
    lin = nn.Linear(130, 96)
    results = []
    for fused in (True, False):
        W, b = dev(W0, requires_grad=W_grad), dev(b0, requires_grad=b_grad)
        leaf = dev(np.ascontiguousarray(x.T), requires_grad=x_grad) if x_T else dev(x, requires_grad=x_grad)
        X = leaf.T if x_T else leaf
        if fused:
            lin._W, lin._b = W, b
            z = lin(X)
            assert type(z.grad_fn).__name__ == "LinearOp"
        else:
            z = X @ W + b
        (z * dev(g)).sum().backward()
        results.append([host(z)] + [None if t.grad is None else host(t.grad) for t in (leaf, W, b)])
        with nt.no_grad():
            lin._W, lin._b = W, b
            assert (lin(X) if fused else X @ W + b).grad_fn is None
    for name, f, c, need in zip(("z", "dx", "dW", "db"), *results, (True, x_grad, W_grad, b_grad)):
        if not need:
            assert f is None and c is None, name
        else:
            assert_bitexact(f, c, name)


def test_linear_fused_saved_input_modified_in_place_raises(gpu):
    """LinearOp saves x and W for its backward: an in-place change to the
    input after the forward invalidates the saved version, and backward
    raises as it does for MatmulOp."""
    from nanotorch_amd import nn
    lin = nn.Linear(8, 4)
    h = dev(np.ones((5, 8), np.float32), requires_grad=True) * 2.0  # a non-leaf input
    z = lin(h)
    assert type(z.grad_fn).__name__ == "LinearOp"
    h += 1.0
    with pytest.raises(RuntimeError):
        z.sum().backward()


def test_matmul_bias_strided_operands(gpu):
    """nt_matmul_bias with a bias read through a stride-2 slice, an A whose
    rows repeat (a stride-0 expand) and a B read through `.T`, on the 128x128
    and the wide kernels: bit-identical to the product, then the add."""
    r = rng(seed_of("mmbias-strided"))
    for M, K_, N in ((200, 96, 136), (512, 512, 512)):
        row = r.standard_normal((1, K_)).astype(np.float32)
        ta = dev(row).expand(M, K_)                       # every row the same
        tb = dev_T((r.standard_normal((K_, N)) / np.sqrt(K_)).astype(np.float32))
        tbias = dev(r.standard_normal(2 * N).astype(np.float32))[::2]
        fused = host(nt.Tensor._new_contiguous(K.matmul_bias(ta, tb, tbias, (M, N)), (M, N)))
        prod = nt.Tensor._new_contiguous(K.matmul(ta, tb, (M, N)), (M, N))
        assert_bitexact(fused, host(prod + tbias), f"strided bias {M}x{K_}x{N}")


# ------------------------------------------- tile shapes, splits, any layout

# K below, at and past one k-tile of 32 and one unrolled pair; M and N on both
# sides of the 32 / 64 / 128 tiles; few rows or columns against a large
# matrix, and a small output over a long K (both split K); odd extents take
# the 4-byte loads, multiples of 4 the 16-byte ones.
TILE_SHAPES = [(1, 31, 257), (8, 2048, 1024), (3, 2047, 515), (31, 33, 129), (65, 64, 63),
               (64, 2080, 64), (100, 2001, 36), (130, 65, 32), (1000, 784, 1000), (515, 4096, 9),
               (257, 1023, 385)]


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("layout", ["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("M,K_,N", TILE_SHAPES)
def test_tile_kernel_edges(gpu, M, K_, N, layout, accumulate):
    """Every output against the fp64 product.  fp32 sums of K products in any
    order: |diff| <= K 2^-24 (|A|.|B|), times 2 for the slices' partial sums,
    plus the accumulate's own rounding."""
    r = rng(seed_of("tile", M, K_, N, layout, accumulate))
    a = r.standard_normal((M, K_)).astype(np.float32)
    b = (r.standard_normal((K_, N)) / np.sqrt(K_)).astype(np.float32)
    old = r.standard_normal((M, N)).astype(np.float32)
    tgt = dev(old)
    K.matmul_into(dev_T(a) if layout[0] == "T" else dev(a),
                  dev_T(b) if layout[1] == "T" else dev(b), tgt, accumulate=accumulate)
    add = old if accumulate else 0.0
    want = a.astype(np.float64) @ b + add
    scale = np.abs(a).astype(np.float64) @ np.abs(b) + np.abs(add)
    err = np.abs(host(tgt) - want) / scale
    assert err.max() <= min(1e-4, 2 * (K_ + 2) * 2.0**-24), err.max()


def test_tile_kernel_strided_outputs_and_batches(gpu):
    """Split and unsplit products into transposed and sliced outputs, batched
    with odd extents, and with row strides past the 32-bit load offsets."""
    r = rng(seed_of("tile-views"))
    for M, K_, N in ((40, 2000, 24), (40, 60, 24)):  # split, unsplit
        a = r.standard_normal((M, K_)).astype(np.float32)
        b = (r.standard_normal((K_, N)) / np.sqrt(K_)).astype(np.float32)
        want = a.astype(np.float64) @ b
        for tgt in (dev(np.zeros((N, M), np.float32)).T, dev(np.zeros((M, 2 * N), np.float32))[:, ::2]):
            K.matmul_into(dev(a), dev(b), tgt, accumulate=False)
            assert np.abs(host(tgt) - want).max() < 1e-4
    a = r.standard_normal((2, 3, 33, 901)).astype(np.float32)  # batched, split, 4-byte loads
    b = (r.standard_normal((2, 3, 901, 17)) / 30).astype(np.float32)
    assert np.abs(_mm(dev(a), dev(b)) - a.astype(np.float64) @ b).max() < 1e-4
    big = nt.zeros(6, 2**22 + 8, device="cuda")  # row stride past 2^22 elements
    a = r.standard_normal((6, 40)).astype(np.float32)
    big[:, 3:43] = dev(a)
    b = (r.standard_normal((40, 9)) / 6).astype(np.float32)
    assert np.abs(_mm(big[:, 3:43], dev(b)) - a.astype(np.float64) @ b).max() < 1e-4


@pytest.mark.parametrize("layout", ["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("M,K_,N", [(1000, 33, 993), (500, 70, 505), (33, 16, 65), (5, 1, 3)])
@pytest.mark.parametrize("dt", [np.float64, np.int64, np.int32])
def test_other_dtypes_exact_in_every_tile(gpu, M, K_, N, layout, dt):
    """The 4x4, 2x2 and 1x1 register tiles (1000, 500 and 33 rows; K below,
    at and past a k-tile) sum in k order with separate roundings: bit for bit
    the oracle's loop, written and accumulated, also batched."""
    r = rng(seed_of("simt", M, K_, N, layout, np.dtype(dt).name))
    a = (r.standard_normal((M, K_)) * 100).astype(dt)
    b = (r.standard_normal((K_, N)) * 100).astype(dt)
    old = (r.standard_normal((M, N)) * 100).astype(dt)
    xa = dev_T(a) if layout[0] == "T" else dev(a)
    xb = dev_T(b) if layout[1] == "T" else dev(b)
    want = O.matmul(a, b, parallel=True)
    assert_bitexact(_mm(xa, xb), want, "product")
    tgt = dev(old)
    K.matmul_into(xa, xb, tgt, accumulate=True)
    assert_bitexact(host(tgt), old + want, "accumulated")
    if M < 100:
        got = _mm(xa.reshape(1, M, K_).expand(3, M, K_), xb.reshape(1, K_, N).expand(3, K_, N))
        assert_bitexact(got, np.broadcast_to(want, (3, M, N)), "batched")


# --------------------------------------- large products on the bf16 planes

def _cached_after(call):
    """Bytes in the allocator's cache after `call` alone: its scratch."""
    import ctypes

    from nanotorch_amd import _lib
    _lib.call("nt_empty_cache")
    call()
    nt.sync()
    used, cached = ctypes.c_size_t(), ctypes.c_size_t()
    _lib.call("nt_memory_stats", ctypes.byref(used), ctypes.byref(cached))
    return cached.value


# one slice and several of K; M, N and K off every tile, step and vector size
SPLIT_SHAPES = [(4096, 320, 4096), (4093, 301, 4090), (1020, 8200, 4100), (2300, 4101, 2305)]


@pytest.mark.parametrize("layout", ["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("M,K_,N", SPLIT_SHAPES)
def test_split_product(gpu, M, K_, N, layout):
    """Products that run as three bf16 parts per operand: every output within
    the bound of a float32 sum in any order (K 2^-24 (|A|.|B|)), and in
    2-norm no further from 64 bits than 1.1 of sqrt(K) / 2 roundings."""
    r = rng(seed_of("split", M, K_, N, layout))
    a = r.standard_normal((M, K_), dtype=np.float32)
    b = r.standard_normal((K_, N), dtype=np.float32) / np.float32(np.sqrt(K_))
    xa = dev_T(a) if layout[0] == "T" else dev(a)
    xb = dev_T(b) if layout[1] == "T" else dev(b)
    old = r.standard_normal((M, N), dtype=np.float32)
    tgt = dev(old)
    packed = 6 * (M * K_ + K_ * N)
    assert _cached_after(lambda: K.matmul_into(xa, xb, tgt, accumulate=False)) >= packed
    want = a.astype(np.float64) @ b
    scale = np.abs(a).astype(np.float64) @ np.abs(b)
    got = host(tgt)
    err = np.abs(got - want)
    assert (err / scale).max() <= K_ * 2.0**-24
    assert np.linalg.norm(err) <= 1.1 * np.sqrt(K_) / 2 * 2.0**-24 * np.linalg.norm(want) + 2.0**-24
    tgt = dev(old)
    K.matmul_into(xa, xb, tgt, accumulate=True)
    assert_bitexact(host(tgt), old + got, "accumulated")


@pytest.mark.parametrize("special", ["inf", "nan", "large", "tiny", "tiny row", "both small", "zeros"])
@pytest.mark.parametrize("M,K_,N", [(4096, 320, 4096), (1020, 8200, 4100)])
def test_split_product_outside_its_range(gpu, M, K_, N, special):
    """Values that the parts cannot represent take the fp32 kernel: the same
    infinities and NaN as the fp32 product, and full relative precision of
    large, tiny and mixed magnitudes; zeros stay in range."""
    r = rng(seed_of("split-range", M, special))
    a = r.standard_normal((M, K_), dtype=np.float32)
    b = r.standard_normal((K_, N), dtype=np.float32)
    if special in ("inf", "nan"):
        a[17, 5] = np.inf if special == "inf" else np.nan
    elif special == "large":
        a *= np.float32(1e30)
    elif special == "tiny":
        a *= np.float32(1e-30)
    elif special == "tiny row":
        a[17] *= np.float32(1e-30)
    elif special == "both small":
        a *= np.float32(1e-15)
        b *= np.float32(1e-15)
    else:
        a[::3] = 0.0
        b[:, ::2] = -0.0
    got = host(nt.Tensor._new_contiguous(K.matmul(dev(a), dev(b), (M, N)), (M, N)))
    if special in ("inf", "nan"):
        with np.errstate(invalid="ignore"):
            row = a[17].astype(np.float64) @ b
        assert (np.isnan(got[17]) == np.isnan(row)).all()
        assert (np.isinf(got[17]) == np.isinf(row)).all()
        a, got = np.delete(a, 17, 0), np.delete(got, 17, 0)
    want = a.astype(np.float64) @ b
    scale = np.abs(a).astype(np.float64) @ np.abs(b)
    assert (np.abs(got - want) <= K_ * 2.0**-24 * scale).all()


@pytest.mark.parametrize("K_", [320, 400])  # the last k step as it is, and packed negated
def test_split_product_zero_sums_are_positive(gpu, K_):
    """Sums of zeros are +0, as every float32 sum that starts at +0."""
    a = np.zeros((4096, K_), np.float32)
    a[::2] = -0.0
    b = rng(seed_of("split-zero", K_)).standard_normal((K_, 4096), dtype=np.float32)
    got = host(nt.Tensor._new_contiguous(K.matmul(dev(a), dev(b), (4096, 4096)), (4096, 4096)))
    assert not got.any() and not np.signbit(got).any()


def test_layer_forward_keeps_the_fp32_rounding(gpu):
    """A layer's forward at a size whose plain product takes the planes: bit
    for bit the values of a run in which another row's infinity keeps that
    product on the fp32 kernel."""
    from nanotorch_amd import nn
    r = rng(seed_of("layer-forward"))
    lin = nn.Linear(1024, 4096)
    lin._W = dev(r.standard_normal((1024, 4096), dtype=np.float32) / np.float32(32))
    x = r.standard_normal((4096, 1024), dtype=np.float32)
    clean = host(lin(dev(x)))
    x[17, 5] = np.inf
    assert_bitexact(np.delete(clean, 17, 0), np.delete(host(lin(dev(x))), 17, 0), "forward")


def _sparse_operand(kind, n, r):
    a = np.zeros((n, n), np.float32)
    i = np.arange(n)
    if kind == "one-hot":
        a[i, r.permutation(n)] = 1
    else:
        a[i, i] = r.standard_normal(n, dtype=np.float32)
    if kind == "two terms":
        a[i, (7 * i + 3) % n] = r.standard_normal(n, dtype=np.float32)
    return a


@pytest.mark.parametrize("kind,most,rms", [("one-hot", 0, 0), ("diagonal", 2, 0.45),
                                           ("two terms", 3, 0.45)])
def test_split_product_of_few_terms(gpu, kind, most, rms):
    """Plane products whose sums have one or two terms, where the running
    sum's rounding does not hide a product's own.  In 2^-24 (|A|.|B|): each
    rounding of the sum is at most 1, the products of parts left out 1 in
    all, the five small products' roundings 1/16; a one-hot operand's parts
    are exact.  rms of one rounding to nearest
    0.425 (a value uniform in an ulp, its size log-uniform); the fp32 kernel
    has 0.425 and 0.436 for one and two terms."""
    n = 4096
    r = rng(seed_of("split-few", kind))
    a = _sparse_operand(kind, n, r)
    b = r.standard_normal((n, n), dtype=np.float32)
    got = _mm(dev(a), dev(b))
    want = a.astype(np.float64) @ b
    err = np.abs(got - want) * 2.0**24
    scale = np.abs(a).astype(np.float64) @ np.abs(b)
    assert (err <= (most + 1 / 16 if most else 0) * scale).all()
    q = err[scale > 0] / scale[scale > 0]
    assert np.sqrt(np.mean(q * q)) <= rms


@pytest.mark.parametrize("K_", [320, 4096])
@pytest.mark.parametrize("dist", ["normal", "positive"])
def test_split_product_has_no_mean_shift(gpu, dist, K_):
    """The matrix cores round the planes' sums down; over 16 million results
    what is left of that is below 2^-29 of their mean size (left alone it was
    2.6e-7, over 2^-22), and a column's mean is no
    further from 64 bits than its 4096 roundings to nearest allow."""
    r = rng(seed_of("split-shift", dist, K_))
    a = r.standard_normal((4096, K_), dtype=np.float32)
    b = r.standard_normal((K_, 4096), dtype=np.float32) / np.float32(np.sqrt(K_))
    if dist == "positive":
        a, b = np.abs(a), np.abs(b)
    got = _mm(dev(a), dev(b))
    want = a.astype(np.float64) @ b
    err = got - want
    assert abs(err.mean()) <= 2.0**-29 * np.abs(want).mean()
    # one rounding per 32 k's and two at the end, of sums no larger than the
    # rows' largest; independent ones: 4.5 of their standard deviations
    per = np.sqrt(K_ / 32 + 2) * 2.0**-24 * np.abs(want).max() / np.sqrt(3 * 4096)
    assert np.abs(err.mean(0)).max() <= 4.5 * per


@pytest.mark.parametrize("layout", ["NN", "TN"])
@pytest.mark.parametrize("M,K_,N", [(1020, 8200, 4100), (2300, 4101, 2305), (2048, 8192, 1024)])
def test_split_product_fallback_is_the_fp32_product(gpu, M, K_, N, layout):
    """A product whose data is outside the planes' range: bit for bit what the
    fp32 kernels give it as a layer's forward (same tiles, same slices of K),
    written, accumulated and with a bias, each added once; 16- and 4-byte
    loads, and the split 256x256 tile."""
    r = rng(seed_of("split-fallback", M, K_, N, layout))
    a = r.standard_normal((M, K_), dtype=np.float32)
    a[17, 5] = np.inf
    xa = dev_T(a) if layout == "TN" else dev(a)
    xb = dev(r.standard_normal((K_, N), dtype=np.float32))
    bias = dev(r.standard_normal(N, dtype=np.float32))
    old = r.standard_normal((M, N), dtype=np.float32)

    def rows(x):
        return np.delete(x, 17, 0)

    def run(op, *args):
        return rows(host(nt.Tensor._new_contiguous(op(*args, (M, N)), (M, N))))

    want = run(K.linear, xa, xb, dev(np.zeros(N, np.float32)))
    assert_bitexact(run(K.matmul, xa, xb), want, "written")
    tgt = dev(old)
    K.matmul_into(xa, xb, tgt, accumulate=True)
    assert_bitexact(rows(host(tgt)), rows(old) + want, "accumulated")
    assert_bitexact(run(K.matmul_bias, xa, xb, bias), run(K.linear, xa, xb, bias), "bias")


@pytest.mark.parametrize("values", ["one tiny", "softmax", "subnormal rows", "far apart"])
def test_split_product_of_wide_ranges(gpu, values):
    """Values down to the subnormals, and operands of very different size,
    stay on the planes (other last bits than the fp32 kernels): less than half
    of the fp32 kernels' error in 2-norm, and each result within the bound of
    a float32 sum (plus the spacing of the subnormals where it is one).  Of
    the softmax-like rows, exp(12 n - 50), one term is nearly all of the
    2-norm: there it is one rounding and the products left out against one
    rounding, rms 0.436 against 0.425 of 2^-24."""
    M, K_, N = 4096, 320, 4096
    r = rng(seed_of("split-wide", values))
    a = r.standard_normal((M, K_), dtype=np.float32)
    b = r.standard_normal((K_, N), dtype=np.float32)
    if values == "one tiny":
        a[17, 5] = 2.0**-70
    elif values == "softmax":
        a = np.exp(12 * a - 50) / np.float32(8192)  # 2^-126 and below to about 1
    elif values == "subnormal rows":
        a[17] *= np.float32(2.0**-130)
        a[18] *= np.float32(2.0**-110)
    else:
        a *= np.float32(2.0**50)
        b *= np.float32(2.0**-60)
    xa, xb = dev(a), dev(b)
    got = _mm(xa, xb)
    zero = dev(np.zeros(N, np.float32))
    fp32 = host(nt.Tensor._new_contiguous(K.linear(xa, xb, zero, (M, N)), (M, N)))
    want = a.astype(np.float64) @ b
    scale = np.abs(a).astype(np.float64) @ np.abs(b)
    assert (np.abs(got - want) <= K_ * 2.0**-24 * scale + 2.0**-149).all()
    assert (got != fp32).any()
    most = 1.05 if values == "softmax" else 0.5
    assert np.linalg.norm(got - want) < most * np.linalg.norm(fp32 - want)


@pytest.mark.parametrize("K_", [68, 71, 2100])  # 16- and 4-byte loads, a tail, K split
@pytest.mark.parametrize("form", ["A", "A.T", "B", "B.T", "both"])
def test_far_strides(gpu, form, K_):
    """Operands whose rows (or, transposed, whose k's) lie over 2^22 elements
    apart, beside one of ordinary strides or another such; 70 rows are two
    tiles, the second ragged.  Every output against the fp64 product, written
    and accumulated."""
    r = rng(seed_of("far", form, K_))
    rows, off = 72 if form.endswith("T") else 70, 4 if K_ % 4 == 0 else 3
    big = nt.zeros(rows, 2**22 + 2200, device="cuda")
    n = 44  # columns of a transposed far operand
    vals = r.standard_normal((rows, n if form.endswith("T") else K_), dtype=np.float32)
    big[:, off:off + vals.shape[1]] = dev(vals)
    far = big[:, off:off + vals.shape[1]]
    if form == "A":  # [rows, K] . [K, n]
        b = r.standard_normal((K_, n), dtype=np.float32)
        xa, xb, a = far, dev(b), vals
    elif form == "B.T":  # [n, rows] . [rows, n]: k walks the far rows of B
        a = r.standard_normal((52, rows), dtype=np.float32)
        xa, xb, b = dev(a), far, vals
    elif form == "A.T":
        b = r.standard_normal((rows, 52), dtype=np.float32)
        xa, xb, a = far.T, dev(b), vals.T
    elif form == "B":  # [52, K] . [K, rows], B column-major
        a = r.standard_normal((52, K_), dtype=np.float32)
        xa, xb, b = dev(a), far.T, vals.T
    else:
        xa, xb, a, b = far, far.T, vals, vals.T
    want = a.astype(np.float64) @ b
    scale = np.abs(a).astype(np.float64) @ np.abs(b)
    old = r.standard_normal(want.shape, dtype=np.float32)
    tgt = dev(old)
    for acc in (False, True):
        K.matmul_into(xa, xb, tgt, accumulate=acc)
        # K products in any order, the slices' sums and the accumulate
        bound = 2 * (a.shape[1] + 2) * 2.0**-24 * scale * (2 if acc else 1)
        assert (np.abs(host(tgt) - want * (2 if acc else 1)) <= bound).all()

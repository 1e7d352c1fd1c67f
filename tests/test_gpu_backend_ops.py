"""ExecutionBackend ops on the device (GPU): the strided fp32 ops a
HipBackend serves to the reference's Tensor (include/backend/backend.hpp:
35-220), against CpuBackend's semantics (src/backend/cpu_backend.cpp).

Bit-exact where the reference's arithmetic fixes every rounding: add / sub /
mul / div and the element-wise backward formulas (one IEEE operation per
step), relu, sum (the reference adds each output's inputs in ascending
input index, serially), matmul against the oracle's Dense product (ascending
k, separately rounded products and sums; the sgemm the reference calls for
row-major operands fixes no order, its naive loop does), embedding, slice
backward.  Within 1e-6 relative where a libm function enters (exp, tanh,
sqrt, log) or a reduction order is free (softmax's sum).
"""
import numpy as np
import pytest

import oracle_py as O
from gpu_util import nnhip

pytestmark = pytest.mark.gpu


def dev(ctx, a):
    return ctx.array(np.ascontiguousarray(a, np.float32))


def strided(ctx, host, perm):
    """A device copy of host transposed by perm, viewed back in host's
    logical order through permuted strides (a non-contiguous operand)."""
    t = np.ascontiguousarray(np.transpose(host, perm))
    d = dev(ctx, t)
    st_t = [int(np.prod(t.shape[i + 1:])) for i in range(t.ndim)]
    inv = np.argsort(perm)
    return d, nnhip.view(d, host.shape, [st_t[i] for i in inv])


def run_binary(ctx, op, a, b, a_view=None, b_view=None, out_shape=None):
    da, db = dev(ctx, a), dev(ctx, b)
    shape = out_shape or np.broadcast_shapes(a.shape, b.shape)
    do = ctx.array(shape=shape)
    nnhip.call("nnhip_binary_f32", ctx.h, op, a_view or nnhip.view(da),
               b_view or nnhip.view(db), nnhip.view(do))
    return do.numpy()


NP_BINARY = {nnhip.OP_ADD: np.add, nnhip.OP_SUB: np.subtract,
             nnhip.OP_MUL: np.multiply, nnhip.OP_DIV: np.divide}


@pytest.mark.parametrize("op", sorted(NP_BINARY))
@pytest.mark.parametrize("sa,sb", [((4, 5, 6), (4, 5, 6)), ((4, 5, 6), (6,)),
                                   ((4, 5, 6), (5, 1)), ((1, 5, 6), (4, 1, 6)),
                                   ((3000,), (3000,)), ((7,), (1,))])
def test_binary_broadcast_bit_exact(ctx, op, sa, sb):
    rng = np.random.default_rng(op)
    a = rng.standard_normal(sa).astype(np.float32)
    b = (rng.standard_normal(sb).astype(np.float32) + np.float32(3.0))
    got = run_binary(ctx, op, a, b)
    np.testing.assert_array_equal(got, NP_BINARY[op](a, b))


def test_binary_strided_and_offset(ctx):
    """Transposed operands, a view at an element offset, and a strided
    output (every second column of a wider buffer)."""
    rng = np.random.default_rng(1)
    a = rng.standard_normal((6, 9)).astype(np.float32)
    b = rng.standard_normal((6, 9)).astype(np.float32)
    da, va = strided(ctx, a, (1, 0))
    pad = np.concatenate([np.zeros(5, np.float32), b.ravel()])
    db = dev(ctx, pad)
    vb = nnhip.view(db, (6, 9), (9, 1), offset=5)
    do = ctx.array(shape=(6, 18))
    nnhip.call("nnhip_fill_f32", ctx.h, do.p, 6 * 18, -7.0)
    vo = nnhip.view(do, (6, 9), (18, 2))
    nnhip.call("nnhip_binary_f32", ctx.h, nnhip.OP_MUL, va, vb, vo)
    out = do.numpy()
    np.testing.assert_array_equal(out[:, 0::2], a * b)
    assert (out[:, 1::2] == -7.0).all()


def test_backward_elementwise_bit_exact(ctx):
    """relu / sigmoid / tanh / sqrt / log backward (cpu_backend.cpp:473-481,
    492-502, 513-521, 659-669, 680-690), each step one IEEE operation."""
    rng = np.random.default_rng(2)
    x = rng.standard_normal((37, 41)).astype(np.float32)
    y = np.abs(x) + np.float32(0.1)
    go = rng.standard_normal((37, 41)).astype(np.float32)
    one, eps = np.float32(1.0), np.float32(1e-8)
    cases = {nnhip.OP_RELU_BACKWARD: (x, np.where(x > 0, go, np.float32(0))),
             nnhip.OP_SIGMOID_BACKWARD: (y, (go * y) * (one - y)),
             nnhip.OP_TANH_BACKWARD: (y, go * (one - y * y)),
             nnhip.OP_SQRT_BACKWARD: (y, go * (np.float32(0.5) / (y + eps))),
             nnhip.OP_LOG_BACKWARD: (y, go / (y + eps))}
    for op, (a, want) in cases.items():
        np.testing.assert_array_equal(run_binary(ctx, op, a, go), want,
                                      err_msg=str(op))


def test_unary_ops(ctx):
    rng = np.random.default_rng(3)
    x = rng.standard_normal((5, 300)).astype(np.float32) * np.float32(3)
    pos = np.abs(x) + np.float32(1e-3)
    x64 = x.astype(np.float64)
    cases = {nnhip.OP_RELU: (x, np.maximum(x64, 0)),
             nnhip.OP_SIGMOID: (x, 1 / (1 + np.exp(-x64))),
             nnhip.OP_TANH: (x, np.tanh(x64)),
             nnhip.OP_SQRT: (pos, np.sqrt(pos.astype(np.float64))),
             nnhip.OP_LOG: (pos, np.log(pos.astype(np.float64) + 1e-8))}
    for op, (a, want) in cases.items():
        da, do = dev(ctx, a), ctx.array(shape=a.shape)
        nnhip.call("nnhip_unary_f32", ctx.h, op, nnhip.view(da), nnhip.view(do))
        got = do.numpy().astype(np.float64)
        # relative to max(|value|, 1): log crosses zero at x = 1, where a
        # correctly rounded fp32 result still differs from float64 by ~1e-8
        err = np.abs(got - want) / np.maximum(np.abs(want), 1.0)
        assert err.max() <= 1e-6, (op, err.max())
    # a transposed input into a contiguous output
    da, va = strided(ctx, x, (1, 0))
    do = ctx.array(shape=x.shape)
    nnhip.call("nnhip_unary_f32", ctx.h, nnhip.OP_RELU, va, nnhip.view(do))
    np.testing.assert_array_equal(do.numpy(), np.maximum(x, 0))


@pytest.mark.parametrize("M,K,N", [(1, 64, 192), (7, 33, 5), (64, 128, 64),
                                   (130, 257, 70)])
def test_matmul_matches_oracle_dense(ctx, M, K, N):
    """Tensor::matmul -> ExecutionBackend::matmul (tensor.cpp:392-428): the
    oracle's Dense product without bias (or_dense: ascending k, separately
    rounded) bit for bit; against float64 within fp32 rounding."""
    rng = np.random.default_rng(M * 1000 + K)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = rng.standard_normal((K, N)).astype(np.float32)
    da, db, do = dev(ctx, a), dev(ctx, b), ctx.array(shape=(M, N))
    nnhip.call("nnhip_matmul_f32", ctx.h, nnhip.view(da), nnhip.view(db),
               nnhip.view(do))
    got = do.numpy()
    want = np.zeros((M, N), np.float32)
    O.lib().or_dense(O.fptr(a), M, K, N, O.fptr(b), None, None, None,
                     O.fptr(want))
    np.testing.assert_array_equal(got, want)
    ex = a.astype(np.float64) @ b.astype(np.float64)
    assert np.abs(got - ex).max() <= 1e-5 * np.abs(a).max() * np.abs(b).max() * K
    # transposed operands (the reference's sgemm Trans cases) and a strided
    # output give the same values
    ta, va = strided(ctx, a, (1, 0))
    tb, vb = strided(ctx, b, (1, 0))
    do2 = ctx.array(shape=(M, 2 * N))
    nnhip.call("nnhip_matmul_f32", ctx.h, va, vb,
               nnhip.view(do2, (M, N), (2 * N, 2)))
    np.testing.assert_array_equal(do2.numpy()[:, 0::2], want)


@pytest.mark.parametrize("M,K,N", [
    # 32 x 32 tiles: remainders of rows, columns and of the 32-wide K steps
    (33, 1, 31), (1, 31, 97), (32, 32, 32), (95, 67, 65), (31, 36, 513),
    # 64 x 64 tiles (from 160 on), the same remainders
    (64 * 13 - 63, 33, 64 * 13 - 1), (64 * 10, 64, 64 * 16), (2, 40, 64 * 160),
    # a short K over many tiles: remainders of rows, columns and of its 16-wide
    # K steps, one side thin either way
    (1, 1, 64 * 1024), (3, 15, 64 * 1023 + 5), (64 * 1023 + 5, 16, 2), (7, 17, 64 * 1088),
    (64 * 1984 - 3, 31, 32), (5, 33, 64 * 8192)])
def test_matmul_tiles_bit_exact(ctx, M, K, N):
    """Each kernel's tiles at their edges, row-major and transposed operands,
    against or_dense (ascending k, separately rounded) bit for bit; the
    entries around the output stay untouched."""
    rng = np.random.default_rng(M + K + N)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = rng.standard_normal((K, N)).astype(np.float32)
    want = np.zeros((M, N), np.float32)
    O.lib().or_dense(O.fptr(a), M, K, N, O.fptr(b), None, None, None,
                     O.fptr(want))
    keep = np.full((M + 1, N + 3), 7.0, np.float32)
    for pa, pb in ((False, False), (True, True)):
        da, va = strided(ctx, a, (1, 0)) if pa else (None, nnhip.view(dev(ctx, a)))
        db, vb = strided(ctx, b, (1, 0)) if pb else (None, nnhip.view(dev(ctx, b)))
        do = ctx.array(keep)
        nnhip.call("nnhip_matmul_f32", ctx.h, va, vb,
                   nnhip.view(do, (M, N), (N + 3, 1)))
        got = do.numpy()
        np.testing.assert_array_equal(got[:M, :N], want)
        assert (got[M] == 7).all() and (got[:, N:] == 7).all()


@pytest.mark.parametrize("K", [33, 70])   # matmul_short_kernel, matmul_kernel
def test_matmul_columns_beyond_one_launch(ctx, K):
    """One row times more columns than the threads of one launch of
    matmul_kernel cover, every column the same one of b (stride 0): all of them
    are written, up to the row's end and not past it.  (In one launch only the
    columns beyond the threads' wrap would be, without an error.)"""
    N = 2 ** 29 + 70
    a, b = np.arange(1, K + 1, dtype=np.float32), np.full(K, 0.5, np.float32)
    da, db, do = dev(ctx, a), dev(ctx, b), ctx.array(shape=(N + 100,))
    nnhip.call("nnhip_fill_f32", ctx.h, do.p, N + 100, 7.0)
    nnhip.call("nnhip_matmul_f32", ctx.h, nnhip.view(da, (1, K)),
               nnhip.view(db, (K, N), (1, 0)), nnhip.view(do, (1, N)))
    got = np.empty(200, np.float32)
    for at in (0, 2 ** 28 - 100, 2 ** 29 - 100, N - 100):
        nnhip.call("nnhip_d2h", ctx.h, nnhip.ptr(got),
                   np.ctypeslib.ctypes.c_void_p(do.p.value + 4 * at), got.nbytes)
        assert (got[:min(200, N - at)] == 0.5 * K * (K + 1) / 2).all(), at
    assert (got[100:] == 7).all()


def test_matmul_known_answer_and_errors(ctx):
    """TensorTest.MatmulContiguous (tensor_test.cpp:82-94): [[1,2,3],[4,5,6]]
    . [[7,8],[9,10],[11,12]] = [[58,64],[139,154]]; shape errors carry the
    reference's messages (cpu_backend.cpp:332-342)."""
    a = np.array([[1, 2, 3], [4, 5, 6]], np.float32)
    b = np.array([[7, 8], [9, 10], [11, 12]], np.float32)
    da, db, do = dev(ctx, a), dev(ctx, b), ctx.array(shape=(2, 2))
    nnhip.call("nnhip_matmul_f32", ctx.h, nnhip.view(da), nnhip.view(db),
               nnhip.view(do))
    np.testing.assert_array_equal(do.numpy(), [[58, 64], [139, 154]])
    with pytest.raises(nnhip.NNHipError, match="Incompatible shapes"):
        nnhip.call("nnhip_matmul_f32", ctx.h, nnhip.view(da), nnhip.view(da),
                   nnhip.view(do))
    with pytest.raises(nnhip.NNHipError, match="only supports 2D"):
        nnhip.call("nnhip_matmul_f32", ctx.h, nnhip.view(da, (6,)),
                   nnhip.view(db), nnhip.view(do))


def serial_sum(x, axes, keep):
    """Sum over `axes` adding each output's inputs in ascending input index
    (float32 running sum: np.cumsum is sequential)."""
    kept = [d for d in range(x.ndim) if d not in axes]
    t = np.transpose(x, kept + sorted(axes))
    flat = t.reshape([x.shape[d] for d in kept] + [-1])
    s = np.cumsum(flat, axis=-1, dtype=np.float32)[..., -1]
    if keep:
        s = s.reshape([1 if d in axes else x.shape[d] for d in range(x.ndim)])
    return s


@pytest.mark.parametrize("axes,keep", [((0,), True), ((1,), False),
                                       ((0, 2), True), ((0, 1, 2), False),
                                       ((2,), False)])
def test_sum_bit_exact(ctx, axes, keep):
    rng = np.random.default_rng(len(axes))
    x = rng.standard_normal((6, 700, 9)).astype(np.float32)
    want = serial_sum(x, axes, keep)
    dx = dev(ctx, x)
    do = ctx.array(shape=want.shape if want.ndim else (1,))
    vo = nnhip.view(do, want.shape)
    ax = (np.ctypeslib.ctypes.c_int64 * len(axes))(*axes)
    nnhip.call("nnhip_sum_f32", ctx.h, nnhip.view(dx), vo, ax, len(axes))
    np.testing.assert_array_equal(do.numpy().reshape(want.shape), want)


@pytest.mark.parametrize("shape,axes,perm", [
    ((1024, 100), (0,), None), ((1024, 100), (0,), (1, 0)),
    ((3, 5000), (1,), None), ((3, 5000), (1,), (1, 0)), ((70001,), (0,), None),
    ((513, 16, 7), (1,), None), ((257, 33, 3), (0, 2), (2, 0, 1)),
    ((2, 3000, 5, 2), (0, 1, 3), None), ((600, 15), (1,), None),
    ((600, 17), (1,), None), ((1, 4, 1), (1,), None), ((5, 0, 3), (1,), None)])
def test_sum_tiles_bit_exact(ctx, shape, axes, perm):
    """Long and short sums of one to hundreds of outputs, the loads along
    either dimension, merged and separate reduced dims, remainders of the
    tiles and an empty sum: the ascending-order float32 sum bit for bit."""
    rng = np.random.default_rng(len(shape) + shape[0])
    x = rng.standard_normal(shape).astype(np.float32)
    want = serial_sum(x, axes, False) if x.size else np.zeros((5, 3), np.float32)
    dx, vx = strided(ctx, x, perm) if perm else (None, nnhip.view(dev(ctx, x)))
    do = ctx.array(shape=want.shape if want.ndim else (1,))
    ax = (np.ctypeslib.ctypes.c_int64 * len(axes))(*axes)
    nnhip.call("nnhip_sum_f32", ctx.h, vx, nnhip.view(do, want.shape), ax,
               len(axes))
    np.testing.assert_array_equal(do.numpy().reshape(want.shape), want)


@pytest.mark.parametrize("shape,axes,perm", [
    # along the outputs: 1 to 32 entries, and more over 65536 outputs and more
    ((1, 777), (0,), None), ((7, 1000), (0,), None), ((8, 3, 500), (0,), None),
    ((32, 1030), (0,), None), ((33, 65536), (0,), None), ((41, 70001), (0,), None),
    # along the sums, up to 12; two reduced dims; a transposed input
    ((999, 12), (1,), None), ((999, 9), (1,), None), ((2, 700, 4), (0, 2), None),
    ((3, 50, 2, 6), (0, 2), (3, 1, 0, 2)), ((500, 11), (1,), (1, 0)),
    ((131072, 17), (1,), None),
    # at the line on either side of it
    ((999, 13), (1,), None), ((33, 65535), (0,), None), ((33, 1030), (0,), None)])
def test_sum_short_bit_exact(ctx, shape, axes, perm):
    """Sums with a thread an output (few entries, or many outputs): remainders
    of the eight entries requested together and of the workgroup, kept and
    dropped dims, into a strided output; the ascending-order float32 sum bit
    for bit, the entries between the outputs untouched."""
    rng = np.random.default_rng(len(shape) + shape[0])
    x = rng.standard_normal(shape).astype(np.float32)
    x.flat[3] = -0.0
    _, vx = strided(ctx, x, perm) if perm else (None, nnhip.view(dev(ctx, x)))
    ax = (np.ctypeslib.ctypes.c_int64 * len(axes))(*axes)
    for keep in (True, False):
        want = serial_sum(x, axes, keep)
        do = ctx.array(np.full((want.size, 2), 7, np.float32))
        st = [2 * int(np.prod(want.shape[i + 1:])) for i in range(want.ndim)]
        nnhip.call("nnhip_sum_f32", ctx.h, vx, nnhip.view(do, want.shape, st),
                   ax, len(axes))
        np.testing.assert_array_equal(do.numpy()[:, 0].reshape(want.shape), want)
        assert (do.numpy()[:, 1] == 7).all()


@pytest.mark.parametrize("shape,axes,strides", [
    ((2 ** 31 + 9, 0), (0, 1), (0, 1)), ((0, 2 ** 31, 3), (0, 1), (0, 0, 1)),
    ((70000, 70000, 0), (0, 1, 2), (70000, 1, 1))])
def test_sum_extents_beyond_32_bits(ctx, shape, axes, strides):
    """Summed extents past 2^31 - 1, alone and merged, are taken (here with an
    empty one beside them, so that the sums are 0 and quick)."""
    kept = [n for d, n in enumerate(shape) if d not in axes]
    do = ctx.array(np.full(3, 7, np.float32))
    ax = (np.ctypeslib.ctypes.c_int64 * len(axes))(*axes)
    nnhip.call("nnhip_sum_f32", ctx.h,
               nnhip.view(dev(ctx, np.ones(4)), shape, strides),
               nnhip.view(do, kept), ax, len(axes))
    n = int(np.prod(kept))
    assert (do.numpy()[:n] == 0).all() and (do.numpy()[n:] == 7).all()


def test_reference_tensor_known_answers(ctx):
    """The reference's Tensor KATs through the backend ops: BroadcastingAdd
    (tensor_test.cpp:53-67, [2,3] + [1,3]), ElementwiseSubAndMul (:69-80),
    SumReduction (:97-118: all axes -> rank 0 = 21, axis 0 -> [5,7,9],
    axis 1 keepdims -> [2,1] = [6,15]); and axis 0 of a transposed input."""
    x = np.array([[1, 2, 3], [4, 5, 6]], np.float32)
    got = run_binary(ctx, nnhip.OP_ADD, x, np.array([[10, 20, 30]], np.float32))
    np.testing.assert_array_equal(got, [[11, 22, 33], [14, 25, 36]])
    a, b = np.array([10, 20], np.float32), np.array([2, 5], np.float32)
    np.testing.assert_array_equal(run_binary(ctx, nnhip.OP_SUB, a, b), [8, 15])
    np.testing.assert_array_equal(run_binary(ctx, nnhip.OP_MUL, a, b), [20, 100])
    for axes, shape, want in (((0, 1), (), [21]), ((0,), (3,), [5, 7, 9]),
                              ((1,), (2, 1), [6, 15])):
        dx = dev(ctx, x)
        do = ctx.array(shape=(len(want),))
        ax = (np.ctypeslib.ctypes.c_int64 * len(axes))(*axes)
        nnhip.call("nnhip_sum_f32", ctx.h, nnhip.view(dx),
                   nnhip.view(do, shape), ax, len(axes))
        np.testing.assert_array_equal(do.numpy(), want)
    _, vt = strided(ctx, x, (1, 0))
    do = ctx.array(shape=(3,))
    ax = (np.ctypeslib.ctypes.c_int64 * 1)(0)
    nnhip.call("nnhip_sum_f32", ctx.h, vt, nnhip.view(do), ax, 1)
    np.testing.assert_array_equal(do.numpy(), [5, 7, 9])


@pytest.mark.parametrize("shape,axis", [((4, 32000), 1), ((37, 5), 0),
                                        ((3, 7, 11), 1), ((2, 1, 9), 2)])
def test_softmax_and_backward(ctx, shape, axis):
    rng = np.random.default_rng(sum(shape))
    x = (rng.standard_normal(shape) * 3).astype(np.float32)
    dx = dev(ctx, x)
    do = ctx.array(shape=shape)
    nnhip.call("nnhip_softmax_f32", ctx.h, nnhip.view(dx), nnhip.view(do), axis)
    y = do.numpy()
    x64 = x.astype(np.float64)
    e = np.exp(x64 - x64.max(axis=axis, keepdims=True))
    want = e / e.sum(axis=axis, keepdims=True)
    assert (np.abs(y - want) / want).max() <= 2e-6
    # softmax_backward: dx = y * (dy - sum(dy * y))
    g = rng.standard_normal(shape).astype(np.float32)
    dg, dgi = dev(ctx, g), ctx.array(shape=shape)
    nnhip.call("nnhip_softmax_backward_f32", ctx.h, nnhip.view(do),
               nnhip.view(dg), nnhip.view(dgi), axis)
    y64 = y.astype(np.float64)
    wb = y64 * (g - (g * y64).sum(axis=axis, keepdims=True))
    scale = np.abs(wb).max()
    assert np.abs(dgi.numpy() - wb).max() <= 1e-5 * scale
    # along a transposed (non-contiguous) input
    if len(shape) == 2:
        _, vt = strided(ctx, x, (1, 0))
        do2 = ctx.array(shape=shape)
        nnhip.call("nnhip_softmax_f32", ctx.h, vt, nnhip.view(do2), axis)
        np.testing.assert_allclose(do2.numpy(), y, rtol=2e-6)


def test_embedding_gather(ctx):
    """Tensor::embedding (tensor.cpp:915-967 -> cpu_backend.cpp:998-1033):
    rows of the weight by fp32 id; ids outside [0, V) take row 0;
    a transposed index tensor."""
    rng = np.random.default_rng(4)
    V, D = 50, 24
    w = rng.standard_normal((V, D)).astype(np.float32)
    ids = rng.integers(0, V, (3, 7)).astype(np.float32)
    ids[0, 0], ids[1, 3], ids[2, 6] = 50, 1e6, -3
    ids[2, 2] = 7.6                                  # truncates to 7
    dw, di = dev(ctx, w), dev(ctx, ids)
    do = ctx.array(shape=(3, 7, D))
    nnhip.call("nnhip_embedding_f32", ctx.h, nnhip.view(dw), nnhip.view(di),
               nnhip.view(do))
    idx = ids.astype(np.int64)
    idx[(ids < 0) | (ids >= V)] = 0
    np.testing.assert_array_equal(do.numpy(), w[idx])
    _, vt = strided(ctx, ids, (1, 0))
    do2 = ctx.array(shape=(3, 7, D))
    nnhip.call("nnhip_embedding_f32", ctx.h, nnhip.view(dw), vt,
               nnhip.view(do2))
    np.testing.assert_array_equal(do2.numpy(), w[idx])


def test_slice_backward_and_fill(ctx):
    rng = np.random.default_rng(5)
    gp = rng.standard_normal((4, 6, 5)).astype(np.float32)
    gs = rng.standard_normal((4, 5)).astype(np.float32)
    dgp, dgs = dev(ctx, gp), dev(ctx, gs)
    nnhip.call("nnhip_slice_backward_f32", ctx.h, nnhip.view(dgs),
               nnhip.view(dgp), 1, 3)
    want = gp.copy()
    want[:, 3, :] += gs
    np.testing.assert_array_equal(dgp.numpy(), want)
    nnhip.call("nnhip_fill_f32", ctx.h, dgp.p, gp.size, 2.5)
    assert (dgp.numpy() == 2.5).all()


def test_non_broadcastable_operands_are_refused(ctx):
    """An operand whose right-aligned dims are neither the output's nor 1
    ([3] against [4, 5]; [2, 5] against [4, 5]) is refused with NNHIP_EARG
    on the host, before any launch: the output keeps its contents."""
    da = dev(ctx, np.ones(3, np.float32))
    db = dev(ctx, np.ones((2, 5), np.float32))
    dc = dev(ctx, np.ones((4, 5), np.float32))
    do = ctx.array(shape=(4, 5))
    nnhip.call("nnhip_fill_f32", ctx.h, do.p, 20, -3.0)
    for bad in (da, db):
        with pytest.raises(nnhip.NNHipError) as e:
            nnhip.call("nnhip_binary_f32", ctx.h, nnhip.OP_ADD, nnhip.view(bad),
                       nnhip.view(dc), nnhip.view(do))
        assert e.value.code == nnhip.EARG
        with pytest.raises(nnhip.NNHipError) as e:
            nnhip.call("nnhip_unary_f32", ctx.h, nnhip.OP_RELU,
                       nnhip.view(bad), nnhip.view(do))
        assert e.value.code == nnhip.EARG
    assert (do.numpy() == -3.0).all()


def test_softmax_backward_broadcast_grad(ctx):
    """CpuBackend::softmax_backward reads grad_out through its broadcast
    offset against the output's shape (cpu_backend.cpp:585-640): a [1, L]
    gradient against [R, L] outputs gives y * (g - sum(g * y)) per row."""
    rng = np.random.default_rng(12)
    R, L = 5, 33
    y = rng.random((R, L)).astype(np.float32)
    y /= y.sum(1, keepdims=True)
    g = rng.standard_normal((1, L)).astype(np.float32)
    dy_, dg, dx = dev(ctx, y), dev(ctx, g), ctx.array(shape=(R, L))
    nnhip.call("nnhip_softmax_backward_f32", ctx.h, nnhip.view(dy_),
               nnhip.view(dg), nnhip.view(dx), 1)
    y64 = y.astype(np.float64)
    want = y64 * (g - (g * y64).sum(1, keepdims=True))
    assert np.abs(dx.numpy() - want).max() <= 1e-5 * np.abs(want).max()

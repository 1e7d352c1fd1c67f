"""Kernel-level parity of libnnhip.so against the oracle (GPU).

Each kernel runs through the C ABI on seeded inputs and is compared with the
oracle function restating the same reference step: bit-exact for the int8
codes, the MFMA digit integers and RoPE; within 1e-4 (row-relative) for fp32
products, attention and probabilities; identical draws given the same
uniforms except at a recorded tie.
"""
import numpy as np
import pytest

import oracle_py as O
from gpu_util import (assert_as_accurate, assert_rows_close, dispatch_rules, nnhip,
                      row_rel_err)

pytestmark = pytest.mark.gpu

call = nnhip.call


def quantize_oracle(w):
    codes = np.zeros(w.shape, np.int8)
    scales = np.zeros(w.shape[1], np.float32)
    O.lib().or_quantize_w8(O.fptr(w), w.shape[0], w.shape[1], O.i8ptr(codes),
                           O.fptr(scales))
    return codes, scales


def dense_oracle(x, codes=None, scales=None, w=None, bias=None):
    rows, K = x.shape
    N = (codes if codes is not None else w).shape[1]
    y = np.zeros((rows, N), np.float32)
    O.lib().or_dense(O.fptr(x), rows, K, N,
                     O.fptr(w) if w is not None else None,
                     O.i8ptr(codes) if codes is not None else None,
                     O.fptr(scales) if scales is not None else None,
                     O.fptr(bias), O.fptr(y))
    return y


def test_quantize_w8_bit_exact(ctx):
    rng = np.random.default_rng(0)
    w = (rng.standard_normal((300, 70)) * 0.02).astype(np.float32)
    w[:, 3] = 0.0
    w[:, 9] = np.float32(0.5) * np.arange(300, dtype=np.float32) - 50
    codes_o, scales_o = quantize_oracle(w)
    dw = ctx.array(w)
    dc = ctx.array(shape=(70, 300), dtype=np.int8)
    ds = ctx.array(shape=(70,))
    call("nnhip_quantize_w8", ctx.h, dw.p, 300, 70, dc.p, ds.p)
    np.testing.assert_array_equal(dc.numpy().T, codes_o)
    np.testing.assert_array_equal(ds.numpy(), scales_o)


GEMV_SHAPES = [(1, 64, 64), (1, 256, 768), (2, 512, 1536), (3, 1024, 1024),
               (4, 1024, 4096), (5, 2048, 512), (8, 4096, 1024),
               (1, 4096, 1024), (6, 128, 320),
               # 32+ rows in 4-row groups (the draft's down projection at
               # 32 / 64 rows), and 8-row groups with a remainder launch
               (32, 512, 1536), (32, 2048, 512), (64, 2048, 512),
               (37, 2048, 512), (64, 512, 4096),
               # column counts that end inside a workgroup's columns
               (3, 512, 200), (2, 2048, 36), (5, 256, 24), (1, 4096, 12)]


@pytest.mark.parametrize("rows,K,N", GEMV_SHAPES)
def test_gemv_w8a32(ctx, rows, K, N):
    rng = np.random.default_rng(rows * 7 + K + N)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    w = (rng.standard_normal((K, N)) * 0.02).astype(np.float32)
    b = (rng.standard_normal(N) * 0.1).astype(np.float32)
    codes, scales = quantize_oracle(w)
    want = dense_oracle(x, codes, scales, bias=b)
    dx, dc = ctx.array(x), ctx.array(np.ascontiguousarray(codes.T))
    ds, db = ctx.array(scales), ctx.array(b)
    dy = ctx.array(shape=(rows, N))
    call("nnhip_linear_w8a32", ctx.h, dx.p, rows, K, dc.p, ds.p, db.p, N,
         dy.p, 1)
    got = dy.numpy()
    assert_rows_close(got, want, 1e-4, "gemv w8a32")
    exact = x.astype(np.float64) @ (codes.astype(np.float64) *
                                    scales.astype(np.float64)) + b
    assert_as_accurate(got, want, exact, what="gemv w8a32")


@pytest.mark.parametrize("rows,K,N", [(1, 64, 192), (3, 128, 512),
                                      (4, 512, 256), (7, 256, 64)])
def test_gemv_f32(ctx, rows, K, N):
    rng = np.random.default_rng(K + N)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    w = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    b = (rng.standard_normal(N) * 0.1).astype(np.float32)
    want = dense_oracle(x, w=w, bias=b)
    dx, dw = ctx.array(x), ctx.array(np.ascontiguousarray(w.T))
    db, dy = ctx.array(b), ctx.array(shape=(rows, N))
    call("nnhip_linear_f32", ctx.h, dx.p, rows, K, dw.p, db.p, N, dy.p)
    assert_rows_close(dy.numpy(), want, 1e-4, "gemv f32")


def digits_reference(x):
    """Restatement of the activation digit split: e = 22 - exponent of the
    row max, X = rint(x * 2^e), balanced base-256 digits (hi, mid, lo)."""
    mx = np.abs(x).max(axis=1)
    e = np.where(mx > 0, 22 - np.frexp(mx)[1], 0).astype(np.int32)
    X = np.rint(np.ldexp(x.astype(np.float64), e[:, None])).astype(np.int64)
    lo = ((X + 128) & 255) - 128
    t = (X - lo) >> 8
    mid = ((t + 128) & 255) - 128
    hi = (t - mid) >> 8
    assert np.abs(hi).max() <= 127
    np.testing.assert_array_equal(hi * 65536 + mid * 256 + lo, X)
    return e, hi, mid, lo


# (2048, 512, 1024): 1024 tiles of 32 x 64, the wide-tile grid (gemm_wide)
MFMA_SHAPES = [(16, 128, 64), (32, 512, 1536), (192, 1024, 3072),
               (70, 4096, 1024), (8, 256, 256), (64, 2048, 512),
               (2048, 512, 1024)]


@pytest.mark.parametrize("rows,K,N", MFMA_SHAPES)
def test_mfma_digits_int_bit_exact(ctx, rows, K, N):
    """int8 x int8 -> int32 MFMA products: the exact integer totals
    sum_k X[m,k] * code[n,k] must equal the CPU's int64 matmul."""
    rng = np.random.default_rng(rows + K * 3 + N)
    x = (rng.standard_normal((rows, K)) * 1.7).astype(np.float32)
    x[0, :] *= 1e-3                        # a row with a different exponent
    w = (rng.standard_normal((K, N)) * 0.02).astype(np.float32)
    codes, _ = quantize_oracle(w)
    e, hi, mid, lo = digits_reference(x)
    rows64 = (rows + 63) // 64 * 64
    dx, dc = ctx.array(x), ctx.array(np.ascontiguousarray(codes.T))
    dt = ctx.array(shape=(rows, N), dtype=np.int64)
    de = ctx.array(shape=(rows,), dtype=np.int32)
    dl = ctx.array(shape=(3, rows64, K), dtype=np.int8)
    call("nnhip_linear_limb_totals", ctx.h, dx.p, rows, K, dc.p, N, dt.p,
         de.p, dl.p)
    np.testing.assert_array_equal(de.numpy(), e)
    limbs = dl.numpy()
    np.testing.assert_array_equal(limbs[0, :rows], hi)
    np.testing.assert_array_equal(limbs[1, :rows], mid)
    np.testing.assert_array_equal(limbs[2, :rows], lo)
    X = hi * 65536 + mid * 256 + lo
    want = X @ codes.astype(np.int64)
    np.testing.assert_array_equal(dt.numpy(), want)


@pytest.mark.parametrize("rows,K,N", MFMA_SHAPES)
def test_mfma_linear_vs_oracle(ctx, rows, K, N):
    rng = np.random.default_rng(rows * 5 + K + N)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    w = (rng.standard_normal((K, N)) * 0.02).astype(np.float32)
    b = (rng.standard_normal(N) * 0.1).astype(np.float32)
    codes, scales = quantize_oracle(w)
    want = dense_oracle(x, codes, scales, bias=b)
    dx, dc = ctx.array(x), ctx.array(np.ascontiguousarray(codes.T))
    ds, db = ctx.array(scales), ctx.array(b)
    dy = ctx.array(shape=(rows, N))
    call("nnhip_linear_w8a32", ctx.h, dx.p, rows, K, dc.p, ds.p, db.p, N,
         dy.p, 2)
    got = dy.numpy()
    assert_rows_close(got, want, 1e-4, "mfma w8a32")
    exact = x.astype(np.float64) @ (codes.astype(np.float64) *
                                    scales.astype(np.float64)) + b
    assert_as_accurate(got, want, exact, what="mfma w8a32")


LDS_SHAPES = [(16, 128, 64), (32, 512, 1536), (192, 1024, 3072),
              (5, 256, 96), (40, 1024, 32000), (64, 512, 4096),
              (33, 128, 160), (2048, 512, 1024)]


def linear_path(ctx, x, codes, scales, b, path):
    rows, K = x.shape
    N = codes.shape[1]
    dx, dc = ctx.array(x), ctx.array(np.ascontiguousarray(codes.T))
    ds, db = ctx.array(scales), ctx.array(b)
    dy = ctx.array(shape=(rows, N))
    call("nnhip_linear_w8a32", ctx.h, dx.p, rows, K, dc.p, ds.p, db.p, N,
         dy.p, path)
    return dy.numpy()


def test_linear_w8a32_scratch_reuse():
    """nnhip_linear_w8a32 on a fresh context, calls queued back to back with
    nothing read in between: the context's scratch grows (after the stream
    drains) from a small call to larger ones and is reused by a small one
    again; every output equals the same call made alone on the oracle's
    terms."""
    c = nnhip.Context(0)
    cases = [(16, 128, 64, 2), (192, 1024, 1024, 2), (64, 512, 4096, 3),
             (192, 1024, 3072, 4), (32, 512, 512, 2)]
    keep, arrays = [], []
    try:
        for i, (rows, K, N, path) in enumerate(cases):
            rng = np.random.default_rng(100 + i)
            x = rng.standard_normal((rows, K)).astype(np.float32)
            w = (rng.standard_normal((K, N)) * 0.02).astype(np.float32)
            b = (rng.standard_normal(N) * 0.1).astype(np.float32)
            codes, scales = quantize_oracle(w)
            dx, dc = c.array(x), c.array(np.ascontiguousarray(codes.T))
            ds, db = c.array(scales), c.array(b)
            dy = c.array(shape=(rows, N))
            arrays += [dx, dc, ds, db, dy]
            call("nnhip_linear_w8a32", c.h, dx.p, rows, K, dc.p, ds.p, db.p,
                 N, dy.p, path)
            keep.append((x, codes, scales, b, dy))
        for i, (x, codes, scales, b, dy) in enumerate(keep):
            want = dense_oracle(x, codes, scales, bias=b)
            assert_rows_close(dy.numpy(), want, 1e-4, f"scratch reuse case {i}")
    finally:
        for a in arrays:
            a.free()
        c.close()


@pytest.mark.parametrize("rows,K,N", LDS_SHAPES)
def test_lds_gemm_matches_digit_gemm(ctx, rows, K, N):
    """The LDS-resident GEMM (digits formed in its prologue, path 3, or read
    from digit planes, path 4) computes the same exact integers and the same
    epilogue as the digit-plane GEMM: bit-identical outputs, and within the
    oracle's accuracy."""
    rng = np.random.default_rng(rows * 7 + K + N)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    x[0] *= 1e-3
    w = (rng.standard_normal((K, N)) * 0.02).astype(np.float32)
    b = (rng.standard_normal(N) * 0.1).astype(np.float32)
    codes, scales = quantize_oracle(w)
    g3 = linear_path(ctx, x, codes, scales, b, 3)
    g4 = linear_path(ctx, x, codes, scales, b, 4)
    np.testing.assert_array_equal(g3, g4)
    if N % 64 == 0:
        np.testing.assert_array_equal(g3, linear_path(ctx, x, codes, scales, b, 2))
    want = dense_oracle(x, codes, scales, bias=b)
    assert_rows_close(g3, want, 1e-4, "lds gemm")
    exact = x.astype(np.float64) @ (codes.astype(np.float64) *
                                    scales.astype(np.float64)) + b
    assert_as_accurate(g3, want, exact, what="lds gemm")


@pytest.mark.parametrize("rows,K,N", [(32, 512, 1536), (192, 1024, 8192),
                                      (20, 128, 256), (7, 256, 64),
                                      (1, 512, 2048), (5, 1024, 512)])
def test_layernorm_linear_vs_oracle(ctx, rows, K, N):
    """LayerNorm fused into the GEMM prologue (rows below 16: the GEMV's
    prologue): LN(h) against the oracle's layernorm, y against the oracle's
    dense over the oracle's LN(h)."""
    rng = np.random.default_rng(rows + K + 3 * N)
    h = (rng.standard_normal((rows, K)) * 2 + 0.3).astype(np.float32)
    g = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    bt = (0.1 * rng.standard_normal(K)).astype(np.float32)
    w = (rng.standard_normal((K, N)) * 0.02).astype(np.float32)
    b = (rng.standard_normal(N) * 0.1).astype(np.float32)
    codes, scales = quantize_oracle(w)
    ln = np.zeros_like(h)
    O.lib().or_layernorm(O.fptr(h), rows, K, O.fptr(g), O.fptr(bt), 1e-5,
                         O.fptr(ln))
    want = dense_oracle(ln, codes, scales, bias=b)
    dh, dg, dbt = ctx.array(h), ctx.array(g), ctx.array(bt)
    dc, ds, db = (ctx.array(np.ascontiguousarray(codes.T)), ctx.array(scales),
                  ctx.array(b))
    dln, dy = ctx.array(shape=(rows, K)), ctx.array(shape=(rows, N))
    call("nnhip_layernorm_linear_w8a32", ctx.h, dh.p, rows, K, dg.p, dbt.p,
         dln.p, dc.p, ds.p, db.p, N, dy.p)
    assert_rows_close(dln.numpy(), ln, 1e-5, "fused layernorm")
    assert_rows_close(dy.numpy(), want, 1e-4, "layernorm linear")


def test_rope_kv_append(ctx):
    rng = np.random.default_rng(11)
    B, S, H, D, cap = 3, 5, 4, 64, 700
    pos = np.array([0, 17, 640], np.int32)
    qkv = rng.standard_normal((B * S, 3 * H * D)).astype(np.float32)
    dq = ctx.array(qkv)
    dpos = ctx.array(pos)
    qo = ctx.array(shape=(B * S, H * D))
    kc = ctx.array(np.zeros((B, H, cap, D), np.float32))
    vc = ctx.array(np.zeros((B, H, cap, D), np.float32))
    call("nnhip_rope_kv_append", ctx.h, dq.p, B, S, H, D, dpos.p, qo.p, kc.p,
         vc.p, cap)
    qg, kg, vg = qo.numpy(), kc.numpy(), vc.numpy()
    for b in range(B):
        rows = qkv[b * S:(b + 1) * S]
        for part, got in ((0, None), (1, None)):
            x = np.ascontiguousarray(
                rows[:, part * H * D:(part + 1) * H * D].reshape(S, H, D)
                .transpose(1, 0, 2))
            O.lib().or_rope(O.fptr(x), H, S, D, int(pos[b]))
            if part == 0:
                got = qg[b * S:(b + 1) * S].reshape(S, H, D).transpose(1, 0, 2)
            else:
                got = kg[b, :, pos[b]:pos[b] + S]
            np.testing.assert_array_equal(got, x)
        v = rows[:, 2 * H * D:].reshape(S, H, D).transpose(1, 0, 2)
        np.testing.assert_array_equal(vg[b, :, pos[b]:pos[b] + S], v)


@pytest.mark.parametrize("H,Hkv,D", [(8, 2, 32), (4, 4, 64), (6, 3, 16)])
def test_rope_kv_append_gqa(ctx, H, Hkv, D):
    """RoPE on q (H heads) and k (Hkv heads), v copied, into a cache of Hkv
    heads (MultiHeadAttention with num_kv_heads, layer.cpp:471-489, 593-807):
    bit-exact against or_rope; Hkv == H equals nnhip_rope_kv_append."""
    rng = np.random.default_rng(13 + H + Hkv)
    B, S, cap = 2, 4, 300
    pos = np.array([3, 250], np.int32)
    E, Ekv = H * D, Hkv * D
    qkv = rng.standard_normal((B * S, E + 2 * Ekv)).astype(np.float32)
    dq, dpos = ctx.array(qkv), ctx.array(pos)
    qo = ctx.array(shape=(B * S, E))
    kc = ctx.array(np.zeros((B, Hkv, cap, D), np.float32))
    vc = ctx.array(np.zeros((B, Hkv, cap, D), np.float32))
    call("nnhip_rope_kv_append_gqa", ctx.h, dq.p, B, S, H, Hkv, D, dpos.p,
         qo.p, kc.p, vc.p, cap)
    qg, kg, vg = qo.numpy(), kc.numpy(), vc.numpy()
    for b in range(B):
        rows = qkv[b * S:(b + 1) * S]
        q = np.ascontiguousarray(rows[:, :E].reshape(S, H, D).transpose(1, 0, 2))
        O.lib().or_rope(O.fptr(q), H, S, D, int(pos[b]))
        np.testing.assert_array_equal(
            qg[b * S:(b + 1) * S].reshape(S, H, D).transpose(1, 0, 2), q)
        k = np.ascontiguousarray(
            rows[:, E:E + Ekv].reshape(S, Hkv, D).transpose(1, 0, 2))
        O.lib().or_rope(O.fptr(k), Hkv, S, D, int(pos[b]))
        np.testing.assert_array_equal(kg[b, :, pos[b]:pos[b] + S], k)
        v = rows[:, E + Ekv:].reshape(S, Hkv, D).transpose(1, 0, 2)
        np.testing.assert_array_equal(vg[b, :, pos[b]:pos[b] + S], v)
    if H == Hkv:
        q2 = ctx.array(shape=(B * S, E))
        k2 = ctx.array(np.zeros((B, H, cap, D), np.float32))
        v2 = ctx.array(np.zeros((B, H, cap, D), np.float32))
        call("nnhip_rope_kv_append", ctx.h, dq.p, B, S, H, D, dpos.p, q2.p,
             k2.p, v2.p, cap)
        np.testing.assert_array_equal(q2.numpy(), qg)
        np.testing.assert_array_equal(k2.numpy(), kg)
        np.testing.assert_array_equal(v2.numpy(), vg)


ATTN_CASES = [(3, 1, 4, 64, [0, 37, 300]), (2, 6, 4, 64, [5, 380]),
              (2, 8, 2, 32, [0, 900]), (2, 13, 2, 64, [0, 20]),
              (16, 8, 8, 64, [2048] * 16)]


@pytest.mark.parametrize("w4", [0, 1])
@pytest.mark.parametrize("B,S,H,D,pos0", ATTN_CASES)
def test_attention_kq(ctx, B, S, H, D, pos0, w4):
    """k-query causal attention against the oracle; w4 = 1 runs the 4-wave
    merged workgroups for rows of 4+ queries."""
    rng = np.random.default_rng(B * 100 + S + D)
    pos0 = np.array(pos0, np.int32)
    cap = int(pos0.max()) + S
    q = rng.standard_normal((B * S, H * D)).astype(np.float32)
    k = rng.standard_normal((B, H, cap, D)).astype(np.float32)
    v = rng.standard_normal((B, H, cap, D)).astype(np.float32)
    dq, dk, dv = ctx.array(q), ctx.array(k), ctx.array(v)
    dp, do = ctx.array(pos0), ctx.array(shape=(B * S, H * D))
    try:
        ctx.set_option("attn_w4", 2 * w4)
        call("nnhip_attention_kq", ctx.h, dq.p, dk.p, dv.p, cap, dp.p, B, S, H, H,
             D, do.p)
    finally:
        ctx.set_option("attn_w4", 1)
    got = do.numpy()
    for b in range(B):
        St = int(pos0[b]) + S
        qb = np.ascontiguousarray(q[b * S:(b + 1) * S].reshape(S, H, D)
                                  .transpose(1, 0, 2))
        kb = np.ascontiguousarray(k[b, :, :St])
        vb = np.ascontiguousarray(v[b, :, :St])
        out = np.zeros((S, H, D), np.float32)
        O.lib().or_attention(O.fptr(qb), O.fptr(kb), O.fptr(vb), H, H, S, St,
                             D, 1, O.fptr(out))
        assert_rows_close(got[b * S:(b + 1) * S].reshape(S, H * D),
                          out.reshape(S, H * D), 1e-4, f"attention seq {b}")


def attention_case(ctx, B, S, H, D, pos0, q8, seed):
    """One attention launch (fp32 or int8 cache, H_kv = H) against the
    oracle's or_attention / or_attention_q8."""
    rng = np.random.default_rng(seed)
    pos0 = np.array(pos0, np.int32)
    cap = int(pos0.max()) + S
    q = rng.standard_normal((B * S, H * D)).astype(np.float32)
    dq, dp = ctx.array(q), ctx.array(pos0)
    do = ctx.array(shape=(B * S, H * D))
    if q8:
        kq = rng.integers(-127, 128, (B, H, cap, D)).astype(np.int8)
        vq = rng.integers(-127, 128, (B, H, cap, D)).astype(np.int8)
        ks = (rng.random((B, H, cap)) * 0.03 + 0.001).astype(np.float32)
        vs = (rng.random((B, H, cap)) * 0.03 + 0.001).astype(np.float32)
        dkq, dvq, dks, dvs = ctx.array(kq), ctx.array(vq), ctx.array(ks), ctx.array(vs)
        call("nnhip_attention_kq_q8", ctx.h, dq.p, dkq.p, dks.p, dvq.p, dvs.p,
             cap, dp.p, B, S, H, H, D, do.p)
    else:
        k = rng.standard_normal((B, H, cap, D)).astype(np.float32)
        v = rng.standard_normal((B, H, cap, D)).astype(np.float32)
        dk, dv = ctx.array(k), ctx.array(v)
        call("nnhip_attention_kq", ctx.h, dq.p, dk.p, dv.p, cap, dp.p, B, S, H, H,
             D, do.p)
    got = do.numpy()
    for b in range(B):
        St = int(pos0[b]) + S
        qb = np.ascontiguousarray(q[b * S:(b + 1) * S].reshape(S, H, D)
                                  .transpose(1, 0, 2))
        if q8:
            out = O.attention_q8(qb, kq[b, :, :St], ks[b, :, :St], vq[b, :, :St],
                                 vs[b, :, :St])
        else:
            out = np.zeros((S, H, D), np.float32)
            O.lib().or_attention(O.fptr(qb), O.fptr(np.ascontiguousarray(k[b, :, :St])),
                                 O.fptr(np.ascontiguousarray(v[b, :, :St])), H, H, S,
                                 St, D, 1, O.fptr(out))
        assert_rows_close(got[b * S:(b + 1) * S].reshape(S, H * D),
                          out.reshape(S, H * D), 1e-4, f"attention seq {b}")


@pytest.mark.parametrize("q8", [False, True])
@pytest.mark.parametrize("qblk", [1, 2, 4, 8])
def test_attention_short_launch_query_blocks(ctx, qblk, q8):
    """A launch of few (sequence, head) pairs takes its queries in blocks of
    the option attn_short_q (one workgroup per block): 5 and 8 queries per
    sequence over fp32 and int8 caches against the oracle, for every block
    size."""
    ctx.set_option("attn_short_q", qblk)
    try:
        for B, S, H, pos0 in ((1, 5, 8, [300]), (2, 8, 4, [0, 411])):
            attention_case(ctx, B, S, H, 64, pos0, q8, seed=qblk * 10 + S)
    finally:
        ctx.set_option("attn_short_q", 1)


# prompts: tiles of 32 positions and chunks of 32 keys dealt to 4 waves:
# remainders of both, a chunk per wave and more, ragged pasts (up to `past`),
# every head dim, grouped heads, pair counts that are a multiple of 8 and not;
# each with the 160 tiles of all pairs that the kernel starts at
PROMPT_CASES = [(10, 20, 16, 16, 64, 0), (5, 31, 32, 32, 64, 3), (3, 33, 32, 8, 64, 97),
                (3, 130, 12, 3, 64, 500), (2, 257, 10, 5, 32, 900), (14, 64, 6, 3, 40, 64),
                (21, 45, 4, 2, 8, 19), (9, 70, 6, 3, 16, 5), (10, 40, 8, 4, 24, 33),
                (14, 63, 6, 2, 48, 2), (8, 129, 4, 4, 56, 1000),
                # 64 dims over more than 1024 keys: fp32 scores of int8 rows
                (2, 130, 16, 16, 64, 1000), (3, 100, 16, 4, 64, 1500)]


@pytest.mark.parametrize("q8", [False, True])
@pytest.mark.parametrize("B,S,H,Hkv,D,past", PROMPT_CASES)
def test_attention_prompt(ctx, B, S, H, Hkv, D, past, q8):
    """Prompt launches against the oracle, the caches' unused rows NaN, and
    one V value infinite at a key that only the later positions see.  Bound:
    a log2 score here is at most about 12 (unit normal q, k of 64 dims, sum
    |q k| / 8 * 1.44), formed with about 12 roundings of 2^-24 on each side:
    9e-6, so 6e-6 of a probability, twice."""
    rng = np.random.default_rng(S * 100 + D + q8)
    pos0 = rng.integers(0, past + 1, B).astype(np.int32)
    pos0[-1] = past
    cap = int(pos0.max()) + S + 5
    assert dispatch_rules().attention_prompt_shape(B, S, H, D, q8, cap)
    late = S - 3                       # the new position of the infinite value
    q = rng.standard_normal((B * S, H * D)).astype(np.float32)
    dq, dp = ctx.array(q), ctx.array(pos0)
    do = ctx.array(shape=(B * S, H * D))
    if q8:
        k = rng.integers(-127, 128, (B, Hkv, cap, D)).astype(np.int8)
        v = rng.integers(-127, 128, (B, Hkv, cap, D)).astype(np.int8)
        v[v == 0] = 1                  # a code times an infinite scale is infinite
        ks, vs = ((rng.random((B, Hkv, cap)) * 0.01 + 0.005).astype(np.float32)
                  for _ in range(2))
        for b in range(B):
            ks[b, :, pos0[b] + S:] = vs[b, :, pos0[b] + S:] = np.nan
        vs[0, 0, pos0[0] + late] = np.inf
        dk, dks, dv, dvs = (ctx.array(a) for a in (k, ks, v, vs))
        call("nnhip_attention_kq_q8", ctx.h, dq.p, dk.p, dks.p, dv.p, dvs.p, cap,
             dp.p, B, S, H, Hkv, D, do.p)
        k = k.astype(np.float32) * ks[..., None]
        v = v.astype(np.float32) * vs[..., None]
    else:
        k = rng.standard_normal((B, Hkv, cap, D)).astype(np.float32)
        v = rng.standard_normal((B, Hkv, cap, D)).astype(np.float32)
        for b in range(B):
            k[b, :, pos0[b] + S:] = v[b, :, pos0[b] + S:] = np.nan
        v[0, 0, pos0[0] + late, D // 2] = np.inf
        dk, dv = ctx.array(k), ctx.array(v)
        call("nnhip_attention_kq", ctx.h, dq.p, dk.p, dv.p, cap, dp.p, B, S, H, Hkv,
             D, do.p)
    got = do.numpy().reshape(B, S, H, D)
    for b in range(B):
        St = int(pos0[b]) + S
        kb, vb = (np.ascontiguousarray(a[b, :, :St]) for a in (k, v))
        qb = np.ascontiguousarray(q[b * S:(b + 1) * S].reshape(S, H, D).transpose(1, 0, 2))
        out = np.zeros((S, H, D), np.float32)
        O.lib().or_attention(O.fptr(qb), O.fptr(kb), O.fptr(vb), H, Hkv, S, St, D, 1,
                             O.fptr(out))
        fin = np.isfinite(out)
        assert fin[:late].all() and (b or not fin[late:].all())
        np.testing.assert_array_equal(np.isfinite(got[b]), fin)
        assert_rows_close(np.where(fin, got[b], 0).reshape(S, H * D),
                          np.where(fin, out, 0).reshape(S, H * D), 1.2e-5, f"seq {b}")


# grouped-query attention (MultiHeadAttention's num_kv_heads, layer.cpp:
# 862-864: query head h reads kv head h / (H / H_kv)): the shapes of
# gqa_test.cpp:115-211 (4 heads on 2 kv heads, B = 2 x 3 queries, and one
# query over a growing cache) at head dim 8 (the device's smallest), the
# batch-32 verify shape on 4 kv heads, and multi-query attention (H_kv = 1)
GQA_CASES = [(2, 3, 4, 2, 8, [0, 0]), (1, 1, 4, 2, 8, [1]),
             (3, 6, 16, 4, 64, [100, 300, 7]), (2, 8, 8, 1, 64, [2048, 17])]


@pytest.mark.parametrize("q8", [False, True])
@pytest.mark.parametrize("B,S,H,Hkv,D,pos0", GQA_CASES)
def test_attention_gqa(ctx, B, S, H, Hkv, D, pos0, q8):
    """Grouped-query attention over fp32 and int8 caches against the
    oracle's or_attention / or_attention_q8 with H_kv < H."""
    rng = np.random.default_rng(B * 1000 + H * 10 + Hkv + q8)
    pos0 = np.array(pos0, np.int32)
    cap = int(pos0.max()) + S
    q = rng.standard_normal((B * S, H * D)).astype(np.float32)
    dq, dp = ctx.array(q), ctx.array(pos0)
    do = ctx.array(shape=(B * S, H * D))
    if q8:
        kq = rng.integers(-127, 128, (B, Hkv, cap, D)).astype(np.int8)
        vq = rng.integers(-127, 128, (B, Hkv, cap, D)).astype(np.int8)
        ks = (rng.random((B, Hkv, cap)) * 0.03 + 0.001).astype(np.float32)
        vs = (rng.random((B, Hkv, cap)) * 0.03 + 0.001).astype(np.float32)
        dk, dv, dks, dvs = ctx.array(kq), ctx.array(vq), ctx.array(ks), ctx.array(vs)
        call("nnhip_attention_kq_q8", ctx.h, dq.p, dk.p, dks.p, dv.p, dvs.p,
             cap, dp.p, B, S, H, Hkv, D, do.p)
    else:
        k = rng.standard_normal((B, Hkv, cap, D)).astype(np.float32)
        v = rng.standard_normal((B, Hkv, cap, D)).astype(np.float32)
        dk, dv = ctx.array(k), ctx.array(v)
        call("nnhip_attention_kq", ctx.h, dq.p, dk.p, dv.p, cap, dp.p, B, S, H,
             Hkv, D, do.p)
    got = do.numpy()
    for b in range(B):
        St = int(pos0[b]) + S
        qb = np.ascontiguousarray(q[b * S:(b + 1) * S].reshape(S, H, D)
                                  .transpose(1, 0, 2))
        if q8:
            out = O.attention_q8(qb, kq[b, :, :St], ks[b, :, :St],
                                 vq[b, :, :St], vs[b, :, :St])
        else:
            out = np.zeros((S, H, D), np.float32)
            O.lib().or_attention(O.fptr(qb), O.fptr(np.ascontiguousarray(k[b, :, :St])),
                                 O.fptr(np.ascontiguousarray(v[b, :, :St])), H,
                                 Hkv, S, St, D, 1, O.fptr(out))
        assert_rows_close(got[b * S:(b + 1) * S].reshape(S, H * D),
                          out.reshape(S, H * D), 1e-4, f"gqa seq {b}")


@pytest.mark.parametrize("D", [64, 32, 8])
def test_rope_kv_append_q8(ctx, D):
    """RoPE + int8 append: q bit-exact with or_rope, codes and scales
    bit-exact with or_quantize_kv of the oracle's rotated k and of v."""
    rng = np.random.default_rng(12 + D)
    B, S, H, cap = 3, 5, 4, 700
    pos = np.array([0, 17, 640], np.int32)
    qkv = rng.standard_normal((B * S, 3 * H * D)).astype(np.float32)
    qkv[2, H * D:2 * H * D] = 0.0          # an all-zero k row: scale 1
    qkv[4, 2 * H * D:2 * H * D + D] = 0.5  # exact halves: round away from 0
    dq, dpos = ctx.array(qkv), ctx.array(pos)
    qo = ctx.array(shape=(B * S, H * D))
    kq = ctx.array(np.zeros((B, H, cap, D), np.int8))
    vq = ctx.array(np.zeros((B, H, cap, D), np.int8))
    ks = ctx.array(np.zeros((B, H, cap), np.float32))
    vs = ctx.array(np.zeros((B, H, cap), np.float32))
    call("nnhip_rope_kv_append_q8", ctx.h, dq.p, B, S, H, D, dpos.p, qo.p,
         kq.p, ks.p, vq.p, vs.p, cap)
    qg, kqg, ksg, vqg, vsg = (qo.numpy(), kq.numpy(), ks.numpy(), vq.numpy(),
                              vs.numpy())
    for b in range(B):
        rows = qkv[b * S:(b + 1) * S]
        sl = slice(int(pos[b]), int(pos[b]) + S)
        heads = []
        for part in range(3):
            x = np.ascontiguousarray(
                rows[:, part * H * D:(part + 1) * H * D].reshape(S, H, D)
                .transpose(1, 0, 2))
            if part < 2:
                O.lib().or_rope(O.fptr(x), H, S, D, int(pos[b]))
            heads.append(x)
        np.testing.assert_array_equal(
            qg[b * S:(b + 1) * S].reshape(S, H, D).transpose(1, 0, 2), heads[0])
        kc, ksc = O.quantize_kv(heads[1])
        vc, vsc = O.quantize_kv(heads[2])
        np.testing.assert_array_equal(kqg[b, :, sl], kc)
        np.testing.assert_array_equal(ksg[b, :, sl], ksc)
        np.testing.assert_array_equal(vqg[b, :, sl], vc)
        np.testing.assert_array_equal(vsg[b, :, sl], vsc)
    # positions outside [pos, pos + S) are untouched
    assert not kqg[0, :, S:].any() and not ksg[1, :, :17].any()


ATTN_Q8_CASES = [(3, 1, 4, 64, [0, 37, 300]), (2, 6, 4, 64, [5, 380]),
                 (2, 8, 2, 32, [0, 900]), (2, 13, 2, 64, [0, 20]),
                 (2, 3, 2, 16, [7, 1200]), (16, 8, 8, 64, [2048] * 16)]


@pytest.mark.parametrize("w4", [0, 1])
@pytest.mark.parametrize("B,S,H,D,pos0", ATTN_Q8_CASES)
def test_attention_kq_q8(ctx, B, S, H, D, pos0, w4):
    """Attention over an int8 cache against or_attention_q8 (merged
    workgroups, 4-wave merged workgroups and the split + combine path)."""
    rng = np.random.default_rng(B * 100 + S + D + 7)
    pos0 = np.array(pos0, np.int32)
    cap = int(pos0.max()) + S
    q = rng.standard_normal((B * S, H * D)).astype(np.float32)
    kq = rng.integers(-127, 128, (B, H, cap, D)).astype(np.int8)
    vq = rng.integers(-127, 128, (B, H, cap, D)).astype(np.int8)
    ks = (rng.random((B, H, cap)) * 0.03 + 0.001).astype(np.float32)
    vs = (rng.random((B, H, cap)) * 0.03 + 0.001).astype(np.float32)
    dq, dkq, dvq = ctx.array(q), ctx.array(kq), ctx.array(vq)
    dks, dvs = ctx.array(ks), ctx.array(vs)
    dp, do = ctx.array(pos0), ctx.array(shape=(B * S, H * D))
    try:
        ctx.set_option("attn_w4", 2 * w4)
        call("nnhip_attention_kq_q8", ctx.h, dq.p, dkq.p, dks.p, dvq.p, dvs.p,
             cap, dp.p, B, S, H, H, D, do.p)
    finally:
        ctx.set_option("attn_w4", 1)
    got = do.numpy()
    for b in range(B):
        St = int(pos0[b]) + S
        qb = q[b * S:(b + 1) * S].reshape(S, H, D).transpose(1, 0, 2)
        out = O.attention_q8(qb, kq[b, :, :St], ks[b, :, :St], vq[b, :, :St],
                             vs[b, :, :St])
        assert_rows_close(got[b * S:(b + 1) * S].reshape(S, H * D),
                          out.reshape(S, H * D), 1e-4, f"int8 attention seq {b}")


def test_attention_kq_q8_returns_drained(ctx):
    """nnhip_attention_kq_q8 returns with its output written: read through
    another context (another stream) right away, behind milliseconds of
    earlier work on its own, it is what a read on its own stream gives."""
    B, S, H, D, cap = 2, 5, 4, 64, 400
    rng = np.random.default_rng(8)
    kv = [ctx.array(rng.integers(-127, 128, (B, H, cap, D)).astype(np.int8)) for _ in "kv"]
    sc = [ctx.array((rng.random((B, H, cap)) * 0.03).astype(np.float32)) for _ in "kv"]
    q = ctx.array(rng.standard_normal((B * S, H * D)).astype(np.float32))
    pos, out = ctx.array(np.array([390, 7], np.int32)), ctx.array(np.zeros((B * S, H * D), np.float32))
    n = 4096
    x, w, y = (ctx.array(shape=(n, n)) for _ in range(3))
    with nnhip.Context(0) as other:
        for _ in range(3):
            call("nnhip_linear_f32", ctx.h, x.p, n, n, w.p, x.p, n, y.p)
        call("nnhip_attention_kq_q8", ctx.h, q.p, kv[0].p, sc[0].p, kv[1].p, sc[1].p,
             cap, pos.p, B, S, H, H, D, out.p)
        got = np.empty((B * S, H * D), np.float32)
        call("nnhip_d2h", other.h, nnhip.ptr(got), out.p, got.nbytes)
    want = out.numpy()
    assert np.abs(want).min(1).max() > 0
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("rows,d", [(7, 64), (5, 1024), (3, 4096), (2, 100)])
def test_layernorm(ctx, rows, d):
    rng = np.random.default_rng(d)
    x = (rng.standard_normal((rows, d)) * 2 + 0.5).astype(np.float32)
    g = rng.standard_normal(d).astype(np.float32)
    b = rng.standard_normal(d).astype(np.float32)
    want = np.zeros_like(x)
    O.lib().or_layernorm(O.fptr(x), rows, d, O.fptr(g), O.fptr(b), 1e-5,
                         O.fptr(want))
    dx, dg, db = ctx.array(x), ctx.array(g), ctx.array(b)
    dy = ctx.array(shape=(rows, d))
    call("nnhip_layernorm", ctx.h, dx.p, rows, d, dg.p, db.p, dy.p)
    assert_rows_close(dy.numpy(), want, 1e-5, "layernorm")


def cdf_tie(probs, u, tol=1e-6):
    c = np.cumsum(probs.astype(np.float64) / probs.astype(np.float64).sum())
    return bool(np.min(np.abs(c - u)) < tol)


@pytest.mark.parametrize("V,T", [(256, 1.0), (4096, 0.7), (32000, 1.0),
                                 (32000, 0.0), (1000, 2.5)])
def test_sample_rows(ctx, V, T):
    B = 24
    rng = np.random.default_rng(V + int(T * 10))
    lg = (rng.standard_normal((B, V)) * 2).astype(np.float32)
    u = np.array([O.uniform(99, b, 3, 1) for b in range(B)], np.float32)
    dl, du = ctx.array(lg), ctx.array(u)
    dt = ctx.array(shape=(B,), dtype=np.int32)
    dp = ctx.array(shape=(B, V))
    call("nnhip_sample_rows", ctx.h, dl.p, B, V, T, 0, 1.0, du.p, dt.p, dp.p)
    tok = dt.numpy()
    mism = 0
    for b in range(B):
        p = O.get_probs(lg[b], T)
        if T <= 0:
            assert tok[b] == int(np.argmax(lg[b]))
            continue
        assert row_rel_err(dp.numpy()[b][None], p[None]) <= 1e-4
        want = O.sample(p, u[b])
        if tok[b] != want:
            assert cdf_tie(p, u[b]), (b, tok[b], want)
            mism += 1
    assert mism <= 1


def exact_kept(p1, top_k, top_p):
    """The kept set of get_probs' top-k / top-p with the running sum taken
    exactly (float64), descending p1, ties by lower index; returns it and
    the exact running sum at each entry's rank."""
    V = p1.size
    order = np.lexsort((np.arange(V), -p1.astype(np.float64)))
    cs = np.cumsum(p1.astype(np.float64)[order])
    R = top_k if 0 < top_k < V else V
    if 0 < top_p < 1:
        r = int(np.searchsorted(cs, top_p))       # first rank with cs >= top_p
        R = min(R, r + 1)
    kept = np.zeros(V, bool)
    kept[order[:R]] = True
    rank = np.empty_like(order)
    rank[order] = np.arange(V)
    return kept, cs[rank]


TOPKP_CASES = [(256, 1.0, 4, 1.0), (32000, 1.0, 0, 0.9), (32000, 0.7, 50, 0.9),
               (4096, 1.0, 4096, 0.5), (1000, 2.5, 0, 0.3), (32000, 1.0, 1, 1.0),
               (5000, 1.0, 7, 0.0)]


@pytest.mark.parametrize("V,T,top_k,top_p", TOPKP_CASES)
def test_sample_rows_top_k_top_p(ctx, V, T, top_k, top_p):
    """get_probs with top-k / top-p (layer.cpp:1447-1489).  The device keeps
    exactly the set the rule gives with an exact running sum (exact_kept;
    an entry may differ only where that sum is within 1e-6 of top_p, i.e.
    where p1 itself differs from the oracle's in its last bits).  The
    oracle, like the reference, sums in float in sorted order, which drifts
    (most over long runs of equal probabilities: rows 0-2 hold duplicated
    logits, so cuts fall inside groups of equal values, kept in index
    order); where its kept set differs from the device's, every differing
    entry lies between the exact and the float crossing.  Otherwise
    probabilities within 1e-4 (row-relative) and the same draws except at a
    CDF tie."""
    B = 16
    rng = np.random.default_rng(V + top_k)
    lg = (rng.standard_normal((B, V)) * 2).astype(np.float32)
    lg[0, :] = np.round(lg[0, :])                 # many exact ties
    lg[1, :V // 2] = lg[1, 0]                     # one large tie group
    lg[2, ::3] = 1.5                              # a tie group at the top
    u = np.array([O.uniform(98, b, 4, 1) for b in range(B)], np.float32)
    dl, du = ctx.array(lg), ctx.array(u)
    dt = ctx.array(shape=(B,), dtype=np.int32)
    dp = ctx.array(shape=(B, V))
    call("nnhip_sample_rows", ctx.h, dl.p, B, V, T, top_k, top_p, du.p, dt.p,
         dp.p)
    tok, got = dt.numpy(), dp.numpy()
    mism = 0
    for b in range(B):
        # p1 exactly normalised (the oracle's own float sums can drift by
        # 1e-4 on rows of many equal logits, as the reference's do)
        z = lg[b].astype(np.float64) / T
        p1 = np.exp(z - z.max())
        p1 /= p1.sum()
        want = O.get_probs(lg[b], T, top_k, top_p)
        kd, ko = got[b] > 0, want > 0
        ke, cs = exact_kept(p1, top_k, top_p)
        off = kd != ke
        assert not off.any() or np.all(np.abs(cs[off] - top_p) < 1e-6), b
        if not np.array_equal(kd, ko):
            # the oracle's float running sum crossed top_p elsewhere
            lo, hi = sorted((ko.sum(), kd.sum()))
            order = np.lexsort((np.arange(V), -p1.astype(np.float64)))
            assert set(np.nonzero(kd != ko)[0]) <= set(order[lo:hi]), b
            common = kd & ko
            ga = got[b] * common / (got[b] * common).sum()
            wa = want * common / (want * common).sum()
            assert row_rel_err(ga[None], wa[None]) <= 1e-4
            continue
        assert row_rel_err(got[b][None], want[None]) <= 1e-4, b
        if 0 < top_k < V and not (0 < top_p < 1):
            assert kd.sum() == top_k
        w = O.sample(want, u[b])
        if tok[b] != w:
            assert cdf_tie(want, u[b]), (b, tok[b], w)
            mism += 1
    assert mism <= 1


@pytest.mark.parametrize("V", [2, 1023, 4097, 32768])
@pytest.mark.parametrize("top_k,top_p", [(3, 1.0), (0, 0.6), (40, 0.95), (2000, 0.999)])
def test_filter_masked_and_equal_rows(ctx, V, top_k, top_p):
    """The filter at the edges of its digit levels: rows masked with -inf and
    with the lowest float (more kept ranks than unmasked entries: zeros in
    index order), one finite entry, all entries equal, probabilities a few
    ulps apart (in one bin of the first two levels): the kept set of the
    rule with an exact sum, entries within 1e-6 of the crossing aside.  A
    row of NaN returns a token in range."""
    rng = np.random.default_rng(V + top_k)
    lg = (rng.standard_normal((7, V)) * 3).astype(np.float32)
    lg[0, V // 3 + 1:] = -np.inf
    lg[1, 1:] = np.finfo(np.float32).min
    lg[2, :] = -np.inf
    lg[2, V // 2] = 1.0
    lg[3, :] = 0.25
    lg[4, :] = 1.0 + 1e-6 * rng.integers(0, 5, V)   # 8 ulps apart: expf keeps the order
    lg[6, V // 2] = np.nan
    u = rng.random(7).astype(np.float32)
    dl, du = ctx.array(lg), ctx.array(u)
    dt, dp = ctx.array(shape=(7,), dtype=np.int32), ctx.array(shape=(7, V))
    call("nnhip_sample_rows", ctx.h, dl.p, 7, V, 1.0, top_k, top_p, du.p, dt.p,
         dp.p)
    tok, got = dt.numpy(), dp.numpy()
    assert (tok >= 0).all() and (tok < V).all()
    for b in range(6):
        z = lg[b].astype(np.float64)
        p1 = np.exp(z - z.max())
        p1 /= p1.sum()
        ke, cs = exact_kept(p1, top_k, top_p)
        off = (got[b] > 0) != (ke & (p1 > 1e-44))
        assert not off.any() or np.all(np.abs(cs[off] - top_p) < 1e-6), b
        if not off.any():
            want = np.where(ke, p1, 0)
            assert row_rel_err(got[b][None], (want / want.sum())[None]) <= 1e-5
            assert got[b][tok[b]] > 0


def test_filter_time_of_equal_rows(ctx):
    """Rows whose entries fall into one histogram bin are not added one by one:
    a filtered call on equal rows takes about twice the time of one on random
    rows (each entry's addition waiting for the last: six times)."""
    B, V = 32, 32000
    rng = np.random.default_rng(1)
    rows = [ctx.array(a.astype(np.float32)) for a in
            (rng.standard_normal((B, V)) * 2.5, np.zeros((B, V)))]
    du, dt, dp = ctx.array(shape=(B,)), ctx.array(shape=(B,), dtype=np.int32), ctx.array(shape=(B, V))
    call("nnhip_fill_f32", ctx.h, du.p, B, 0.5)

    def ms(dl):
        for n in (3, 20):
            ctx.timer_begin()
            for _ in range(n):
                call("nnhip_sample_rows", ctx.h, dl.p, B, V, 0.8, 0, 0.9, du.p, dt.p, dp.p)
            t = ctx.timer_end() / n
        return t
    times = [[ms(dl) for dl in rows] for _ in range(3)]
    assert min(e / r for r, e in times) <= 3.5, times


def accept_case(ctx, B, k, V, T, corr, seed):
    rng = np.random.default_rng(seed)
    tl = (rng.standard_normal((B, k, V)) * 2).astype(np.float32)
    dl = (corr * tl + (1 - corr) * rng.standard_normal((B, k, V)) * 2
          ).astype(np.float32)
    ua = rng.random((B, k)).astype(np.float32)
    ur = rng.random(B).astype(np.float32)
    dtok = np.zeros((B, k), np.int32)
    for b in range(B):
        for j in range(k):
            q = O.get_probs(dl[b, j], T if T > 0 else 1.0)
            dtok[b, j] = O.sample(q, rng.random())
    dt_, dd, dk = ctx.array(tl), ctx.array(dl), ctx.array(dtok)
    dua, dur = ctx.array(ua), ctx.array(ur)
    dn = ctx.array(shape=(B,), dtype=np.int32)
    dx = ctx.array(shape=(B,), dtype=np.int32)
    call("nnhip_spec_accept", ctx.h, dt_.p, dd.p, dk.p, dua.p, dur.p, B, k, V,
         T, dn.p, dx.p)
    n_gpu, tok_gpu = dn.numpy(), dx.numpy()
    ties = 0
    for b in range(B):
        p = np.stack([O.get_probs(tl[b, j], T) for j in range(k)])
        q = np.stack([O.get_probs(dl[b, j], T) for j in range(k)])
        n, tok, nt = O.accept_step(p, q, dtok[b], T <= 0, False, ua[b], ur[b])
        if (n, tok) != (int(n_gpu[b]), int(tok_gpu[b])):
            # allowed only where the oracle met an accept or CDF tie
            j = min(n, int(n_gpu[b]))
            r = ua[b, j] if j < k else 0
            at_tie = nt > 0 or (j < k and abs(
                r - p[j, dtok[b, j]] / q[j, dtok[b, j]]) < 1e-6)
            if not at_tie and n == int(n_gpu[b]) and n < k:
                rec = np.maximum(0, p[n] - q[n])
                at_tie = cdf_tie(rec if rec.sum() > 0 else p[n], ur[b])
            assert at_tie, (b, n, tok, n_gpu[b], tok_gpu[b])
            ties += 1
    return n_gpu, ties


@pytest.mark.parametrize("T,corr", [(1.0, 0.0), (1.0, 0.97), (0.0, 0.9)])
def test_spec_accept_vs_oracle(ctx, T, corr):
    n, ties = accept_case(ctx, 48, 8, 32000, T, corr, seed=int(corr * 100))
    assert ties <= 1
    if corr > 0.9 and T > 0:
        assert n.max() >= 3          # the correlated case accepts runs


def test_spec_accept_kept_state_across_sizes(ctx):
    """nnhip_spec_accept keeps its state and scratch in the context for the
    next call of the same (B, k, V): calls of sizes A, B, A again and of A
    at another temperature on one context each agree with the oracle, and
    the repeated call with A's inputs gives A's first results."""
    n1, t1 = accept_case(ctx, 24, 6, 5000, 1.0, 0.9, seed=5)
    n2, t2 = accept_case(ctx, 8, 3, 700, 0.8, 0.9, seed=6)
    n3, t3 = accept_case(ctx, 24, 6, 5000, 1.0, 0.9, seed=5)
    n4, t4 = accept_case(ctx, 24, 6, 5000, 0.0, 0.9, seed=7)
    np.testing.assert_array_equal(n1, n3)
    assert t1 + t2 + t3 + t4 <= 2


@pytest.mark.parametrize("V", [4097, 1000, 130])
def test_spec_accept_odd_vocab(ctx, V):
    """Vocabularies whose rows are not 8-byte aligned (odd V: the draft
    statistics read single columns) or end inside a run of tiles."""
    n, ties = accept_case(ctx, 16, 4, V, 0.7, 0.9, seed=V)
    assert ties <= 1


def _linear_rows(ctx, x, codes, sc, b, path, step):
    """nnhip_linear_w8a32 over x in slices of `step` rows."""
    dc, ds, db = ctx.array(codes), ctx.array(sc), ctx.array(b)
    out = []
    for r in range(0, len(x), step):
        dx = ctx.array(x[r:r + step])
        y = ctx.array(shape=(len(x[r:r + step]), len(codes)))
        nnhip.call("nnhip_linear_w8a32", ctx.h, dx.p, y.shape[0], x.shape[1],
                   dc.p, ds.p, db.p, len(codes), y.p, path)
        out.append(y.numpy())
    return np.concatenate(out)


@pytest.mark.parametrize("rows,K,N", [
    (12 * 128 - 127, 128, 8 * 256),        # 96 tiles, the last with one row
    (4 * 128, 256, 23 * 256 + 64),         # a last column tile of 64
    (1000, 384, 3072), (2050, 512, 1536), (200, 1024, 12288),
    (8 * 128 + 37, 4096, 12 * 256 - 64),
    (64, 128, 96 * 256), (70, 512, 128 * 256 - 64)])   # half a row tile
def test_tall_gemm_matches_short_slices(ctx, rows, K, N):
    """The 128 x 256-tile GEMM forms the same exact digit totals and the same
    rounding as the GEMMs of short inputs, so its rows are bit for bit those of
    32-row slices; against float64 within the digit resolution (2^-22 of a row's
    maximum per entry)."""
    assert dispatch_rules().gemm_tall_shape(rows, K, N, 0)
    assert not dispatch_rules().gemm_tall_shape(32, K, N, 0)
    rng = np.random.default_rng(rows + K)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    x[::7] *= 1e-3
    x[5] = 0
    codes = rng.integers(-127, 128, (N, K)).astype(np.int8)
    sc = (rng.random(N) * 0.01 + 1e-4).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    got = _linear_rows(ctx, x, codes, sc, b, 2, rows)
    np.testing.assert_array_equal(got, _linear_rows(ctx, x, codes, sc, b, 2, 32))
    pick = np.r_[0, 5, 7, rows - 1]
    w = codes.astype(np.float64) * sc[:, None]
    ex = x[pick].astype(np.float64) @ w.T + b
    # each entry is off by at most half a digit unit, max|x| 2^-22 (the row
    # exponent keeps |X| < 2^22, at least 2^21); then one fp32 rounding
    tol = (np.abs(x[pick]).max(1) * 2.0 ** -21)[:, None] * np.abs(w).sum(1) + \
        np.abs(ex) * 2.0 ** -23 + np.abs(b) * 2.0 ** -23 + 1e-30
    assert (np.abs(got[pick] - ex) <= tol).all()


def test_tall_layernorm_linear(ctx):
    """nnhip_layernorm_linear_w8a32 on a tall input (one LayerNorm launch,
    then the 128 x 256-tile GEMM), with and without ln_out, against float64."""
    rows, K, N = 1570, 512, 2048
    assert dispatch_rules().gemm_tall_shape(rows, K, N, 1)
    rng = np.random.default_rng(3)
    h = (rng.standard_normal((rows, K)) + 0.2).astype(np.float32)
    g = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    be = (0.1 * rng.standard_normal(K)).astype(np.float32)
    codes = rng.integers(-127, 128, (N, K)).astype(np.int8)
    sc = np.full(N, 0.002, np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    a = [ctx.array(v) for v in (h, g, be, codes, sc, b)]
    ys = []
    ln, y = ctx.array(shape=(rows, K)), ctx.array(shape=(rows, N))
    for out in (ln.p, None):
        nnhip.call("nnhip_layernorm_linear_w8a32", ctx.h, a[0].p, rows, K,
                   a[1].p, a[2].p, out, a[3].p, a[4].p, a[5].p, N, y.p)
        ys.append(y.numpy())
    np.testing.assert_array_equal(ys[0], ys[1])
    h64 = h.astype(np.float64)
    hc = h64 - h64.mean(1, keepdims=True)
    ex = hc / np.sqrt((hc ** 2).mean(1, keepdims=True) + 1e-5) * g + be
    # LayerNorm: three roundings of values below ~5 and the sums' own errors
    assert np.abs(ln.numpy() - ex).max() <= 4e-6
    exy = ex @ (codes.astype(np.float64) * 0.002).T + b
    # the digits' 2^-22 of the row maximum per entry and ln's 4e-6, random
    # signs over K entries of |w| <= 0.254
    assert np.abs(ys[0] - exy).max() <= 5e-6 * 0.254 * np.sqrt(K) * 6


@pytest.mark.parametrize("d,B,S,q8,tall", [
    (512, 9, 300, False, "qkv gu"), (512, 4, 293, False, "gu"), (512, 9, 300, True, "gu"),
    (1024, 11, 282, False, "qkv o gu down lm"), (1024, 11, 282, True, "o gu down lm")])
def test_tall_forward_matches_short_batches(ctx, d, B, S, q8, tall):
    """A prompt forward whose projections run on the 128 x 256-tile GEMM (RoPE,
    residual, SwiGLU and bias epilogues over ragged last row tiles; `tall` names
    the products that do) gives its first and last sequence the logits and cache
    rows they get as a batch of two (GEMMs of short inputs): the products are
    bit-identical, attention and norms are per sequence.  Two sequences of 9
    position tiles are enough for the attention's MFMA kernel, so both sides run
    it: a sequence alone would run the split-K kernel, whose other rounding
    (1.4e-7 of a row each, from float64) flips codes of an int8 cache."""
    H, F, V, L = d // 64, 4 * d if d == 512 else 768, 640 if d == 512 else 1056, 2
    rules, rows = dispatch_rules(), B * S
    # an int8 append is not in the tall GEMM's epilogue; the down projection's
    # other kernel is the digit-plane GEMM, the rest's the LDS-resident one
    shapes = dict(qkv=(d, 3 * d, 1), o=(d, d, 1), gu=(d, 2 * F, 1), down=(F, d, 0), lm=(d, V, 1))
    assert tall.split() == [n for n, (K, N, lds) in shapes.items() if not (q8 and n == "qkv")
                            and rules.gemm_tall_shape(rows, K, N, lds)]
    assert not any(rules.gemm_tall_shape(2 * S, K, N, lds) for K, N, lds in shapes.values())
    for b in (2, B):
        assert rules.attention_prompt_shape(b, S, H, 64, q8, S)
    m = nnhip.Decoder(ctx, V, d, H, F, L, 512)
    m.init_normal(5, 0.05)
    m.quantize()
    ids = np.random.default_rng(S).integers(0, V, (B, S)).astype(np.int32)
    many = nnhip.KVCache(m, B, q8)
    got = m.forward(ids, many)
    two = nnhip.KVCache(m, 2, q8)
    want = m.forward(ids[[0, B - 1]], two)
    for i, b in enumerate((0, B - 1)):
        np.testing.assert_allclose(got[b], want[i], rtol=0,
                                   atol=2e-6 * np.abs(want[i]).max())
        read = (lambda c, i: c.read_q8(1, i, H, 64)) if q8 else \
            (lambda c, i: c.read(1, i, H, 64))
        for u, v in zip(read(many, b), read(two, i)):
            if u.dtype == np.int8:
                assert (u != v).mean() <= 1e-4
            else:
                np.testing.assert_allclose(u, v, rtol=0, atol=2e-6 * np.abs(v).max())
    two.free()
    many.free()
    m.free()


@pytest.mark.parametrize("q8", [False, True])
@pytest.mark.parametrize("rows,K,N", [
    # 64 x 64 tiles, K below 64: remainders of rows, columns and K steps
    (1000, 60, 91), (1000, 4, 91),
    # 32 x 32 tiles over 4 waves, K from 64 on, then over 8 (256 tiles or fewer)
    (1407, 64, 64), (301, 252, 301),
    (333, 260, 1544), (500, 772, 1001), (40, 508, 2251), (97, 1000, 929),
    (16, 4096, 5625), (352, 4092, 257),
    # 64 x 64 tiles of a large product
    (1409, 256, 1409)])
def test_linear_mfma_f32(ctx, rows, K, N, q8):
    """The fp32 MFMA GEMM of tall fp32 (and odd-shaped int8) inputs: within
    the rounding of its sums of float64 (chains of 8 products, two pairwise
    levels, then double and one rounding: 11 roundings at most, each 2^-24 of
    the row's sum of |x w|), and no further from it than the GEMV's rows."""
    assert dispatch_rules().gemm_f32_shape(rows, N)
    rng = np.random.default_rng(rows * 7 + K)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    dx, db, y = ctx.array(x), ctx.array(b), ctx.array(shape=(rows, N))
    few = min(rows, 8)
    y8 = ctx.array(shape=(few, N))
    if q8:
        w8 = rng.integers(-127, 128, (N, K)).astype(np.int8)
        sc = (rng.random(N) * 0.01 + 1e-4).astype(np.float32)
        w = w8.astype(np.float64) * sc[:, None]
        dw, ds = ctx.array(w8), ctx.array(sc)
        for r, o in ((rows, y), (few, y8)):
            call("nnhip_linear_w8a32", ctx.h, dx.p, r, K, dw.p, ds.p, db.p, N, o.p, 1)
    else:
        wf = (rng.standard_normal((N, K)) * 0.05).astype(np.float32)
        w = wf.astype(np.float64)
        dw = ctx.array(wf)
        for r, o in ((rows, y), (few, y8)):
            call("nnhip_linear_f32", ctx.h, dx.p, r, K, dw.p, db.p, N, o.p)
    got = y.numpy()
    ex = x.astype(np.float64) @ w.T + b
    size = np.abs(x).astype(np.float64) @ np.abs(w).T + np.abs(b)
    assert (np.abs(got - ex) <= 11 * 2.0 ** -24 * size).all()
    err = np.linalg.norm(got - ex) / np.linalg.norm(ex)
    gemv = np.linalg.norm(y8.numpy() - ex[:few]) / np.linalg.norm(ex[:few])
    assert err <= 1.1 * gemv + 2e-9, (err, gemv)


def test_linear_mfma_f32_inf_nan(ctx):
    """Infinities and NaN of one row or column stay in it."""
    rows, K, N = 400, 300, 300
    x, w = np.ones((rows, K), np.float32), np.full((N, K), 0.5, np.float32)
    x[3, 7], x[5, 1], w[9, 2] = np.inf, np.nan, -np.inf
    b = np.zeros(N, np.float32)
    a = [ctx.array(v) for v in (x, w, b)]
    y = ctx.array(shape=(rows, N))
    call("nnhip_linear_f32", ctx.h, a[0].p, rows, K, a[1].p, a[2].p, N, y.p)
    with np.errstate(invalid="ignore"):
        ex = x.astype(np.float64) @ w.T
    np.testing.assert_array_equal(y.numpy(), ex.astype(np.float32))


@pytest.mark.parametrize("d,H,F,B,S,waves", [
    # RoPE, residual, SwiGLU, residual of the down projection, bias: the tile of
    # each (waves over K; 0 the 64 x 64 tiles, -1 the GEMV)
    (192, 6, 300, 3, 130, (4, -1, 4, -1, 4)), (192, 6, 300, 6, 67, (4, -1, 4, -1, 4)),
    (256, 8, 300, 3, 130, (4, 4, 4, 4, 4)), (512, 8, 300, 2, 95, (4, 8, 8, 4, -1)),
    (512, 8, 600, 3, 60, (4, 8, 8, 8, -1)), (512, 8, 300, 3, 50, (8, -1, 8, -1, -1)),
    (48, 6, 100, 8, 240, (0, 0, 0, 4, 0))])
def test_unquantised_forward_tall(ctx, d, H, F, B, S, waves):
    """A prompt forward of an fp32 model, its projections on the fp32 MFMA GEMM
    with every epilogue over every tile of it, against the oracle."""
    V, L, rules, rows = 300, 2, dispatch_rules(), B * S
    assert waves == tuple(rules.gemm_f32_waves(rows, K, N) if rules.gemm_f32_shape(rows, N) else -1
                          for K, N in ((d, 3 * d), (d, d), (d, 2 * F), (F, d), (d, V)))
    p = O.make_params(V, d, H, F, L, 11, std=0.1)
    m = nnhip.Decoder(ctx, V, d, H, F, L, 256)
    m.set_params(p)
    o = O.Model(V, d, H, F, L, 256, p, False)
    ids = np.random.default_rng(B).integers(0, V, (B, S)).astype(np.int32)
    got = m.forward(ids)
    for b in range(B):
        assert_rows_close(got[b], o.forward(ids[b]), what=f"sequence {b}")
    m.free()


@pytest.mark.parametrize("q8", [False, True])
def test_prompt_after_1024_keys(ctx, q8):
    """A quantised model's prompt of 150 ids after 900 cached ones: over more
    than 1024 keys the attention's MFMA kernel is followed by a launch that
    digitises its rows for the output projection.  An fp32 cache against the
    oracle, an int8 one against its sequences one by one (split-K kernel and
    combine)."""
    V, d, H, F, L, B, past, S = 200, 256, 4, 512, 1, 8, 900, 150
    rules = dispatch_rules()
    assert rules.attention_prompt_shape(B, S, H, 64, q8, past + S)
    assert not rules.attention_prompt_shape(1, S, H, 64, q8, past + S)
    p = O.make_params(V, d, H, F, L, 5, std=0.1)
    m = nnhip.Decoder(ctx, V, d, H, F, L, 1100)
    m.set_params(p)
    m.quantize()
    ids = np.random.default_rng(3).integers(0, V, (B, past + S)).astype(np.int32)
    cache = nnhip.KVCache(m, B, q8)
    m.forward(ids[:, :past], cache)
    got = m.forward(ids[:, past:], cache)
    cache.free()
    o = None if q8 else O.Model(V, d, H, F, L, 1100, p, True)
    for b in (0, B - 1):
        if q8:
            one = nnhip.KVCache(m, 1, True)
            m.forward(ids[b:b + 1, :past], one)
            want = m.forward(ids[b:b + 1, past:], one)[0]
            one.free()
        else:
            want = o.forward(ids[b])[past:]
        assert_rows_close(got[b], want, what=f"sequence {b}")
    m.free()

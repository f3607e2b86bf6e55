"""The tiled MFMA GEMM of batches above 32 columns at its edges: last row tiles, last column tiles, every column-tile
width, formats whose rows straddle 16-byte chunks, K other than the weight-stationary kernel's, unaligned outputs."""
import os

import numpy as np
import pytest

from oracle import dequant as dq
from oracle import step as ost
from tests._dev import down, empty, up
from tests.conftest import rel_l2
from vte_amd import synthetic as syn

pytestmark = pytest.mark.gpu
TOL = 1e-3  # fp32 sums of fp16 activations (2.1e-4 with fp32 inputs rounded, fp16 results likewise)


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k"])
@pytest.mark.parametrize("n,k,M,io", [(8960, 256, 33, "f32"), (8961, 512, 64, "f16"), (4100, 1536, 96, "f16f32"),
                                      (1, 256, 97, "f16f32"), (33333, 256, 65, "f16"), (130, 768, 515, "f32"),
                                      (17000, 512, 161, "f16f32")])
def test_gemm_tiled(hip, K, fmt, n, k, M, io):
    """vte_gemm_mfma above 32 columns, with bias, residual and scale when the results are fp16."""
    rng = np.random.default_rng(n + M)
    raw = syn.random_matrix(fmt, rng, n, k, balanced=True)
    x = rng.standard_normal((M, k)).astype(np.float32 if io == "f32" else np.float16)
    odt = np.float16 if io == "f16" else np.float32
    y = empty(hip, (M, n), odt)
    kw, bias, res = {}, None, None
    if io == "f16":
        bias, res = rng.standard_normal(n).astype(odt), rng.standard_normal((M, n)).astype(odt)
        kw = dict(bias=up(hip, bias), residual=up(hip, res), residual_scale=0.5)
    K.gemm_mfma(fmt, up(hip, x), up(hip, raw), y, M, k, n, in_dtype="f32" if io == "f32" else "f16",
                out_dtype="f16" if io == "f16" else "f32", stream=hip.stream, **kw)
    rows = np.unique(np.concatenate([np.arange(min(n, 150)), np.arange(max(0, n - 150), n)]))
    ref = dq.gemv(fmt, raw.reshape(n, -1)[rows].reshape(-1), len(rows), k, x.astype(np.float32))
    if io == "f16":
        ref = dq.gemv_epilogue(ref, bias[rows], res[:, rows], 0.5)
    got = down(y)[:, rows].astype(np.float64)
    assert np.isfinite(got).all()
    for m0 in range(0, M, 16):  # a wrong column tile cannot hide in the norm of the others
        assert rel_l2(got[m0:m0 + 16], ref[m0:m0 + 16]) <= TOL, m0


@pytest.mark.parametrize("k,ffn,B", [(256, 8200, 70), (512, 4099, 129), (1536, 9001, 33), (2048, 5000, 100)])
def test_ffn_in_tiled(hip, K, k, ffn, B):
    """Gate/up + SwiGLU: ragged last pairs and columns, rows of the output off 16-byte alignment."""
    rng = np.random.default_rng(ffn)
    wg, wu = (syn.random_matrix("q4_k", rng, ffn, k, balanced=True) for _ in range(2))
    x = rng.standard_normal((B, k)).astype(np.float16)
    out = empty(hip, (B, ffn), np.float16)
    K.ffn_in(up(hip, x), None, 1e-6, up(hip, wg), up(hip, wu), "q4_k", out, B, k, ffn, stream=hip.stream)
    g, u = (dq.gemv("q4_k", w, ffn, k, x.astype(np.float32)).astype(np.float16) for w in (wg, wu))
    got, ref = down(out), ost.swiglu(g, u)
    assert rel_l2(got, ref) <= TOL
    assert rel_l2(got[-1], ref[-1]) <= TOL and rel_l2(got[:, -8:], ref[:, -8:]) <= TOL


@pytest.mark.parametrize("fmt,k,n,M,splits", [("q4_k", 8960, 1536, 164, 5), ("q6_k", 2048, 1537, 300, 8),
                                              ("q6_k", 8960, 1500, 200, 7), ("q4_k", 256, 9000, 512, 1)])
def test_splitk_tiled(hip, K, fmt, k, n, M, splits):
    """Split-K partial sums of the tiled form: the bits of the 32-column launches."""
    import os
    rng = np.random.default_rng(k + M)
    raw = syn.random_matrix(fmt, rng, n, k, balanced=True)
    x = rng.standard_normal((M, k)).astype(np.float16)
    dx, dw = up(hip, x), up(hip, raw)

    def run():
        part = empty(hip, (splits, M, n), np.float32)
        K.gemm_mfma_splitk(fmt, dx, dw, part, M, k, n, splits, stream=hip.stream)
        return down(part)

    got = run()
    os.environ["VTE_MM_WS"] = "0"
    try:
        one = run()
    finally:
        del os.environ["VTE_MM_WS"]
    assert np.array_equal(got.view(np.uint32), one.view(np.uint32))
    ref = dq.gemv(fmt, raw, n, k, x.astype(np.float32))
    assert rel_l2(got.sum(0, dtype=np.float64), ref) <= TOL


@pytest.mark.parametrize("k,n,M,splits", [(1792, 1, 16, 0), (2304, 17, 3, 0), (8960, 301, 16, 0), (4096, 4101, 9, 0),
                                          (8960, 1537, 16, 5), (2048, 33, 5, 8)])
def test_q6k_weights_through_lds(hip, K, k, n, M, splits):
    """Q6_K batches of at most 16 columns: super-blocks at every offset in a 16-byte chunk, ragged rows and waves."""
    rng = np.random.default_rng(k + n)
    raw = syn.random_matrix("q6_k", rng, n, k, balanced=True)
    x = rng.standard_normal((M, k)).astype(np.float16)
    y = empty(hip, (max(splits, 1), M, n), np.float32)
    if splits:
        K.gemm_mfma_splitk("q6_k", up(hip, x), up(hip, raw), y, M, k, n, splits, stream=hip.stream)
    else:
        K.gemm_mfma("q6_k", up(hip, x), up(hip, raw), y, M, k, n, in_dtype="f16", out_dtype="f32", stream=hip.stream)
    got, ref = down(y).sum(axis=0), dq.gemv("q6_k", raw, n, k, x.astype(np.float32))
    assert np.isfinite(got).all()
    for m in range(M):
        assert rel_l2(got[m], ref[m]) <= TOL, m


@pytest.mark.parametrize("k,n_q,n_kv,B,fmt_v,bias", [
    (512, 4, 1, 100, "q6_k", True), (512, 7, 1, 515, "q4_k", True), (256, 3, 3, 65, "q6_k", False),
    (2048, 5, 1, 129, "q6_k", True), (2048, 12, 2, 333, "q4_k", False),
    (1536, 12, 2, 801, "q6_k", True), (1536, 28, 4, 385, "q4_k", True),
    (1536, 12, 2, 65, "q6_k", True), (1536, 4, 2, 128, "q4_k", True)])
def test_attn_in_above_32_columns(hip, K, k, n_q, n_kv, B, fmt_v, bias):
    """q/k/v + bias + RoPE + K/V rows in the tiled form (hidden sizes other than 1536, long batches of it, Q4_K and Q6_K
    rows in one launch) and in the weight-stationary form of 32 rows per block: against the oracle, the bits of the
    32-column launches (a wave there owns at most one super-block), and no other cache row written."""
    hd, max_seq = 128, 900
    rng = np.random.default_rng(k + B)
    wq, wk = (syn.random_matrix("q4_k", rng, n * hd, k, balanced=True) for n in (n_q, n_kv))
    wv = syn.random_matrix(fmt_v, rng, n_kv * hd, k, balanced=True)
    b = [(0.5 * rng.standard_normal(n * hd)).astype(np.float16) for n in (n_q, n_kv, n_kv)]
    x = rng.standard_normal((B, k)).astype(np.float16)
    pos = rng.permutation(max_seq)[:B].astype(np.int32)
    cos_c, sin_c = ost.rope_cache(max_seq, hd, 1e6)
    dx, dq_, dk, dv, dpos, dc, ds = (up(hip, a) for a in (x, wq, wk, wv, pos, cos_c, sin_c))
    db = [up(hip, a) if bias else None for a in b]

    def run():
        q, kc, vc = (empty(hip, s, np.float16) for s in ((B, n_q * hd), (max_seq, n_kv, hd), (max_seq, n_kv, hd)))
        K.attn_in(dx, None, 1e-6, dq_, db[0], "q4_k", dk, db[1], "q4_k", dv, db[2], fmt_v, q, kc, vc, dpos, 0, dc, ds, B,
                  k, n_q, n_kv, stream=hip.stream)  # stride 0: the columns are positions of one sequence
        return down(q), down(kc), down(vc)

    got = run()
    os.environ["VTE_MM_WS"] = "0"
    try:
        one = run()
    finally:
        del os.environ["VTE_MM_WS"]
    for a, c in zip(got, one):
        assert np.array_equal(a.view(np.uint16), c.view(np.uint16))
    x32 = x.astype(np.float32)
    ref = [dq.gemv(f, w, n * hd, k, x32) + (bb.astype(np.float32) if bias else 0)
           for f, w, n, bb in (("q4_k", wq, n_q, b[0]), ("q4_k", wk, n_kv, b[1]), (fmt_v, wv, n_kv, b[2]))]
    ref = [r.astype(np.float16).reshape(B, -1, hd) for r in ref]
    for m, p in enumerate(pos):
        assert rel_l2(got[0][m], ost.rope_neox(ref[0][m], p, cos_c, sin_c).reshape(-1)) <= TOL, m
        assert rel_l2(got[1][p], ost.rope_neox(ref[1][m], p, cos_c, sin_c)) <= TOL, m
        assert rel_l2(got[2][p], ref[2][m]) <= TOL, m
    others = np.delete(np.arange(max_seq), pos)
    assert not got[1][others].any() and not got[2][others].any()


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k"])
@pytest.mark.parametrize("n,k,M", [(8961, 2048, 40), (1000, 1536, 515), (4100, 768, 96)])
def test_gemm_tiled_bits(hip, K, fmt, n, k, M):
    """vte_gemm_mfma tiled: the bits of the 32-column launches where a wave of those owns at most one super-block."""
    rng = np.random.default_rng(n)
    raw = syn.random_matrix(fmt, rng, n, k, balanced=True)
    dx, dw = up(hip, rng.standard_normal((M, k)).astype(np.float16)), up(hip, raw)

    def run():
        y = empty(hip, (M, n), np.float32)
        K.gemm_mfma(fmt, dx, dw, y, M, k, n, in_dtype="f16", out_dtype="f32", stream=hip.stream)
        return down(y)

    got = run()
    os.environ["VTE_MM_WS"] = "0"
    try:
        one = run()
    finally:
        del os.environ["VTE_MM_WS"]
    assert np.array_equal(got.view(np.uint32), one.view(np.uint32))


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k"])
@pytest.mark.parametrize("k,n,M,splits", [(256, 17, 3, 1), (1024, 4100, 16, 1), (768, 1537, 5, 2), (2048, 1000, 8, 8),
                                          (1792, 555, 16, 2), (1280, 40, 9, 1)])
def test_splitk_few_super_blocks(hip, K, fmt, k, n, M, splits):
    """At most 16 columns with up to four super-blocks per split (four-wave blocks), uneven shares, and five (eight waves):
    every split's sums against the oracle over its super-blocks."""
    rng = np.random.default_rng(k + n)
    raw = syn.random_matrix(fmt, rng, n, k, balanced=True)
    x = rng.standard_normal((M, k)).astype(np.float16)
    y = empty(hip, (splits, M, n), np.float32)
    K.gemm_mfma_splitk(fmt, up(hip, x), up(hip, raw), y, M, k, n, splits, stream=hip.stream)
    got, sb = down(y), k // 256
    blocks = raw.reshape(n, sb, -1)
    for s in range(splits):
        a, b = sb * s // splits, sb * (s + 1) // splits
        ref = dq.gemv(fmt, np.ascontiguousarray(blocks[:, a:b]).reshape(-1), n, 256 * (b - a),
                      x[:, 256 * a:256 * b].astype(np.float32))
        for m in range(M):
            assert rel_l2(got[s, m], ref[m]) <= 1e-5, (s, m)  # fp32 sums of exact products

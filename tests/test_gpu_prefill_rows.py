"""GPU tests of the prompt layer's row products (prefill_rows.h, up to 128
tokens) and of the tiled q/k/v products that end in head norms, RoPE and the
cache writes (above).

Token counts sit on the edges of their 16- and 32-token tiles and of the rules
that pick an instance.  Each product is checked against a 64-bit product of the
GPU's own input rows and the f16 weights.  Bound: an f32 sum of K exact f16
products is off by at most K 2^-24 sum |x w| in any order; rounding to f16 adds
half an ulp, 2^-11 relative (2^-25 for subnormals).
"""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_decode import f64, fill_cache_layer, rope_tol

pytestmark = pytest.mark.gpu

LAYER = 5


@pytest.fixture(scope="module")
def D():
    from qwen3_iree_amd import decode

    return decode


@pytest.fixture(scope="module")
def dmodel(gpu, D, model_host):
    m = D.DeviceWeights(model_host, prefill_f16=True)
    yield m
    m.free()


@pytest.fixture(scope="module")
def w64(O, model_host):
    w = model_host
    return {name: O.q8_dequant_f16(m[LAYER], n, k).astype(np.float64)
            for name, m, n, k in (("q", w.wq, 2048, 1024), ("k", w.wk, 1024, 1024),
                                  ("v", w.wv, 1024, 1024), ("o", w.wo, 1024, 2048),
                                  ("gu", w.wgu, 6144, 1024), ("dn", w.wdn, 1024, 3072))}


def product(x, w):
    """x w^T in 64 bits and the error bound of its f16 result."""
    x = x.astype(np.float64)
    ref = x @ w.T
    return ref, 2.0 ** -11 * np.abs(ref) + 2.0 ** -25 + x.shape[1] * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T)


def assert_within(got, ref, tol, what):
    bad = np.argwhere(~(np.abs(got.astype(np.float64) - ref) <= tol))
    assert bad.size == 0, (what, len(bad), bad[:4].tolist())


def check_layer(g, h_in, w64):
    for name in ("q", "k", "v"):
        assert_within(g[name], *product(g["xn"], w64[name]), name)
    for name, x, base, out in (("o", "attn", h_in, "res"), ("dn", "act", g["res"], "h")):
        ref, tol = product(g[x], w64[name])
        ref = base.astype(np.float64) + ref
        assert_within(g[out], ref, tol + 2.0 ** -11 * (np.abs(ref) + tol) + 2.0 ** -25, out)
    ref, tol = product(g["fn"], w64["gu"])
    gate, up = ref[:, :3072], ref[:, 3072:]
    sig = 1 / (1 + np.exp(-gate))
    # |d silu / d gate| <= 1.1; exp, 1 + e, 1 / den, gate sig and silu up each
    # round to f16 once: five half-ulp steps on the way to the result
    rel = 5 * 2.0 ** -11 + 2.0 ** -10
    want = gate * sig * up
    assert_within(g["act"], want,
                  1.1 * np.abs(up) * tol[:, :3072] + np.abs(gate * sig) * tol[:, 3072:]
                  + rel * np.abs(want) + 2.0 ** -20 * (1 + np.abs(up)), "act")


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 49, 63, 64, 65, 81, 127, 128, 129, 160,
                               255, 256, 257])
def test_row_products_match_f64_and_both_weight_forms_agree(gpu, D, dmodel, w64, n):
    rng = np.random.default_rng(4100 + n)
    p0 = 7
    sess = D.DecodeSession(dmodel, p0 + n + 3)
    try:
        kc = np.zeros((28 * sess.max_seq, 1024), np.float16)
        fill_cache_layer(sess, LAYER, p0, rng, kc, np.zeros_like(kc))
        h_in = (1.5 * rng.standard_normal((n, 1024))).astype(np.float16)
        res = []
        for f16 in (True, False):
            print(f"row products n {n} f16 {f16}", flush=True)
            dmodel.use_prefill_matrices(f16)
            g = sess.prefill_layer(LAYER, h_in, p0)
            res.append((g, sess.cache_rows(LAYER, 0, sess.max_seq)))
        (ga, ca), (gb, cb) = res
        for name in ga:
            assert np.array_equal(ga[name].view(np.uint16), gb[name].view(np.uint16)), name
        for a, b in zip(ca, cb):
            assert np.array_equal(a.view(np.uint16), b.view(np.uint16))
        check_layer(ga, h_in, w64)
        assert np.array_equal(ca[1][p0:p0 + n].view(np.uint16), ga["v"].view(np.uint16))
        assert not ca[0][p0 + n:].any() and not ca[1][p0 + n:].any()
    finally:
        dmodel.use_prefill_matrices(True)
        sess.free()


@pytest.mark.parametrize("n", [1, 17, 65, 129, 257, 511, 512, 513, 1030, 1930])
def test_head_norms_rope_and_cache(O, gpu, D, dmodel, model_host, n):
    """q_roped, the K slots and the V slots against the oracle's head norm and
    RoPE of the GPU's own q, k and v (2 ulp plus one ulp of the head's largest
    input), tokens at the tile edges; both weight forms the same bits."""
    p0 = 9
    h_in = (1.5 * np.random.default_rng(4300 + n).standard_normal((n, 1024))).astype(np.float16)
    sess = D.DecodeSession(dmodel, p0 + n + 1)
    res = []
    try:
        for f16 in (True, False):
            print(f"q/k/v epilogue n {n} f16 {f16}", flush=True)
            dmodel.use_prefill_matrices(f16)
            g = sess.prefill_layer(LAYER, h_in, p0, True)
            res.append((g["q_roped"], g["q"], g["k"], g["v"],
                        *sess.cache_rows(LAYER, 0, p0 + n + 1)))
    finally:
        dmodel.use_prefill_matrices(True)
        sess.free()
    for a, b in zip(*res):
        assert np.array_equal(a.view(np.uint16), b.view(np.uint16))
    q_roped, q, k, v, k_rows, v_rows = res[0]
    assert np.array_equal(v_rows[p0:p0 + n].view(np.uint16), v.view(np.uint16))
    for rows in (k_rows, v_rows):
        assert not rows[:p0].any() and not rows[p0 + n:].any()
    for i in sorted({t for t in (0, 1, 15, 16, 63, 64, 127, 128, n // 2, n - 2, n - 1) if 0 <= t < n}):
        for x, w, got in ((q, model_host.q_norm, q_roped[i]), (k, model_host.k_norm, k_rows[p0 + i])):
            normed = O.head_rmsnorm(x[i], w[LAYER])
            want = O.rope(normed, p0 + i)
            assert (np.abs(f64(got) - f64(want)) <= rope_tol(O, normed, want)).all(), i


@pytest.mark.parametrize("f16", [True, False])
def test_head_rows_do_not_depend_on_the_prompt_length(gpu, D, dmodel, f16):
    """From 65 tokens on a q or k row is one chain of products over K, so the
    first tokens' raw rows are the same in longer prompts; so must be what head
    norm and RoPE make of them, in the row product's epilogue (up to 128 tokens)
    and the tiled ones'.  Token 5's row is zero."""
    h_in = (1.5 * np.random.default_rng(4500).standard_normal((1100, 1024))).astype(np.float16)
    h_in[5] = 0
    p0, first = 11, 100
    dmodel.use_prefill_matrices(f16)
    res = {}
    try:
        for n in (first, 129, 300, 700, 1100):
            print(f"head rows n {n} f16 {f16}", flush=True)
            sess = D.DecodeSession(dmodel, p0 + n)
            try:
                g = sess.prefill_layer(LAYER, h_in[:n], p0, True)
                res[n] = [g[name][:first] for name in ("q", "k", "v", "q_roped")] + [
                    r[p0:p0 + first] for r in sess.cache_rows(LAYER, 0, p0 + n)]
            finally:
                sess.free()
    finally:
        dmodel.use_prefill_matrices(True)
    for n, rows in res.items():
        for name, a, b in zip(("q", "k", "v", "q_roped", "k_cache", "v_cache"), rows, res[first]):
            assert np.array_equal(a.view(np.uint16), b.view(np.uint16)), (n, name)


@pytest.mark.parametrize("n", [513, 575, 992, 993, 1024, 1025, 1153, 1920, 1921, 2047, 2560, 2561])
def test_unsplit_residual_products(gpu, D, dmodel, w64, n):
    """attn_o and ffn_down around the edges of the one-round products with the
    residual in the epilogue (513 to 2560 tokens, one K range or two): the
    64-bit product's bound on the first and last token tiles, and the bits of
    the Q8_0 route (split products and their reduce)."""
    h_in = (1.5 * np.random.default_rng(4400 + n).standard_normal((n, 1024))).astype(np.float16)
    sess = D.DecodeSession(dmodel, n)
    res = []
    try:
        for f16 in (True, False):
            print(f"residual products n {n} f16 {f16}", flush=True)
            dmodel.use_prefill_matrices(f16)
            res.append(sess.prefill_layer(LAYER, h_in, 0))
    finally:
        dmodel.use_prefill_matrices(True)
        sess.free()
    ga, gb = res
    for name in ga:
        assert np.array_equal(ga[name].view(np.uint16), gb[name].view(np.uint16)), name
    rows = np.r_[0:130, n - 130:n]
    check_layer({name: a[rows] for name, a in ga.items()}, h_in[rows], w64)


@pytest.mark.parametrize("n", [16, 100, 200])
def test_row_products_with_the_prompts_rope_table(gpu, D, dmodel, model_host, n):
    """qwen3_prefill_batched computes the RoPE table in its first layer and
    reads it in the others; a layer on its own computes its angles: every
    layer's cache rows must be the same bits."""
    prompt = np.random.default_rng(4200 + n).integers(0, D.VOCAB, n).astype(np.int32)
    print(f"row products rope table n {n}", flush=True)
    a, b = D.DecodeSession(dmodel, n + 1), D.DecodeSession(dmodel, n + 1)
    try:
        a.set_state(0, 0)
        a.prefill_batched(prompt)
        h = model_host.token_embd[prompt]
        for layer in range(28):
            h = b.prefill_layer(layer, h, 0)["h"]
            for x, y in zip(a.cache_rows(layer, 0, n), b.cache_rows(layer, 0, n)):
                assert np.array_equal(x.view(np.uint16), y.view(np.uint16)), layer
    finally:
        a.free()
        b.free()

"""GPU test of the prompt attention under its default division into splits:
token and position counts on both sides of every line of the rule (no splits,
about 0.6 sqrt(nb) blocks, at least 8 from 8 query blocks on, nb / 3 from 32),
with ragged last query blocks.  The oracle's attention over the GPU's own
cache and roped q, bound 2 ulp + 1e-5 as in the other attention tests."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_decode import f64, ulp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    from qwen3_iree_amd import decode

    return decode


@pytest.fixture(scope="module")
def dmodel(gpu, D, model_host):
    m = D.DeviceWeights(model_host, prefill_f16=True)
    yield m
    m.free()


@pytest.mark.parametrize("n,p0,chunk_local", [
    (1, 255, False), (1, 256, False), (1, 1700, False), (33, 200, False), (33, 1111, False),
    (224, 40, False), (225, 40, False), (225, 300, False), (300, 1000, False), (300, 1000, True),
    (992, 0, False), (1000, 31, False)])
def test_default_splits(O, gpu, D, dmodel, n, p0, chunk_local):
    layer = 11
    rng = np.random.default_rng(100 * n + p0)
    sess = D.DecodeSession(dmodel, p0 + n)
    try:
        if p0:
            sess.k_cache.upload(rng.standard_normal((p0, 1024)).astype(np.float16),
                                layer * sess.max_seq * 2048)
            sess.v_cache.upload((0.6 * rng.standard_normal((p0, 1024))).astype(np.float16),
                                layer * sess.max_seq * 2048)
        h_in = (1.5 * rng.standard_normal((n, 1024))).astype(np.float16)
        print(f"prompt attention n {n} p0 {p0} chunk_local {chunk_local}", flush=True)
        g = sess.prefill_layer(layer, h_in, p0, chunk_local)
        k_rows, v_rows = sess.cache_rows(layer, 0, p0 + n)
        lo = p0 if chunk_local else 0
        tokens = range(n) if n <= 48 else sorted({0, 1, 31, 32, n // 2, n - 33, n - 2, n - 1})
        for i in tokens:
            want = O.attention(g["q_roped"][i], k_rows[lo:p0 + i + 1], v_rows[lo:p0 + i + 1])
            d = np.abs(f64(g["attn"][i]) - f64(want))
            assert (d <= 2 * ulp(O, want) + 1e-5).all(), (i, d.max())
    finally:
        sess.free()

"""GPU tests of the decode attention where the number of position splits per
kv head changes: 32 up to a context of 1280 positions, 64 above.

- One layer's attention over the GPU's own cache against the oracle, at
  contexts on both sides of the change and at ragged ones (uneven splits, the
  last split a few positions long).  Bound as in the other attention tests:
  2 ulp of the f16 result for the f16 rounding of the output and 1e-5 for f32
  sums over weights carried to 2^-22.
- A whole step at such contexts: both step modes give the same bits.
"""
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
    m = D.DeviceWeights(model_host)
    yield m
    m.free()


@pytest.mark.parametrize("ctx", [1279, 1280, 1281, 1282, 1313, 1999, 2047, 2048, 2049, 2050, 2081, 3333, 4096, 4097, 6200])
def test_layer_attention_where_the_splits_change(O, gpu, D, dmodel, ctx):
    layer, pos = 4, ctx - 1
    rng = np.random.default_rng(ctx)
    sess = D.DecodeSession(dmodel, ctx + 1)
    k = rng.standard_normal((pos, 1024)).astype(np.float16)
    v = (0.6 * rng.standard_normal((pos, 1024))).astype(np.float16)
    sess.k_cache.upload(k, layer * sess.max_seq * 2048)
    sess.v_cache.upload(v, layer * sess.max_seq * 2048)
    hin = gpu.DeviceBuffer.from_array((1.5 * rng.standard_normal(1024)).astype(np.float16))
    hout = gpu.DeviceBuffer(2048)
    try:
        sess.set_state(0, pos)
        print(f"decode layer at context {ctx}", flush=True)
        sess.layer(layer, hin, hout)
        q, got = sess.scratch_f16("q_roped", 2048), sess.scratch_f16("attn", 2048)
        k_rows, v_rows = sess.cache_rows(layer, 0, ctx + 1)
        assert np.array_equal(k_rows[:pos], k) and np.array_equal(v_rows[:pos], v)
        assert np.array_equal(v_rows[pos].view(np.uint16),
                              sess.scratch_f16("v", 1024).view(np.uint16))
        assert not k_rows[ctx:].any() and not v_rows[ctx:].any()
        want = O.attention(q, k_rows[:ctx], v_rows[:ctx])
        d = np.abs(f64(got) - f64(want))
        assert (d <= 2 * ulp(O, want) + 1e-5).all(), d.max()
    finally:
        hin.free()
        hout.free()
        sess.free()


@pytest.mark.parametrize("ctx", [1280, 1281, 2048, 2049, 3333])
def test_step_modes_bit_identical_where_the_splits_change(gpu, D, dmodel, ctx):
    rng = np.random.default_rng(7 + ctx)
    k = rng.standard_normal((ctx, 1024)).astype(np.float16)
    v = (0.6 * rng.standard_normal((ctx, 1024))).astype(np.float16)
    before, out = D.step_mode(), []
    for mode in (1, 0):
        sess = D.DecodeSession(dmodel, ctx + 2)
        try:
            D.set_step_mode(mode)
            for layer in range(28):
                sess.k_cache.upload(np.roll(k, layer, 0), layer * sess.max_seq * 2048)
                sess.v_cache.upload(np.roll(v, layer, 0), layer * sess.max_seq * 2048)
            sess.set_state(77, ctx - 2)
            print(f"step mode {mode} at contexts {ctx - 1}, {ctx}, {ctx + 1}", flush=True)
            for _ in range(3):  # across the change where ctx is next to it
                sess.step(advance=True, logits=True)
            assert sess.check_status() == 0
            out.append((sess.get_state(), sess.read_logits(),
                        [sess.cache_rows(layer, ctx - 2, ctx + 1) for layer in (0, 13, 27)]))
        finally:
            D.set_step_mode(before)
            sess.free()
    (sa, la, ca), (sb, lb, cb) = out
    assert sa == sb and np.array_equal(la.view(np.uint16), lb.view(np.uint16))
    for x, y in zip(ca, cb):
        for a, b in zip(x, y):
            assert np.array_equal(a.view(np.uint16), b.view(np.uint16))


def _filled(D, dmodel, max_seq, pos, stream=None):
    rng = np.random.default_rng(pos)
    k = rng.standard_normal((pos, 1024)).astype(np.float16)
    v = (0.6 * rng.standard_normal((pos, 1024))).astype(np.float16)
    sess = D.DecodeSession(dmodel, max_seq, stream)
    for layer in range(28):
        sess.k_cache.upload(np.roll(k, layer, 0), layer * max_seq * 2048)
        sess.v_cache.upload(np.roll(v, layer, 0), layer * max_seq * 2048)
    sess.set_state(1234, pos)
    return sess


@pytest.mark.parametrize("how", ["prompt_steps", "graph"])
def test_other_ways_over_the_switch(gpu, D, dmodel, how):
    """Positions 1278 to 1282 as prompt steps (no vocab product before the last)
    and as replays of one captured step: the bits of eager per-phase steps."""
    pos, max_seq, n = 1278, 1290, 5
    prompt = [5, 151935, 17, 0, 42]

    def run(mode):
        D.set_step_mode(mode)
        graph = how == "graph" and mode == 1
        stream = gpu.Stream() if graph else None
        sess = _filled(D, dmodel, max_seq, pos, stream)
        try:
            print(f"{how} from position {pos}, mode {mode}", flush=True)
            if how == "prompt_steps":
                sess.prefill(prompt)
            else:
                for _ in range(n):
                    sess.replay() if graph else sess.step(advance=True, logits=False)
                    sess.synchronize()
            assert sess.check_status() == 0
            return sess.get_state(), [r.view(np.uint16).copy() for layer in (0, 13, 27)
                                      for r in sess.cache_rows(layer, 0, max_seq)]
        finally:
            sess.free()
            if stream is not None:
                stream.destroy()

    before = D.step_mode()
    try:
        (sa, ca), (sb, cb) = run(1), run(0)
    finally:
        D.set_step_mode(before)
    assert sa == sb and sa[1] == pos + n
    for a, b in zip(ca, cb):
        assert np.array_equal(a, b)

"""Batched prefill over the row counts at which its GEMMs change block tile,
K split and remainder, against the token-by-token path."""
import numpy as np
import pytest

from gemma_amd import capi, synth

from gpu_util import rel, say

pytestmark = pytest.mark.gpu
# fp32 sums in another order and bf16 hi + lo products (2^-17 per input) over
# at most 6912 inputs and two layers stay below 1e-4 of the largest value
TOL = 1e-4
_MODELS = {}

SHAPES = {
    "270m": synth.Shape(hidden=640, layers=2, n_q=4, inter=2048, vocab=4096, ctx=4096),
    "1b": synth.Shape(hidden=1152, layers=2, n_q=4, inter=6912, vocab=4096, ctx=4096),
    # few 32-blocks per row (4 and 18), 2 query heads
    "ragged": synth.Shape(hidden=128, layers=2, n_q=2, inter=576, vocab=4096, ctx=4096),
}


@pytest.mark.parametrize("name", list(SHAPES))
def test_prefill_rows_around_every_tile_edge(gpu, name):
    shape = SHAPES[name].gemma3_mode(window=100)
    t = synth.make_model(shape, seed=5)
    n_max = 2100
    prompt = synth.prompt_ids(n_max, seed=9, vocab=shape.vocab)
    ref = capi.Engine(shape.gg_config(prefill_batch=0))
    ref.upload_model(t)
    ref.finalize()
    ref.prefill(prompt, 0)
    kv = {(w, l): ref.read(w, l).reshape(shape.ctx, 256) for w in (capi.READ_K_CACHE, capi.READ_V_CACHE)
          for l in range(shape.layers)}
    hidden = {}
    rows = [2, 16, 31, 32, 33, 63, 64, 65, 127, 129, 187, 300, 511, 512, 513, 777, 1025, 1537, n_max]
    for n in rows:   # the last row's hidden state, token by token
        ref.step(int(prompt[n - 1]), n - 1)
        hidden[n] = [ref.read(capi.READ_LAYER_HIDDEN, l) for l in range(shape.layers)]
    ref.close()
    e = capi.Engine(shape.gg_config(prefill_batch=n_max))
    e.upload_model(t)
    e.finalize()
    for n in rows:
        say(name, "rows", n)
        e.reset_kv()
        e.prefill(prompt[:n], 0)
        for l in range(shape.layers):
            assert rel(e.read(capi.READ_LAYER_HIDDEN, l), hidden[n][l]) < TOL, (n, l)
            for w in (capi.READ_K_CACHE, capi.READ_V_CACHE):
                got = e.read(w, l).reshape(shape.ctx, 256)
                assert rel(got[:n], kv[w, l][:n]) < TOL, (n, l, w)
                assert not np.any(got[n:]), (n, l, w)
    # the same rows as a second turn on reused KV
    for start, n in [(1, 33), (700, 64), (1309, 187), (777, 1025)]:
        say(name, "turn", start, n)
        e.reset_kv()
        e.prefill(prompt[:start], 0)
        e.prefill(prompt[start:start + n], start)
        for l in range(shape.layers):
            for w in (capi.READ_K_CACHE, capi.READ_V_CACHE):
                assert rel(e.read(w, l).reshape(shape.ctx, 256)[:start + n], kv[w, l][:start + n]) < TOL, (start, n, l, w)
    e.close()

"""Turns on reused KV through a batched prefill with local and global layers,
against the token-by-token path: the spans at which the attention takes 16- and
32-row query tiles, one or several key chunks, and a ragged last query tile."""
import os
import subprocess

import pytest

from gemma_amd import capi, synth

from gpu_util import rel, say

# fp32 sums in another order and bf16 hi + lo products (2^-17 per input) over
# at most 2048 inputs and three layers stay below 1e-4 of the largest value
TOL = 1e-4
WINDOW = 700
# layer 0 and 2 local, layer 1 global: layer 1's and 2's K/V check every row of
# the layer before, the hidden states the last row of every layer
SHAPES = {n_q: synth.Shape(hidden=hidden, layers=3, n_q=n_q, inter=inter, vocab=4096, ctx=6144, swa_period=2)
          for n_q, hidden, inter in [(4, 640, 2048), (2, 128, 576), (1, 256, 192)]}
# (start, rows): (rows per query tile / 16, several chunks) on global and on local layers
TURNS = {(0, 1537): ((2, True), (1, True)), (0, 2100): ((2, True), (2, True)), (1309, 187): ((1, True), (1, True)),
         (2047, 2049): ((2, True), (2, True)), (0, 3000): ((2, True), (1, False)), (0, 16): ((1, False), (1, False)),
         (4100, 995): ((2, True), (1, True)), (5000, 33): ((1, True), (1, True)), (5000, 1100): ((2, True), (1, True))}
PLAN = r"""
#include <cstdio>
#include <cstdlib>
#include "gg_internal.h"
int main(int, char** argv) {
  const int window = atoi(argv[1]), start = atoi(argv[2]), rows = atoi(argv[3]);
  const gg::PrefillPlan p = gg::prefill_plan(window, start, rows);
  printf("%d %d\n", p.rt, gg::prefill_max_tiles(window, start, rows, 16 * p.rt) > p.chunk);
}
"""


def test_turns_reach_every_form_of_the_attention(tmp_path):
    """The rule that picks them, on the CPU: the turns below run what they are listed for."""
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "webgpu-gemma_amd", "csrc")
    (tmp_path / "plan.cpp").write_text(PLAN)
    subprocess.run(["g++", "-std=c++17", "-D__host__=", "-D__device__=", "-I", csrc, str(tmp_path / "plan.cpp"), "-o",
                    str(tmp_path / "plan")], check=True)
    seen = set()
    for (start, n), forms in TURNS.items():
        for window, want in zip((0, WINDOW), forms):
            out = subprocess.run([str(tmp_path / "plan"), str(window), str(start), str(n)], check=True,
                                 capture_output=True, text=True).stdout.split()
            assert (int(out[0]), bool(int(out[1]))) == want, (window, start, n)
            seen.add((window, *want))
    assert seen >= {(0, 1, False), (0, 1, True), (0, 2, True), (WINDOW, 1, False), (WINDOW, 1, True), (WINDOW, 2, True)}


@pytest.mark.gpu
@pytest.mark.parametrize("n_q", list(SHAPES))
def test_prefill_turns_on_local_and_global_layers(gpu, n_q):
    shape = SHAPES[n_q].gemma3_mode(window=WINDOW)
    t = synth.make_model(shape, seed=11)
    n_max = max(start + n for start, n in TURNS)
    prompt = synth.prompt_ids(n_max, seed=12, vocab=shape.vocab)
    ref = capi.Engine(shape.gg_config(prefill_batch=0))
    ref.upload_model(t)
    ref.finalize()
    ref.prefill(prompt, 0)
    kv = {(w, l): ref.read(w, l).reshape(shape.ctx, 256) for w in (capi.READ_K_CACHE, capi.READ_V_CACHE)
          for l in range(shape.layers)}
    hidden = {}
    for last in {start + n for start, n in TURNS}:   # the last row's hidden states, token by token
        ref.step(int(prompt[last - 1]), last - 1)
        hidden[last] = [ref.read(capi.READ_LAYER_HIDDEN, l) for l in range(shape.layers)]
    ref.close()
    e = capi.Engine(shape.gg_config(prefill_batch=4096))
    e.upload_model(t)
    e.finalize()
    for start, n in TURNS:
        say("heads", n_q, "turn", start, n)
        e.reset_kv()
        if start:
            e.prefill(prompt[:start], 0)
        e.prefill(prompt[start:start + n], start)
        for l in range(shape.layers):
            assert rel(e.read(capi.READ_LAYER_HIDDEN, l), hidden[start + n][l]) < TOL, (start, n, l)
            for w in (capi.READ_K_CACHE, capi.READ_V_CACHE):
                got = e.read(w, l).reshape(shape.ctx, 256)[:start + n]
                assert rel(got, kv[w, l][:start + n]) < TOL, (start, n, l, w)
    e.close()

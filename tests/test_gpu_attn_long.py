"""Decode attention around the bound of its long-context path and the edges of
its segments (224 positions, two a round; runs of 64 positions a workgroup):
a token fed one at a time behind a batched prompt leaves the bits of a prompt
that holds it too (the batched prefill's attention forms the same sums
another way)."""
import numpy as np
import pytest
from tmq import model_synth, tmacfile

pytestmark = pytest.mark.gpu

MAX_SEQ = 1400


@pytest.fixture(scope="module")
def model(ctx):
    import tmq
    print("[attn] generating a 2-layer model", flush=True)
    m = tmq.Model(ctx, tmacfile.to_bytes(model_synth.gen_model(5, n_layers=2, vocab=512)), max_seq=MAX_SEQ)
    yield m
    m.free()


@pytest.mark.parametrize("n", [478, 511, 575, 671, 672, 895, 896, 1023, 1343, 1397])
def test_long_decode(model, n):
    print(f"[attn] {n} positions", flush=True)
    toks = np.random.default_rng(n).integers(0, 512, MAX_SEQ).astype(np.int32)
    model.prompt(toks[:n])
    for i in range(n, min(n + 3, MAX_SEQ)):
        model.feed(int(toks[i]))
    h0, l0 = model.hidden(), model.logits()
    model.prompt(toks[:min(n + 3, MAX_SEQ)])
    h1, l1 = model.hidden(), model.logits()
    assert np.array_equal(h0.view(np.uint32), h1.view(np.uint32))
    assert np.array_equal(l0.view(np.uint32), l1.view(np.uint32))

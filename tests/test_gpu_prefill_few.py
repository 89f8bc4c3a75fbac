"""Batched prefill of few tokens (its own GEMM kernel up to 192 tokens a
chunk) around its 32-token blocks and its bound, whole and as the last chunk
of a longer prompt: the bits of one token at a time."""
import numpy as np
import pytest
from tmq import model_synth, tmacfile

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(ctx):
    import tmq
    print("[few] generating a 3-layer model (Q8_0 and Q5_0 attn_v, Q6_K and Q4_K ffn_down)", flush=True)
    m = tmq.Model(ctx, tmacfile.to_bytes(model_synth.gen_model(6, n_layers=3, vocab=512)), max_seq=512)
    yield m
    m.free()


@pytest.mark.parametrize("n, chunk", [(2, 512), (31, 512), (32, 512), (33, 512), (64, 512), (65, 512), (128, 512),
                                      (129, 512), (191, 512), (192, 512), (193, 512), (300, 256), (385, 128), (200, 33)])
def test_few_tokens(model, n, chunk):
    print(f"[few] {n} tokens in chunks of {chunk}", flush=True)
    toks = np.random.default_rng(n).integers(0, 512, n).astype(np.int32)
    out = []
    for c in (0, chunk):
        model.set_prefill(c)
        model.prompt(toks)
        model.feed(7)
        out.append((model.hidden(), model.logits()))
    model.set_prefill(512)
    for a, b in zip(*out):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))

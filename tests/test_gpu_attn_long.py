"""Decode attention around the bound of its long-context path and the edges of
its segments (224 positions, two a round; runs of 64 positions a workgroup):
a token fed one at a time behind a batched prompt leaves the bits of a prompt
that holds it too (the batched prefill's attention forms the same sums
another way); and the context of one layer against the reference's loops
restated in numpy, up to the last position of the largest cache, in every
form that q, k and v reach the attention in."""
import ctypes

import numpy as np
import pytest
from oracle import Q5_0, Q8_0
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


# ------------------------------------------------- against the reference's loops
_M = ctypes.CDLL("libm.so.6")
for _f in ("expf", "logf", "powf", "cosf", "sinf"):
    getattr(_M, _f).restype = ctypes.c_float
    getattr(_M, _f).argtypes = [ctypes.c_float] * (2 if _f == "powf" else 1)
F = np.float32
CACHE = 3072  # 16 workgroups a head, 14 segments, six scores a thread


def matmul(oracle, flags, t, x):
    import tmq
    args = (t.type, t.data, x, t.rows, t.cols)
    if not flags:
        return oracle.matmul_fp32(*args)
    return oracle.matmul(*args) if flags == tmq.FLAGS_ALL else oracle.matmul_int16(*args)[0]


def rope(v, pos, base):
    """apply_rope (sim/tmac_gguf.cpp:1531-1539) of [n, heads, 64] rows at the positions pos"""
    out = np.empty_like(v)
    for j in range(32):
        theta = F(1) / F(_M.powf(base, 2 * j / 64))
        fr = [float(F(p) * theta) for p in pos]
        c = np.array([_M.cosf(f) for f in fr], F)[:, None]
        s = np.array([_M.sinf(f) for f in fr], F)[:, None]
        a, b = v[:, :, 2 * j], v[:, :, 2 * j + 1]
        out[:, :, 2 * j] = a * c - b * s
        out[:, :, 2 * j + 1] = a * s + b * c
    return out


def attention(q, k, v):
    """one query [heads, 64] over [n, kv heads, 64] rows, every sum in the reference's order (:1639-1660)"""
    heads, per = q.shape[0], q.shape[0] // k.shape[1]
    out = np.zeros((heads, 64), F)
    for h in range(heads):
        s = np.zeros(k.shape[0], F)
        for d in range(64):
            s = s + q[h, d] * k[:, h // per, d]
        s = s / F(8)
        m = s.max()
        e = F(0)
        for x in s - m:
            e = e + F(_M.expf(x))
        ls = F(_M.logf(e)) + m
        for p in range(k.shape[0]):
            out[h] = out[h] + F(_M.expf(s[p] - ls)) * v[p, h // per]
    return out.reshape(-1)


# q, k and v: fitted products with Q8_0 tiles in v, and without; tiles in all
# three (INT16); final values (FP32); the exp sum's every segment run again
@pytest.mark.parametrize("flags,q8v,miss", [("all", True, False), ("all", False, False), ("int16", True, False),
                                            ("none", True, False), ("all", True, True)])
def test_context_vs_reference(ctx, oracle, monkeypatch, flags, q8v, miss):
    import tmq
    flags = {"all": tmq.FLAGS_ALL, "int16": tmq.FLAG_FPGA, "none": 0}[flags]
    if miss:
        monkeypatch.setenv("TMQ_SPEC_MISS", "1")
    ts = model_synth.gen_model(15, n_layers=1, vocab=64, q8_v_layers=(0,) if q8v else ())
    by = {t.name: t for t in ts}
    assert by["blk.0.attn_v.weight"].type == (Q8_0 if q8v else Q5_0)
    m = tmq.Model(ctx, tmacfile.to_bytes(ts), max_seq=CACHE)
    try:
        m.set_flags(flags)
        H, base = m.config["hidden"], m.config["rope_base"]
        rows = []  # q, k, v of each token before RoPE: the first layer's depend on nothing else
        for tok in range(8):
            m.prompt([tok])
            x = np.ascontiguousarray(m.feed_capture(tok)[0, :H])
            rows.append([matmul(oracle, flags, by[f"blk.0.attn_{n}.weight"], x) + by[f"blk.0.attn_{n}.bias"].data.view(F)
                         for n in "qkv"])
        toks = np.random.default_rng(9).integers(0, 8, CACHE).astype(np.int32)
        k = rope(np.stack([rows[t][1] for t in toks]).reshape(CACHE, -1, 64), np.arange(CACHE), base)
        v = np.stack([rows[t][2] for t in toks]).reshape(CACHE, -1, 64)
        # the last short position and the first long one; one before and at a
        # fourth segment; 9 and 16 workgroups; the cache's last position
        for n in (479, 480, 671, 672, 1727, 2049, CACHE - 1):
            print(f"[attn] flags {flags} q8_0 v {q8v} miss {miss}: position {n}", flush=True)
            m.prompt(toks[:n])
            got = m.feed_capture(int(toks[n]))[0, H:2 * H]
            q = rope(rows[toks[n]][0].reshape(1, -1, 64), [n], base)[0]
            want = attention(q, k[:n + 1], v[:n + 1])
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), n
    finally:
        m.free()

"""GPU parity of the single-launch GEMVs at the edges of their tiling, bit
for bit against the CPU oracle: row remainders, one tile and the last tile
of an LDS batch, half tiles, and results stored over the activation."""
import numpy as np
import pytest
from oracle import F16, F32, Q4_K, Q5_0, Q6_K, Q8_0
from tmq import synth

pytestmark = pytest.mark.gpu


def bits(a):
    return np.asarray(a, dtype=np.float32).view(np.uint32)


# 64-column tiles: 1 (half), 2 (the second half full), 14, 128 = one LDS
# batch, 129 (a half tile in a second batch), 200; rows 1, 8k, 8k + 1, 64k + 1
@pytest.mark.parametrize("qt,rows,cols", [(F32, 1, 32), (Q8_0, 9, 96), (Q5_0, 65, 896), (Q4_K, 24, 8192),
                                          (F16, 3, 8224), (Q5_0, 130, 12800), (Q6_K, 7, 4864)])
def test_int16_edges(ctx, oracle, qt, rows, cols):
    import tmq
    print(f"[single] int16 type={qt} {rows}x{cols}", flush=True)
    w = synth.gen_weights(qt, rows, cols, 41 + rows)
    x = synth.gen_x(cols, 42 + cols)
    t = ctx.upload(qt, rows, cols, w)
    try:
        acc, xs = ctx.partials_int16(t, x)
        y = ctx.matmul_path(t, x, tmq.PATH_INT16)
    finally:
        t.free()
    ye, te, _ = oracle.matmul_int16(qt, w, x, rows, cols)
    assert xs == oracle.quantize_act(x)[1]
    assert np.array_equal(acc, te)
    assert np.array_equal(bits(y), bits(ye))


# the last row count of the 8-row workgroups and the first of a lane a row:
# 57344 up to 128 columns, 768 a column above
@pytest.mark.parametrize("rows,cols", [(57344, 32), (57345, 96), (57345, 128), (122880, 160), (122881, 160)])
def test_int16_bounds(ctx, oracle, rows, cols):
    import tmq
    print(f"[single] int16 {rows}x{cols}", flush=True)
    w = synth.gen_weights(Q5_0, rows, cols, 43 + cols)
    x = synth.gen_x(cols, 44 + cols)
    t = ctx.upload(Q5_0, rows, cols, w)
    try:
        acc, xs = ctx.partials_int16(t, x)
        y = ctx.matmul_path(t, x, tmq.PATH_INT16)
    finally:
        t.free()
    ye, te, _ = oracle.matmul_int16(Q5_0, w, x, rows, cols)
    assert xs == oracle.quantize_act(x)[1]
    assert np.array_equal(acc, te)
    assert np.array_equal(bits(y), bits(ye))


# 384 columns a batch: one block, one batch exactly, one block more, two
# batches and a half; rows 1, 16k, 16k + 1; very many of a lane a row
@pytest.mark.parametrize("qt,rows,cols", [(F32, 1, 32), (Q8_0, 16, 384), (Q5_0, 17, 416), (F16, 40, 960), (Q4_K, 5, 1024),
                                          (Q6_K, 33, 4864), (Q5_0, 65536, 32), (Q5_0, 65537, 64)])
def test_fp32_edges(ctx, oracle, qt, rows, cols):
    import tmq
    print(f"[single] fp32 type={qt} {rows}x{cols}", flush=True)
    w = synth.gen_weights(qt, rows, cols, 61 + rows)
    x = synth.gen_x(cols, 62 + cols)
    t = ctx.upload(qt, rows, cols, w)
    try:
        y = ctx.matmul_path(t, x, tmq.PATH_FP32)
    finally:
        t.free()
    assert np.array_equal(bits(y), bits(oracle.matmul_fp32(qt, w, x, rows, cols)))


# the last row count of the 16-row workgroups and the first of a lane a row, by
# type: 32, 48 and 60 rows a column, and the narrowest of them
@pytest.mark.parametrize("qt,cols", [(F32, 128), (F32, 160), (F16, 96), (F16, 128), (Q8_0, 160), (Q5_0, 128), (Q4_K, 256)])
def test_fp32_bounds(ctx, oracle, qt, cols):
    import tmq
    per = {F32: 32, F16: 48, Q8_0: 48}.get(qt, 60)
    x = synth.gen_x(cols, 63 + cols)
    for rows in (per * cols, per * cols + 1):
        print(f"[single] fp32 type={qt} {rows}x{cols}", flush=True)
        w = synth.gen_weights(qt, rows, cols, 64 + cols)
        t = ctx.upload(qt, rows, cols, w)
        try:
            y = ctx.matmul_path(t, x, tmq.PATH_FP32)
        finally:
            t.free()
        assert np.array_equal(bits(y), bits(oracle.matmul_fp32(qt, w, x, rows, cols))), rows


# the 16-row MFMA GEMVs: 1 and 3 blocks of a step's 4, 8 waves' worth (32) and
# one step more, the widest; one and two super-blocks, more than 8 waves', the
# bounds of the x registers (1024, 5120); rows 1, 16k, 16k + 1, and the first
# row count past the rule
@pytest.mark.parametrize("qt,rows,cols", [
    (Q5_0, 1, 32), (Q5_0, 17, 96), (Q5_0, 48, 1024), (Q5_0, 65, 1056), (Q5_0, 16, 8192), (Q5_0, 16385, 96),
    (Q4_K, 1, 256), (Q4_K, 33, 1024), (Q4_K, 64, 1280), (Q4_K, 15, 8192),
    (Q6_K, 1, 256), (Q6_K, 31, 512), (Q6_K, 80, 5120), (Q6_K, 17, 5376), (Q6_K, 4097, 8192),
    (Q6_K, 12288, 256), (Q6_K, 12289, 256), (Q4_K, 12289, 256), (Q4_K, 12289, 1280)])
@pytest.mark.parametrize("force", [0, 1])
def test_fpga_edges(ctx, oracle, monkeypatch, qt, rows, cols, force):
    if force and rows * cols > 1 << 22:
        pytest.skip("millions of corrections, of a path that the smaller ones take")
    print(f"[single] fpga type={qt} {rows}x{cols} force={force}", flush=True)
    if force:
        monkeypatch.setenv("TMQ_IFIT_FORCE", "1")
    w = synth.gen_weights(qt, rows, cols, 71 + rows)
    x = synth.gen_x(cols, 72 + cols)
    t = ctx.upload(qt, rows, cols, w)
    try:
        acc, xs = ctx.partials(t, x)
        y = ctx.matmul(t, x)
        z = ctx.matmul(t, np.zeros_like(x))
    finally:
        t.free()
    assert xs == oracle.quantize_act(x)[1]
    assert np.array_equal(bits(y), bits(oracle.matmul(qt, w, x, rows, cols)))
    assert np.array_equal(bits(z), bits(oracle.matmul(qt, w, np.zeros_like(x), rows, cols)))
    assert np.array_equal(acc, oracle.acc(qt, w, rows, cols, oracle.quantize_act(x)[0], oracle.row_inv(qt, w, rows, cols)))


@pytest.mark.parametrize("path", ["int16", "fpga"])
def test_result_over_activation(ctx, oracle, path):
    """y written where x lies: every row still reads the whole x"""
    import torch
    import tmq
    n = 896
    w = synth.gen_weights(Q5_0, n, n, 51)
    x = synth.gen_x(n, 52)
    want = oracle.matmul_int16(Q5_0, w, x, n, n)[0] if path == "int16" else oracle.matmul(Q5_0, w, x, n, n)
    t = ctx.upload(Q5_0, n, n, w)
    try:
        for off in (0, 64, -64):
            buf = torch.zeros(n + 128, dtype=torch.float32, device="cuda")
            buf[64:64 + n] = torch.from_numpy(x)
            torch.cuda.synchronize()
            xp, yp = buf.data_ptr() + 256, buf.data_ptr() + 256 + 4 * off
            if path == "int16":
                ctx.gemv_dev_path(t, tmq.PATH_INT16, xp, yp)
            else:
                (ctx.gemv_dev if off else ctx.gemv_dev_noalloc)(t, xp, yp)
            ctx.sync()
            assert np.array_equal(bits(buf[64 + off:64 + off + n].cpu().numpy()), bits(want)), off
    finally:
        t.free()


# one 16-row workgroup, the last row count of one wave, the first of several,
# and several workgroups' worth; y before, on and behind the start of x
@pytest.mark.parametrize("rows", [16, 17, 40, 64, 65, 896])
def test_fp32_result_over_activation(ctx, oracle, rows):
    """the same of the FP32 branch, whose 16-row workgroups read x while others store"""
    import torch
    import tmq
    n = 896
    print(f"[single] fp32 in place {rows}x{n}", flush=True)
    w = synth.gen_weights(Q5_0, rows, n, 53 + rows)
    x = synth.gen_x(n, 54)
    want = oracle.matmul_fp32(Q5_0, w, x, rows, n)
    t = ctx.upload(Q5_0, rows, n, w)
    try:
        for off in (0, 64, -8, n - 4):
            buf = torch.zeros(3 * n, dtype=torch.float32, device="cuda")
            buf[64:64 + n] = torch.from_numpy(x)
            torch.cuda.synchronize()
            ctx.gemv_dev_path(t, tmq.PATH_FP32, buf.data_ptr() + 256, buf.data_ptr() + 256 + 4 * off)
            ctx.sync()
            assert np.array_equal(bits(buf[64 + off:64 + off + rows].cpu().numpy()), bits(want)), off
    finally:
        t.free()


def chain_of(ctx, torch, shapes, share=None):
    """(chain, xs, x host, y, weights) of (type, rows, cols, activation) rows"""
    import tmq
    per = {Q5_0: 8, Q8_0: 64, Q4_K: 56, Q6_K: 32}
    xh = {a: synth.gen_x(c, 90 + a) for _, _, c, a in shapes}
    xs = {a: torch.from_numpy(x).cuda() for a, x in xh.items()}
    ys = [torch.zeros(r, dtype=torch.float32, device="cuda") for _, r, _, _ in shapes]
    if share:  # y of one descriptor over x of another
        ys[share[0]] = xs[share[1]]
    ws, descs, ts = [], [], []
    for i, (qt, r, c, a) in enumerate(shapes):
        w = synth.gen_weights(qt, r, c, 80 + i)
        t = ctx.upload(qt, r, c, w)
        p = max(k for k in range(1, per[qt] + 1) if r % k == 0)
        cg = c // 256 if qt in (Q4_K, Q6_K) else 1
        descs.append((t, xs[a].data_ptr(), ys[i].data_ptr(), None, r // p * cg, p, cg))
        ws.append(w)
        ts.append(t)
    torch.cuda.synchronize()
    return tmq.Chain(ctx, descs), xs, xh, ys, ws


# every decoder of the one-launch chain with a ragged last workgroup: 16- and
# 64-row Q5_0, wide Q5_0, Q8_0 of one half tile and of 8 waves' tiles and one
# more, both K-quants at both register bounds
CHAIN = [(Q5_0, 2050, 896, 0), (Q5_0, 17, 896, 0), (Q5_0, 33, 2048, 1), (Q8_0, 65, 96, 2), (Q8_0, 70, 544, 3),
         (Q4_K, 9, 256, 4), (Q6_K, 18, 4864, 5), (Q4_K, 17, 5376, 6), (Q6_K, 31, 256, 4)]


def test_chain_one_launch(ctx, oracle):
    import torch
    ch, xs, xh, ys, ws = chain_of(ctx, torch, CHAIN)
    want = [oracle.matmul(qt, w, xh[a], r, c) for (qt, r, c, a), w in zip(CHAIN, ws)]
    for rep in range(3):
        for y in ys:
            y.zero_()
        torch.cuda.synchronize()
        # the third time from the activations the last run prepared
        (ch.launch if rep == 2 else ch.run)()
        ctx.sync()
        for (qt, r, c, a), y, e in zip(CHAIN, ys, want):
            assert np.array_equal(bits(y.cpu().numpy()), bits(e)), (rep, qt, r, c)
        if rep == 1:
            for x in xs.values():
                x.zero_()
            torch.cuda.synchronize()
    ch.free()


# Q6_K of 6144 and of 8192 columns (two and one workgroup a CU) on either side
# of their bounds: 32 and 33, 16 and 17 tensors of 256 rows on 256 CUs
@pytest.mark.parametrize("cols,n", [(6144, 32), (6144, 33), (8192, 16), (8192, 17)])
def test_chain_one_bounds(ctx, oracle, cols, n):
    import torch
    import tmq
    rows = 256
    print(f"[single] chain of {n} q6_k {rows}x{cols}", flush=True)
    x = synth.gen_x(cols, 95)
    w = synth.gen_weights(Q6_K, rows, cols, 96)
    want = oracle.matmul(Q6_K, w, x, rows, cols)
    t = ctx.upload(Q6_K, rows, cols, w)
    xd = torch.from_numpy(x).cuda()
    ys = [torch.zeros(rows, dtype=torch.float32, device="cuda") for _ in range(n)]
    torch.cuda.synchronize()
    ch = tmq.Chain(ctx, [(t, xd.data_ptr(), y.data_ptr(), None, 8 * (cols // 256), 32, cols // 256) for y in ys])
    ch.run()
    ctx.sync()
    for i, y in enumerate(ys):
        assert np.array_equal(bits(y.cpu().numpy()), bits(want)), i
    ch.free()
    t.free()


def test_chain_result_over_activation(ctx, oracle):
    """every activation is quantised before any result is stored"""
    import torch
    shapes = [(Q5_0, 896, 896, 0), (Q8_0, 100, 896, 1), (Q6_K, 20, 512, 2)]
    ch, xs, xh, ys, ws = chain_of(ctx, torch, shapes, share=(0, 1))
    ch.run()
    ctx.sync()
    for (qt, r, c, a), y, w in zip(shapes, ys, ws):
        assert np.array_equal(bits(y.cpu().numpy()), bits(oracle.matmul(qt, w, xh[a], r, c))), (qt, r, c)
    ch.free()


def test_chain_shared_result(ctx, oracle):
    """two descriptors of one result: the later format's launch wins, as ever"""
    import torch
    shapes = [(Q6_K, 32, 256, 0), (Q5_0, 32, 96, 1)]
    ch, xs, xh, ys, ws = chain_of(ctx, torch, shapes)
    y = ys[0].data_ptr()
    ch.free()
    import tmq
    ts = [ctx.upload(qt, r, c, w) for (qt, r, c, _), w in zip(shapes, ws)]
    ch = tmq.Chain(ctx, [(ts[0], xs[0].data_ptr(), y, None, 1, 32, 1), (ts[1], xs[1].data_ptr(), y, None, 4, 8, 1)])
    for _ in range(5):
        ch.run()
    ctx.sync()
    assert np.array_equal(bits(ys[0].cpu().numpy()), bits(oracle.matmul(Q6_K, ws[0], xh[0], 32, 256)))
    ch.free()


# both one-launch Q8_0 kernels around their bound, half tiles, batches
@pytest.mark.parametrize("rows,cols", [(1, 32), (9, 544), (7, 8192), (33, 9248), (8192, 96), (8193, 96), (8257, 544),
                                       (8193, 4096), (8200, 4128), (196608, 32), (196609, 32)])
def test_q8_edges(ctx, oracle, rows, cols):
    print(f"[single] q8_0 {rows}x{cols}", flush=True)
    w = synth.gen_weights(Q8_0, rows, cols, 31 + rows)
    x = synth.gen_x(cols, 32 + cols)
    t = ctx.upload(Q8_0, rows, cols, w)
    try:
        acc, xs = ctx.partials(t, x)
        y = ctx.matmul(t, x)
    finally:
        t.free()
    assert xs == oracle.quantize_act(x)[1]
    rs = oracle.q8_row_scale(oracle.row_max_abs_q8(w, rows, cols))
    assert np.array_equal(acc, oracle.tiles_q8(w, rows, cols, oracle.quantize_act(x)[0], rs).reshape(acc.shape))
    assert np.array_equal(bits(y), bits(oracle.matmul(Q8_0, w, x, rows, cols)))


# host vectors: x read over the bus (up to 1024 x 1024) or brought by a
# launch, y through the pinned buffer or, above its 4 MiB, copied
@pytest.mark.parametrize("rows,cols", [(1024, 1024), (1025, 1024), (1024, 1056), (1048577, 32)])
def test_host_vectors(ctx, oracle, rows, cols):
    import tmq
    print(f"[single] host {rows}x{cols}", flush=True)
    w = synth.gen_weights(Q5_0, rows, cols, 21 + cols)
    t = ctx.upload(Q5_0, rows, cols, w)
    try:
        for seed in (1, 2):
            x = synth.gen_x(cols, seed)
            assert np.array_equal(bits(ctx.matmul(t, x)), bits(oracle.matmul(Q5_0, w, x, rows, cols)))
        assert np.array_equal(bits(ctx.matmul_path(t, x, tmq.PATH_FP32)), bits(oracle.matmul_fp32(Q5_0, w, x, rows, cols)))
    finally:
        t.free()

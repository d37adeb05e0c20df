"""The f32 products on the bf16 matrix cores (three bf16 pieces per operand) through the entry points that use them, at the edges of
their tiles: rows around 32 / 64 / a second tile, output widths that end inside a 128-column tile, more layers than one launch
takes, both FFN forms.  Against float64 (cross K/V, weights with all 24 bits and rows of very different size) and the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,width,xw,layers", [(17, 64, 32, 1), (32, 128, 64, 2), (64, 192, 160, 3), (65, 128, 96, 34), (129, 768, 768, 2)])
def test_cross_kv_tiles(backend, pkg, orc, rows, width, xw, layers):
    print("[gpu-case] cross K/V rows=%d width=%d xw=%d layers=%d" % (rows, width, xw, layers), flush=True)
    rng = np.random.default_rng(rows)
    backend.set_quant(pkg.F32)
    gains = [backend.keep((1.0 + 0.1 * rng.standard_normal(width)).astype(np.float32)) for _ in range(layers)]
    scale = (10.0 ** rng.uniform(-12, 12, size=(2 * xw, 1))).astype(np.float32)
    kvw = [backend.keep(rng.standard_normal((2 * xw, width)).astype(np.float32) * scale) for _ in range(layers)]
    memory = rng.standard_normal((rows, width)).astype(np.float32)
    dmem = backend.alloc(rows * width).write(memory)
    guard = np.full(xw, 7.0, np.float32)
    dk, dv = (backend.alloc(layers * rows * xw + xw).write(guard, layers * rows * xw) for _ in range(2))
    backend.cross_kv_dev(dmem.ptr, rows, width, gains, None, kvw, xw, dk.ptr, dv.ptr)
    gk, gv = dk.read(), dv.read()
    assert np.array_equal(gk[-xw:], guard) and np.array_equal(gv[-xw:], guard)
    got = np.concatenate([gk[:-xw].reshape(layers, rows, xw), gv[:-xw].reshape(layers, rows, xw)], axis=2)
    for l in (0, layers // 2, layers - 1):
        normed = np.stack([orc.layernorm(r, gains[l], None) for r in memory]).astype(np.float64)
        want = normed @ kvw[l].astype(np.float64).T
        err = np.linalg.norm(got[l] - want, axis=0) / np.linalg.norm(want, axis=0)     # per output: their sizes span 24 decades
        assert err.max() < 2e-6, (l, float(err.max()))
    for d in (dmem, dk, dv):
        d.free()


@pytest.mark.parametrize("rows,xw,layers", [(5, 32, 9), (17, 32, 9), (64, 224, 5), (130, 96, 3), (100, 768, 12), (130, 448, 12), (65, 768, 33)])
def test_cross_kv_layers_together(backend, pkg, rows, xw, layers):
    """The layers' column tiles share one list: counts that no multiple of eight divides, a last tile that is not full (17 rows of 32 columns:
    nine tiles, each half empty), and every layer's values are those of a call for that layer alone, bit for bit.  (Five rows of this width
    go layer by layer; of twelve layers, 100 rows by 768 and 130 by 448, each starts at a place of its own in the list.)"""
    print("[gpu-case] cross K/V together rows=%d xw=%d layers=%d" % (rows, xw, layers), flush=True)
    rng, width = np.random.default_rng(rows + layers), 128
    backend.set_quant(pkg.F32)
    gains = [backend.keep((1.0 + 0.1 * rng.standard_normal(width)).astype(np.float32)) for _ in range(layers)]
    kvw = [backend.keep(rng.standard_normal((2 * xw, width)).astype(np.float32)) for _ in range(layers)]
    dmem = backend.alloc(rows * width).write(rng.standard_normal((rows, width)).astype(np.float32))
    dk, dv = (backend.alloc(layers * rows * xw) for _ in range(2))
    one_k, one_v = (backend.alloc(rows * xw) for _ in range(2))
    backend.cross_kv_dev(dmem.ptr, rows, width, gains, None, kvw, xw, dk.ptr, dv.ptr)
    k, v = dk.read().reshape(layers, -1), dv.read().reshape(layers, -1)
    for l in range(layers):
        backend.cross_kv_dev(dmem.ptr, rows, width, [gains[l]], None, [kvw[l]], xw, one_k.ptr, one_v.ptr)
        assert np.array_equal(one_k.read(), k[l]) and np.array_equal(one_v.read(), v[l]), l
    for d in (dmem, dk, dv, one_k, one_v):
        d.free()


@pytest.mark.parametrize("storage", ["F32", "F16", "INT8", "INT4"])
@pytest.mark.parametrize("rows,xw,layers", [(3, 768, 2), (4, 36, 1), (5, 96, 34), (8, 768, 1), (9, 768, 3), (16, 160, 2)])
def test_cross_kv_few_rows_as_a_list(backend, pkg, storage, rows, xw, layers):
    """Three to sixteen rows of width 768: every layer's products in one launch (more than 32 layers: two).  A row's values are those of a call
    for that row and layer alone, which takes the matvecs one by one, bit for bit."""
    print("[gpu-case] cross K/V list %s rows=%d xw=%d layers=%d" % (storage, rows, xw, layers), flush=True)
    rng, width = np.random.default_rng(rows + layers), 768
    backend.set_quant(getattr(pkg, storage))
    try:
        gains = [backend.keep((1.0 + 0.1 * rng.standard_normal(width)).astype(np.float32)) for _ in range(layers)]
        biases = [backend.keep((0.02 * rng.standard_normal(width)).astype(np.float32)) for _ in range(layers)] if rows % 2 else None
        kvw = [backend.keep(rng.standard_normal((2 * xw, width)).astype(np.float32)) for _ in range(layers)]
        dmem = backend.alloc(rows * width).write(rng.standard_normal((rows, width)).astype(np.float32))
        guard = np.full(xw, 7.0, np.float32)
        dk, dv = (backend.alloc(layers * rows * xw + xw).write(guard, layers * rows * xw) for _ in range(2))
        one_k, one_v = (backend.alloc(xw) for _ in range(2))
        for _ in range(2):
            backend.cross_kv_dev(dmem.ptr, rows, width, gains, biases, kvw, xw, dk.ptr, dv.ptr)
        k, v = dk.read(), dv.read()
        assert np.array_equal(k[-xw:], guard) and np.array_equal(v[-xw:], guard)
        k, v = k[:-xw].reshape(layers, rows, xw), v[:-xw].reshape(layers, rows, xw)
        for l in sorted({0, layers // 2, layers - 1}):
            for r in range(rows):
                backend.cross_kv_dev(dmem.ptr + 4 * r * width, 1, width, [gains[l]], [biases[l]] if biases else None, [kvw[l]], xw, one_k.ptr, one_v.ptr)
                assert np.array_equal(one_k.read(), k[l, r]) and np.array_equal(one_v.read(), v[l, r]), (l, r)
        for d in (dmem, dk, dv, one_k, one_v):
            d.free()
    finally:
        backend.set_quant(pkg.F32)


def test_cross_kv_few_rows_of_many_wide_layers(backend, pkg):
    """A list of products so long and wide that its rows per workgroup reach what a launch's packed arguments hold: taken like any other, every
    layer's values those of a call for that layer alone."""
    rows, width, xw, layers = 3, 768, 49152, 32
    print("[gpu-case] cross K/V list of %d layers of %d" % (layers, xw), flush=True)
    rng = np.random.default_rng(5)
    backend.set_quant(pkg.F32)
    gains = [backend.keep((1.0 + 0.1 * rng.standard_normal(width)).astype(np.float32)) for _ in range(layers)]
    kvw = backend.keep(rng.standard_normal((2 * xw, width), dtype=np.float32))     # one tensor for all: their normalised rows differ
    dmem = backend.alloc(rows * width).write(rng.standard_normal((rows, width)).astype(np.float32))
    dk, dv = (backend.alloc(layers * rows * xw) for _ in range(2))
    one_k, one_v = (backend.alloc(rows * xw) for _ in range(2))
    backend.cross_kv_dev(dmem.ptr, rows, width, gains, None, [kvw] * layers, xw, dk.ptr, dv.ptr)
    k, v = dk.read().reshape(layers, -1), dv.read().reshape(layers, -1)
    for l in (0, 1, 17, layers - 1):
        backend.cross_kv_dev(dmem.ptr, rows, width, [gains[l]], None, [kvw], xw, one_k.ptr, one_v.ptr)
        assert np.array_equal(one_k.read(), k[l]) and np.array_equal(one_v.read(), v[l]), l
    for d in (dmem, dk, dv, one_k, one_v):
        d.free()


@pytest.mark.parametrize("kernel", [1, 3])
@pytest.mark.parametrize("tokens", [31, 32, 33, 64, 65, 97])
def test_encoder_f32_tiles(backend, pkg, orc, synth, nerr, kernel, tokens):
    print("[gpu-case] encoder f32 tokens=%d kernel=%d" % (tokens, kernel), flush=True)
    cfg = dict(synth.encoder_config(layers=2, width=192, heads=3, ffn=320, vocab=64, max_positions=128), causal=tokens % 2 == 0, ffn_kernel=kernel)
    w = synth.encoder_weights_f16(cfg, seed=90 + kernel, kernel=kernel)
    ids = np.random.default_rng(tokens).integers(0, cfg["vocab"], size=tokens).astype(np.int32)
    enc = pkg.Encoder(backend, dict(cfg, operands_f32=True), w)
    dout = backend.alloc(tokens * cfg["width"])
    enc.prefill(ids, 0, dout.ptr)
    got = dout.read().reshape(tokens, cfg["width"])
    enc.destroy()
    bits = {"tok_table": "tok_table", "pos_table": "pos_table", "qkv_w": "qkv", "o_w": "o", "up_w": "up", "down_w": "down"}
    packed = {k: w[v].astype(np.float16).view(np.uint16) for k, v in bits.items()}
    packed.update({k: w.get(k) for k in ("norm1_g", "norm1_b", "norm2_g", "norm2_b", "norm_out_g", "norm_out_b")})
    _, want = orc.encoder_prefill(cfg, packed, ids)
    assert nerr(got, want) < 1e-5


def test_one_buffer_under_two_shapes(backend, pkg, orc):
    """A weight's stored form may depend on its shape (the order of a split product's blocks and of a convolution's, the scales of int8
    rows): the same memory used under two shapes of equal size gives each its own products."""
    print("[gpu-case] one weight buffer, two shapes", flush=True)
    rng = np.random.default_rng(5)
    shared = backend.keep(rng.standard_normal(128 * 64).astype(np.float32))
    rows = 40
    backend.set_quant(pkg.F32)
    for width, xw in ((128, 32), (64, 64)):
        gain = backend.keep(np.ones(width, np.float32))
        memory = rng.standard_normal((rows, width)).astype(np.float32)
        dmem, dk, dv = backend.alloc(rows * width).write(memory), backend.alloc(rows * xw), backend.alloc(rows * xw)
        backend.cross_kv_dev(dmem.ptr, rows, width, [gain], None, [shared], xw, dk.ptr, dv.ptr)
        got = np.concatenate([dk.read().reshape(rows, xw), dv.read().reshape(rows, xw)], axis=1)
        want = np.stack([orc.layernorm(r, gain, None) for r in memory]).astype(np.float64) @ shared.reshape(2 * xw, width).astype(np.float64).T
        assert np.linalg.norm(got - want) < 2e-6 * np.linalg.norm(want), (width, xw)
        for d in (dmem, dk, dv):
            d.free()
    for out_ch, in_ch in ((64, 128), (128, 64)):
        x, w = rng.standard_normal((in_ch, 70)).astype(np.float32), shared.reshape(out_ch, in_ch, 1)
        dx, dy = backend.alloc(x.size).write(x), backend.alloc(out_ch * 70)
        backend.conv1d(dx.ptr, dy.ptr, in_ch, out_ch, 70, 1, 1, w, None)
        want = w[:, :, 0].astype(np.float64) @ x.astype(np.float64)
        assert np.linalg.norm(dy.read().reshape(want.shape) - want) < 2e-6 * np.linalg.norm(want), (out_ch, in_ch)
        dx.free()
        dy.free()
    backend.set_quant(pkg.INT8)
    for n, k in ((64, 128), (128, 64)):
        w, x = shared.reshape(n, k), rng.standard_normal((1, k)).astype(np.float32)
        want = x.astype(np.float64) @ w.astype(np.float64).T
        # both factors rounded to int8: a step of 1 / 127 of the largest value, uniform, over k terms -- about 1e-2 of the product's norm
        assert np.linalg.norm(backend.matmul(x, w) - want) < 3e-2 * np.linalg.norm(want), (n, k)
    backend.set_quant(pkg.F32)


def test_cross_kv_extremes(backend, pkg, orc):
    """Operands without three finite bf16 pieces: infinities, NaN, values from 2^128 - 2^119 on.  What f32 multiply-adds give, and only in
    the outputs that they enter."""
    print("[gpu-case] cross K/V extremes", flush=True)
    rng = np.random.default_rng(8)
    backend.set_quant(pkg.F32)
    rows, width, xw = 70, 128, 96
    gain = backend.keep(np.full(width, 0.2, np.float32))
    memory = rng.standard_normal((rows, width)).astype(np.float32)
    memory[5, 3] = np.inf                                   # a row of NaN behind the LayerNorm: the other rows do not change
    w = rng.standard_normal((2 * xw, width)).astype(np.float32)
    w[7, 11], w[8, 12], w[9, 13] = np.inf, -np.inf, np.nan
    w[100, 20:22] = np.inf, -np.inf
    w[40, 2], w[41, 127] = 3.4028235e38, -3.3962e38          # finite sums: |normed| < 1 there nearly everywhere
    w[42, 60] = 3.396e38                                     # just below the limit
    w = backend.keep(w)
    dmem, dk, dv = backend.alloc(rows * width).write(memory), backend.alloc(rows * xw), backend.alloc(rows * xw)
    backend.cross_kv_dev(dmem.ptr, rows, width, [gain], None, [w], xw, dk.ptr, dv.ptr)
    got = np.concatenate([dk.read().reshape(rows, xw), dv.read().reshape(rows, xw)], axis=1).astype(np.float64)
    with np.errstate(invalid="ignore"):
        normed = np.stack([orc.layernorm(r, gain, None) for r in memory]).astype(np.float64)
        want = normed @ w.astype(np.float64).T               # beyond f32's range: an infinity of that sign
        want = np.where(np.abs(want) > 3.4028235e38, np.sign(want) * np.inf, want)
    assert np.isnan(got[5]).all()
    keep = np.arange(rows) != 5
    got, want = got[keep], want[keep]
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isinf(want[:, [7, 8]]).all() and np.isnan(want[:, 9]).all()
    assert np.isnan(want[:, 100]).any() and np.isinf(want[:, 100]).any()   # (as the two factors' signs differ or agree)
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    finite = np.isfinite(want)
    assert finite[:, [40, 41, 42]].mean() > 0.9
    # (a normalised value near zero carries the rounding of its row's mean, up to 2^-23, whatever its own size)
    size = np.nan_to_num(np.abs(w.astype(np.float64)), posinf=0)
    allowed = 2e-6 * np.abs(normed[keep]) @ size.T + 2.0 ** -23 * size.sum(axis=1)
    assert (np.abs(got[finite] - want[finite]) < allowed[finite]).all()
    for d in (dmem, dk, dv):
        d.free()


@pytest.mark.parametrize("taps", [1, 3])
def test_encoder_f32_large_weights(backend, pkg, synth, nerr, taps):
    """A value row and an FFN row that fill f32's range, their products scaled back by the weights behind them: the same stack as with both
    in the ordinary range (powers of two throughout; the FFN row's GELU is saturated in both)."""
    print("[gpu-case] encoder f32, weights at the range's end, taps=%d" % taps, flush=True)
    cfg = dict(synth.encoder_config(layers=1, width=128, heads=2, ffn=192, vocab=32, max_positions=64), causal=True, ffn_kernel=taps, operands_f32=True)
    rng = np.random.default_rng(taps)
    normal = lambda *shape: (0.02 * rng.standard_normal(shape)).astype(np.float32)
    base = {"tok_table": normal(32, 128), "pos_table": normal(64, 128), "qkv": normal(1, 384, 128), "o": normal(1, 128, 128),
            "up": normal(1, 192, 128 * taps), "down": normal(1, 128, 192 * taps), "norm_out_g": np.ones(128, np.float32), "norm_out_b": None}
    for name in ("norm1", "norm2"):
        base[name + "_g"], base[name + "_b"] = np.full((1, 128), 1e-3, np.float32), None
    top = np.float32(3.4e38 * 2.0 ** -128)                   # at 2^128 times its size above the first piece's range
    base["qkv"][0, 256 + 70, 9] = base["up"][0, 33, 5 * taps] = top
    base["o"][0, :, 70] = rng.standard_normal(128) * 2.0 ** 30    # (scaled back: 2^-98, above the range in which an operand loses bits)
    base["up"][0, 33] *= np.float32(2.0 ** 44)               # (GELU differs from max(x, 0) by 0.17 at most: 1e-11 of such values)
    base["down"].reshape(1, 128, 192, taps)[0, :, 33] *= np.float32(2.0 ** -10)
    large = {k: None if v is None else v.copy() for k, v in base.items()}
    large["qkv"][0, 256 + 70] *= np.float32(2.0 ** 64)
    large["qkv"][0, 256 + 70] *= np.float32(2.0 ** 64)
    large["o"][0, :, 70] *= np.float32(2.0 ** -64)
    large["o"][0, :, 70] *= np.float32(2.0 ** -64)
    large["up"][0, 33] *= np.float32(2.0 ** 84)
    large["down"].reshape(1, 128, 192, taps)[0, :, 33] *= np.float32(2.0 ** -84)
    ids = rng.integers(0, 32, size=41).astype(np.int32)
    out = []
    for w in (base, large):
        enc = pkg.Encoder(backend, cfg, w)
        dout = backend.alloc(41 * 128)
        enc.prefill(ids, 0, dout.ptr)
        out.append(dout.read())
        enc.destroy()
        dout.free()
    assert np.isfinite(out[1]).all()
    assert nerr(out[1], out[0]) < 1e-5


def test_cross_kv_tiny_weights(backend, pkg, orc):
    """Below 2^-110 an operand keeps fewer than its 24 bits: its third piece ends at bf16's smallest subnormal, 2^-133, so that at most half
    of that is lost."""
    print("[gpu-case] cross K/V, tiny weights", flush=True)
    rng = np.random.default_rng(9)
    backend.set_quant(pkg.F32)
    rows, width, xw = 33, 64, 64
    gain = backend.keep(np.ones(width, np.float32))
    memory = rng.standard_normal((rows, width)).astype(np.float32)
    w = backend.keep((rng.standard_normal((2 * xw, width)) * np.exp2(rng.integers(-126, -105, size=(2 * xw, 1)))).astype(np.float32))
    dmem, dk, dv = backend.alloc(rows * width).write(memory), backend.alloc(rows * xw), backend.alloc(rows * xw)
    backend.cross_kv_dev(dmem.ptr, rows, width, [gain], None, [w], xw, dk.ptr, dv.ptr)
    got = np.concatenate([dk.read().reshape(rows, xw), dv.read().reshape(rows, xw)], axis=1).astype(np.float64)
    normed = np.stack([orc.layernorm(r, gain, None) for r in memory]).astype(np.float64)
    want, lost = normed @ w.astype(np.float64).T, np.abs(normed).sum(axis=1, keepdims=True) * 2.0 ** -134
    rounding = 2e-6 * np.abs(normed) @ np.abs(w.astype(np.float64)).T + width * 2.0 ** -150
    over = (np.abs(got - want) - rounding) / lost
    print("largest loss, of half a smallest subnormal a term: %g" % over.max(), flush=True)
    assert over.max() < 1.0
    for d in (dmem, dk, dv):
        d.free()


def test_workspace_and_weight_memory(backend, pkg, synth):
    """What the encoder with f32 operands allocates follows the partial sums that its products can leave (tiles times splits are at most the
    chip's CUs), and a packed convolution weight is its steps and the three that are requested ahead."""
    import ctypes

    def free():
        values = ctypes.c_size_t(), ctypes.c_size_t()
        assert backend.lib.hipMemGetInfo(ctypes.byref(values[0]), ctypes.byref(values[1])) == 0   # (the runtime that the library is linked to)
        return values[0].value

    print("[gpu-case] memory of the f32 encoder and of a convolution weight", flush=True)
    cfg = dict(synth.encoder_config(layers=1, width=768, heads=12, ffn=3072, vocab=32, max_positions=1024), causal=True, ffn_kernel=1, operands_f32=True)
    w = synth.encoder_weights_f16(cfg, seed=4, kernel=1)
    backend.sync()
    before, kept = free(), backend.cached_weight_bytes()
    enc = pkg.Encoder(backend, cfg, w)
    used = before - free() - (backend.cached_weight_bytes() - kept)
    enc.destroy()
    rows = 1024 * 4 * (4 * 768 + 2 * 768 + 3072)                             # x, normalised, context, q/k/v, hidden
    partial = 4 * max(256 * 64 * 128, 1024 * 3072)
    staging = 4 * 768 * 3072                                                 # the backend's own, for the largest weight
    assert used < rows + partial + staging + (16 << 20), used                # (allocations are rounded up to 2 MiB)
    kept = backend.cached_weight_bytes()
    conv = np.ones((40, 33, 7), np.float32)
    x, y = backend.alloc(33 * 10), backend.alloc(40 * 10)
    backend.conv1d(x.ptr, y.ptr, 33, 40, 10, 7, 1, conv, None)
    assert backend.cached_weight_bytes() - kept == (2 * 3 * 7 + 3) * 3072
    x.free()
    y.free()


@pytest.mark.parametrize("bias", ["none", "all", "some"])
@pytest.mark.parametrize("rows", [65, 128, 129, 193, 256, 257, 300])
def test_cross_kv_wide_tiles(backend, pkg, orc, rows, bias):
    """More rows than one 64-row tile: the last row of a tile and the first of the next, widths that end inside a 128-column tile, with and
    without LayerNorm biases (and in only some of the layers), an infinity in one row."""
    print("[gpu-case] cross K/V wide rows=%d bias=%s" % (rows, bias), flush=True)
    rng = np.random.default_rng(rows)
    backend.set_quant(pkg.F32)
    width, xw, layers = 128, 96, 3
    gains = [backend.keep((1.0 + 0.1 * rng.standard_normal(width)).astype(np.float32)) for _ in range(layers)]
    biases = [backend.keep(rng.standard_normal(width).astype(np.float32)) if bias == "all" or (bias == "some" and l == 1) else None for l in range(layers)]
    kvw = [backend.keep(rng.standard_normal((2 * xw, width)).astype(np.float32)) for _ in range(layers)]
    memory = rng.standard_normal((rows, width)).astype(np.float32)
    memory[rows - 2, 5] = np.inf
    dmem = backend.alloc(rows * width).write(memory)
    guard = np.full(xw, 7.0, np.float32)
    dk, dv = (backend.alloc(layers * rows * xw + xw).write(guard, layers * rows * xw) for _ in range(2))
    backend.cross_kv_dev(dmem.ptr, rows, width, gains, None if bias == "none" else biases, kvw, xw, dk.ptr, dv.ptr)
    gk, gv = dk.read(), dv.read()
    assert np.array_equal(gk[-xw:], guard) and np.array_equal(gv[-xw:], guard)
    got = np.concatenate([gk[:-xw].reshape(layers, rows, xw), gv[:-xw].reshape(layers, rows, xw)], axis=2).astype(np.float64)
    keep = np.arange(rows) != rows - 2
    assert np.isnan(got[:, rows - 2]).all()
    for l in range(layers):
        normed = np.stack([orc.layernorm(r, gains[l], biases[l]) for r in memory[keep]]).astype(np.float64)
        want = normed @ kvw[l].astype(np.float64).T
        assert np.linalg.norm(got[l][keep] - want) < 1e-6 * np.linalg.norm(want), l       # (f32 sums of 128 terms)
    for d in (dmem, dk, dv):
        d.free()


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("rows", [40, 70, 150, 256, 300])
def test_cross_kv_rows_of_different_size(backend, pkg, orc, rows, bias):
    """Rows that lie beside much larger ones in a tile (the LayerNorm's eps leaves a row of 1e-9 at 3e-7), and channels of very different
    gain under weights that make up for it: f32's accuracy in every row.  An infinity in one row changes no other, and a row's bits do not depend
    on how many are beside it."""
    print("[gpu-case] cross K/V rows of different size, %d, bias %s" % (rows, bias), flush=True)
    rng = np.random.default_rng(rows)
    backend.set_quant(pkg.F32)
    width, xw = 128, 96
    size = np.exp2(rng.choice([0, -6, -16, -24], size=(1, width))).astype(np.float32)
    gain = backend.keep(((1.0 + 0.1 * rng.standard_normal((1, width))) * size).astype(np.float32)[0])
    biases = [backend.keep((1e-8 * rng.standard_normal((1, width)) * size).astype(np.float32)[0])] if bias else None
    kvw = backend.keep((rng.standard_normal((2 * xw, width)) / size).astype(np.float32))
    memory = (rng.standard_normal((rows, width)) * 10.0 ** rng.choice([0, -5, -7, -9], size=(rows, 1))).astype(np.float32)
    infinite = rows // 3
    memory[infinite, 5] = np.inf
    dmem = backend.alloc(rows * width).write(memory)
    dk, dv = (backend.alloc(rows * xw) for _ in range(2))
    backend.cross_kv_dev(dmem.ptr, rows, width, [gain], biases, [kvw], xw, dk.ptr, dv.ptr)
    got = np.concatenate([dk.read().reshape(rows, xw), dv.read().reshape(rows, xw)], axis=1)
    assert np.isnan(got[infinite]).all()
    keep = np.arange(rows) != infinite
    normed = np.stack([orc.layernorm(r, gain, biases[0] if bias else None) for r in memory[keep]]).astype(np.float64)
    want = normed @ kvw.astype(np.float64).T
    # operands in full, f32 sums of 128 terms, and the rounding of the row's mean (some 2^-24 of the row): the bar of test_cross_kv_tiles, row by row
    err = np.linalg.norm(got[keep] - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() < 2e-6, float(err.max())
    some = min(50, rows)                                     # (up to 16 rows go through the matvecs, which add in another order)
    for first in {*range(0, rows - some, some), rows - some}:
        backend.cross_kv_dev(dmem.ptr + 4 * first * width, some, width, [gain], biases, [kvw], xw, dk.ptr, dv.ptr)
        part = np.concatenate([dk.read()[:some * xw].reshape(some, xw), dv.read()[:some * xw].reshape(some, xw)], axis=1)
        assert np.array_equal(part, got[first:first + some], equal_nan=True), first
    for d in (dmem, dk, dv):
        d.free()


@pytest.mark.parametrize("taps,tokens", [(1, 20), (1, 100), (3, 20), (3, 100)])
def test_encoder_f32_channels_of_different_size(backend, pkg, synth, taps, tokens):
    """LayerNorm gains of 2^-30 in some channels and 2^30 in the weights behind them: powers of two, so every product is the one of the even
    stack and the output is the same bits."""
    print("[gpu-case] encoder f32, channels of different size, taps=%d tokens=%d" % (taps, tokens), flush=True)
    cfg = dict(synth.encoder_config(layers=2, width=128, heads=2, ffn=192, vocab=32, max_positions=128), causal=True, ffn_kernel=taps, operands_f32=True)
    rng = np.random.default_rng(taps)
    normal = lambda *shape: (0.02 * rng.standard_normal(shape)).astype(np.float32)
    even = {"tok_table": normal(32, 128), "pos_table": normal(128, 128), "qkv": normal(2, 384, 128), "o": normal(2, 128, 128),
            "up": normal(2, 192, 128 * taps), "down": normal(2, 128, 192 * taps), "norm_out_g": np.ones(128, np.float32), "norm_out_b": None}
    for name in ("norm1", "norm2"):
        even[name + "_g"], even[name + "_b"] = (1.0 + normal(2, 128)), None
    uneven = {k: None if v is None else v.copy() for k, v in even.items()}
    quiet = rng.random(128) < 0.5
    for name, behind, each in (("norm1_g", "qkv", 1), ("norm2_g", "up", taps)):
        uneven[name][:, quiet] *= np.float32(2.0 ** -30)
        uneven[behind].reshape(2, -1, 128, each)[:, :, quiet] *= np.float32(2.0 ** 30)
    ids = rng.integers(0, 32, size=tokens).astype(np.int32)
    out = []
    for w in (even, uneven):
        enc = pkg.Encoder(backend, cfg, w)
        dout = backend.alloc(tokens * 128)
        enc.prefill(ids, 0, dout.ptr)
        out.append(dout.read())
        enc.destroy()
        dout.free()
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])

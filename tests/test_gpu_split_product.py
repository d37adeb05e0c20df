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

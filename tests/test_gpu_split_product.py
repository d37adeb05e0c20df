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

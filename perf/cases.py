"""Performance cases of the library: the calls a speech server makes, at the sizes it makes them.

An utterance is encoded (text-encoder prefill, cross-attention K/V), decoded frame by frame (decoder step with its output head,
local-transformer frame) for one to sixteen utterances at a time, and turned into samples by the codec.  Each case is one such
call, or for the codec one such sequence of calls, through the package's public entry points; `listed` holds named sizes and
`draw` gives further ones of the same ranges.  Model shapes are those of `synth` and of the benchmark: a 12-layer d = 768 decoder
with 12 x 64 heads and an 8 x 1024 head, a one-layer local transformer with 16 positions and 2048 codes, a six-layer encoder,
and the codec's five stages.

A process holds one backend for all states of a case, as a server does, and closes it with the last of them.  Every state has
weights, caches and inputs of its own, all made from its seed.
"""
import importlib
import math
import random
import weakref

import numpy as np
import torch

import __graft_entry__ as entry

pkg = entry.load_package()
synth = importlib.import_module(pkg.__name__ + ".synth")
codec = importlib.import_module(pkg.__name__ + ".codec")

STORAGE = {"f32": pkg.F32, "int8": pkg.INT8, "int4": pkg.INT4, "f16": pkg.F16}
STREAMS, LOCAL_VOCAB = 16, 2048                 # codebook positions of a frame, rows of each position's projection
HEAD_ROWS, HEAD_VOCAB = 8 * 1024, 1024          # output head: eight codebooks of 1024
RATES, KERNELS, DILATIONS, CODEC_CHANNELS = (8, 8, 4, 2, 2), (3, 7, 11), (1, 3, 5), 864
MAX_KEYS, MAX_MEMORY, MAX_TOKENS, MAX_TOKENS_F32, MAX_FRAMES = 2048, 256, 512, 192, 64


def _text(values):
    return ",".join(str(int(v)) for v in values)


def _numbers(text):
    return [int(v) for v in text.split(",")]


def listed():
    self8, cross8 = synth.ragged_lengths(8, seed=3)
    self16, cross16 = synth.ragged_lengths(16, seed=5)
    return [
        # the first frames of a short sentence spoken to one listener: nothing but latency
        {"name": "step int8, 1 stream, start", "kind": "step", "storage": "int8", "rows": "5", "memory": "19"},
        # one long utterance: the benchmark's decode step
        {"name": "step int8, 1 stream, 1024", "kind": "step", "storage": "int8", "rows": "1023", "memory": "256"},
        # a few listeners on the smallest storage
        {"name": "step int4, 3 streams", "kind": "step", "storage": "int4", "rows": "611,1339,87", "memory": "101,230,48"},
        # continuous batching: the benchmark's eight ragged streams
        {"name": "step int8, 8 streams", "kind": "step", "storage": "int8", "rows": _text(n - 1 for n in self8), "memory": _text(cross8)},
        # a full server that keeps its weights in half precision
        {"name": "step f16, 16 streams", "kind": "step", "storage": "f16", "rows": _text(n - 1 for n in self16), "memory": _text(cross16)},
        # the sixteen tokens of a frame, sampled as the model's usual setting does (top 80, temperature 0.6)
        {"name": "local frame int8, 1 stream", "kind": "local", "storage": "int8", "batch": 1, "topk": 80, "temperature": 0.6},
        {"name": "local frame int8, 8 streams", "kind": "local", "storage": "int8", "batch": 8, "topk": 50, "temperature": 0.8},
        # a paragraph through the text encoder on f16 operands: the benchmark's prefill
        {"name": "prefill f16, 256 tokens", "kind": "prefill", "operands": "f16", "causal": False, "taps": 1, "tokens": 256},
        # a few sentences in the reference's own form and precision: causal, kernel-3 FFN, f32
        {"name": "prefill f32 causal, 192 tokens", "kind": "prefill", "operands": "f32", "causal": True, "taps": 3, "tokens": 192},
        # the encoded text handed to the decoder: cross-attention K/V of every layer
        {"name": "cross K/V, 180 tokens", "kind": "cross_kv", "tokens": 180},
        # samples: a short chunk for a listener who is waiting, and the benchmark's 64 frames
        {"name": "codec, 5 frames", "kind": "codec", "frames": 5},
        {"name": "codec, 64 frames", "kind": "codec", "frames": 64},
    ]


def _spread(rng, low, high):
    """A whole number of [low, high], evenly over its logarithm."""
    return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))


def draw(rng):
    kind = rng.choice(("step", "step", "step", "local", "local", "prefill", "prefill", "cross_kv", "codec"))
    if kind == "step":
        batch = _spread(rng, 1, 16)
        return {"kind": "step", "storage": rng.choice(("int8", "int8", "int4", "f16", "f32")),
                "rows": _text(_spread(rng, 1, MAX_KEYS - 1) for _ in range(batch)),
                "memory": _text(_spread(rng, 8, MAX_MEMORY) for _ in range(batch))}
    if kind == "local":
        return {"kind": "local", "storage": rng.choice(("int8", "int8", "int4", "f16", "f32")), "batch": _spread(rng, 1, 16),
                "topk": _spread(rng, 1, 100), "temperature": round(rng.uniform(0.4, 1.2), 2)}
    if kind == "prefill":
        operands = rng.choice(("f16", "f32"))
        return {"kind": "prefill", "operands": operands, "causal": rng.random() < 0.5, "taps": rng.choice((1, 3)),
                "tokens": _spread(rng, 4, MAX_TOKENS if operands == "f16" else MAX_TOKENS_F32)}
    if kind == "cross_kv":
        return {"kind": "cross_kv", "tokens": _spread(rng, 8, MAX_MEMORY)}
    return {"kind": "codec", "frames": _spread(rng, 2, MAX_FRAMES)}


# ---- what a program holds --------------------------------------------------------------------------------------------

class _Engine:
    """The process's backend; it closes when the last state that uses it is gone."""
    current = None

    def __init__(self):
        self.backend = pkg.Backend()
        weakref.finalize(self, self.backend.close)

    @classmethod
    def get(cls):
        engine = cls.current() if cls.current is not None else None
        if engine is None:
            engine = cls()
            cls.current = weakref.ref(engine)
        return engine


class _State:
    """One case's handles and buffers.  `call` makes the pass and leaves its results in `results` (device buffers) or
    returns them (what the entry point itself hands to the host)."""

    def __init__(self, case, seed):
        self.engine = _Engine.get()
        self.backend = self.engine.backend
        self.gen = torch.Generator("cuda").manual_seed(int(seed))
        self.rng = random.Random(int(seed))
        self.results, self.call = None, None
        _PREPARE[case["kind"]](self, case)

    def normal(self, shape, std=1.0, mean=0.0):
        return torch.empty(shape, device="cuda", dtype=torch.float32).normal_(mean, std, generator=self.gen)

    def host(self, shape, std=1.0, mean=0.0):
        return self.normal(shape, std, mean).cpu().numpy()

    def owns(self, handle):
        """The handle is destroyed with the state and before its backend closes."""
        weakref.finalize(self, lambda h, engine: h.destroy(), handle, self.engine)
        return handle


def _decoder_weights(state, cfg, bias=True, final=True):
    """The tensors of synth.decoder_weights, from the state's generator."""
    L, w, f, x = cfg["layers"], cfg["width"], cfg["ffn"], max(cfg["cross_heads"] * cfg["cross_head_width"], 1)
    out = {}
    for name in ("norm_self", "norm_cross", "norm_ff"):
        out[name + "_g"] = state.host((L, w), 0.1, 1.0)
        out[name + "_b"] = state.host((L, w), 0.02) if bias else None
    for name, shape in (("qkv", (L, 3 * w, w)), ("o_self", (L, w, w)), ("q_cross", (L, x, w)), ("o_cross", (L, w, x)), ("ffn_up", (L, f, w)),
                        ("ffn_down", (L, w, f)), ("position", (cfg["capacity"], w))):
        out[name] = state.host(shape, 0.02)
    out["norm_out_g"] = state.host((w,), 0.1, 1.0) if final else None
    out["norm_out_b"] = state.host((w,), 0.02) if final and bias else None
    return out


def _prepare_step(state, case):
    """One decode step of every stream and the output head on its rows, as the one call a serving loop makes per frame."""
    rows, memory = _numbers(case["rows"]), _numbers(case["memory"])
    cfg = synth.decoder_config(capacity=1024 if max(rows) < 1024 else MAX_KEYS)
    L, w = cfg["layers"], cfg["width"]
    state.backend.set_quant(STORAGE[case["storage"]])
    decoder = state.owns(pkg.Decoder(state.backend, cfg, _decoder_weights(state, cfg)))
    head = state.backend.keep(state.host((HEAD_ROWS, w), 0.02))
    hidden = torch.zeros((len(rows), w), device="cuda")
    logits, probs = (torch.zeros((len(rows), HEAD_ROWS), device="cuda") for _ in range(2))
    slots, keys, values, state.inputs = [], [], [], []
    for b, (n, m) in enumerate(zip(rows, memory)):
        k, v = (torch.zeros((L, cfg["capacity"], w), device="cuda") for _ in range(2))
        k[:, :n].normal_(generator=state.gen)
        v[:, :n].normal_(generator=state.gen)
        ck, cv, x = state.normal((L, m, w)), state.normal((L, m, w)), state.normal((w,))
        state.inputs.append((k, v, ck, cv, x))
        slots.append({"k": k.data_ptr(), "v": v.data_ptr(), "ck": ck.data_ptr(), "cv": cv.data_ptr(), "length": n, "memory_length": m,
                      "inp": x.data_ptr(), "out": hidden[b].data_ptr()})
        keys.append(k[:, n])        # the rows the step appends
        values.append(v[:, n])
    state.results = {"hidden": hidden, "logits": logits, "probs": probs, "keys": keys, "values": values}
    dlogits, dprobs = ([row.data_ptr() for row in t] for t in (logits, probs))
    state.call = lambda: decoder.step_head(slots, head, None, HEAD_ROWS, HEAD_VOCAB, dlogits, dprobs)


def _prepare_local(state, case):
    """The sixteen positions of one frame, tokens chosen on the device."""
    cfg = synth.decoder_config(layers=1, capacity=STREAMS + 1, cross_heads=0)
    w, batch = cfg["width"], case["batch"]
    state.backend.set_quant(STORAGE[case["storage"]])
    projections = [state.host((LOCAL_VOCAB, w), 0.05) for _ in range(STREAMS)]
    tables = [state.host((LOCAL_VOCAB, w)) for _ in range(STREAMS)]
    frame = state.owns(pkg.Local(state.backend, cfg, _decoder_weights(state, cfg, bias=False, final=False), projections, None, tables,
                                 LOCAL_VOCAB - 32, LOCAL_VOCAB - 31, STREAMS // 2))
    state.inputs = state.normal((batch, w))
    items = [{"row": state.inputs[b].data_ptr(), "temperature": case["temperature"], "topk": case["topk"],
              "rng_state": state.rng.getrandbits(63) | 1, "forbid_eos": True} for b in range(batch)]

    def call():
        out = frame.frame(items)
        out["rng_state"] = np.array(out["rng_state"], np.uint64).view(np.int64)
        return out

    state.call = call


def _prepare_prefill(state, case):
    cfg = synth.encoder_config()
    L, w, f, taps = cfg["layers"], cfg["width"], cfg["ffn"], case["taps"]
    cfg.update(causal=case["causal"], ffn_kernel=taps, operands_f32=case["operands"] == "f32")
    weights = {"tok_table": state.host((cfg["vocab"], w), 0.02), "pos_table": state.host((cfg["max_positions"], w), 0.02),
               "qkv": state.host((L, 3 * w, w), 0.02), "o": state.host((L, w, w), 0.02),
               "up": state.host((L, f, w * taps), 0.02), "down": state.host((L, w, f * taps), 0.02)}
    for name in ("norm1", "norm2"):
        weights[name + "_g"], weights[name + "_b"] = state.host((L, w), 0.1, 1.0), state.host((L, w), 0.02)
    weights["norm_out_g"], weights["norm_out_b"] = state.host((w,), 0.1, 1.0), state.host((w,), 0.02)
    encoder = state.owns(pkg.Encoder(state.backend, cfg, weights))
    ids = np.array([state.rng.randrange(cfg["vocab"]) for _ in range(case["tokens"])], np.int32)
    state.results = torch.zeros((case["tokens"], w), device="cuda")
    out = state.results.data_ptr()
    state.call = lambda: encoder.prefill(ids, 0, out)


def _prepare_cross_kv(state, case):
    cfg = synth.decoder_config()
    L, w, tokens, backend = cfg["layers"], cfg["width"], case["tokens"], state.backend
    backend.set_quant(pkg.F32)
    gains = [backend.keep(state.host((w,), 0.1, 1.0)) for _ in range(L)]
    weights = [backend.keep(state.host((2 * w, w), 0.02)) for _ in range(L)]
    state.inputs = memory = state.normal((tokens, w))
    k, v = (torch.zeros((L, tokens, w), device="cuda") for _ in range(2))
    state.results = {"k": k, "v": v}
    pointers = memory.data_ptr(), k.data_ptr(), v.data_ptr()
    state.call = lambda: backend.cross_kv_dev(pointers[0], tokens, w, gains, None, weights, w, pointers[1], pointers[2])


def _prepare_codec(state, case):
    """The codec's decode: pre-convolution, five stages of transposed convolution and residual layer, post-convolution, clip.  A
    residual layer's branches run side by side, as the benchmark's decode does."""
    frames, backend = case["frames"], state.backend

    def conv(out_ch, in_ch, k):
        return backend.keep(state.host((out_ch, in_ch, k), 1.0 / math.sqrt(in_ch * k))), backend.keep(state.host((out_ch,), 0.1))

    def alpha(channels):
        return backend.keep(np.abs(state.host((channels // 2,))) + np.float32(0.1))

    pre, channels, stages = conv(CODEC_CHANNELS, 32, 7), CODEC_CHANNELS, []
    for rate in RATES:
        half = channels // 2
        up = backend.keep(state.host((channels, 1, 2 * rate), 0.3)), backend.keep(state.host((half,), 0.1))
        blocks = [[(alpha(half), conv(half, half, k), alpha(half), conv(half, half, k), d) for d in DILATIONS] for k in KERNELS]
        stages.append((alpha(channels), up, blocks, rate))
        channels = half
    post_alpha, post = alpha(channels), conv(1, channels, 3)
    samples = frames * math.prod(RATES)
    most = max([CODEC_CHANNELS * frames] + [(CODEC_CHANNELS >> (i + 1)) * frames * math.prod(RATES[:i + 1]) for i in range(len(RATES))])
    latent = torch.empty(32 * frames, device="cuda").uniform_(-1, 1, generator=state.gen)
    space = torch.zeros((12, most), device="cuda")
    audio = torch.zeros(samples, device="cuda")
    state.inputs, state.results = (latent, space), audio
    first, second, up, *side = [space[i].data_ptr() for i in range(12)]
    latent_at, audio_at = latent.data_ptr(), audio.data_ptr()

    def call():
        c, n, cur, out = CODEC_CHANNELS, frames, first, second
        backend.conv1d_fused(latent_at, cur, 32, c, n, 7, 1, *pre, alpha=stages[0][0])
        for index, (_, up_conv, blocks, rate) in enumerate(stages):
            half, longer = c // 2, n * rate
            backend.conv_transpose_dev(cur, up, c, half, n, longer, 2 * rate, rate, half, *up_conv)
            codec.res_layer_batched(backend, blocks, up, out, half, longer, side[0:3], side[3:6], side[6:9],
                                    then_alpha=stages[index + 1][0] if index + 1 < len(stages) else post_alpha)
            cur, out, c, n = out, cur, half, longer
        backend.conv1d(cur, audio_at, c, 1, n, 3, 1, *post)
        backend.clip_dev(audio_at, n)

    state.call = call


_PREPARE = {"step": _prepare_step, "local": _prepare_local, "prefill": _prepare_prefill, "cross_kv": _prepare_cross_kv,
            "codec": _prepare_codec}


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    out = state.call()
    return state.results if out is None else out


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def work(case):
    """Weights, caches and inputs once, results once; two operations per multiply-add of the products and of attention."""
    kind = case["kind"]
    if kind == "step":
        rows, memory = _numbers(case["rows"]), _numbers(case["memory"])
        cfg = synth.decoder_config()
        L, w, f, batch = cfg["layers"], cfg["width"], cfg["ffn"], len(rows)
        moved = synth.decoder_step_bytes(cfg, STORAGE[case["storage"]], rows, memory)["total"]
        moved += synth.weight_bytes(HEAD_ROWS, w, STORAGE[case["storage"]]) + batch * 4 * (2 * w + 2 * HEAD_ROWS)
        flops = 2 * batch * (L * (6 * w * w + 2 * w * f) + HEAD_ROWS * w) + sum(4 * L * w * (n + 1 + m) for n, m in zip(rows, memory))
        return {"bytes": moved, "flops": flops}
    if kind == "local":
        cfg = synth.decoder_config(layers=1, cross_heads=0)
        w, f, storage, batch = cfg["width"], cfg["ffn"], STORAGE[case["storage"]], case["batch"]
        layer = sum(synth.weight_bytes(n, k, storage) for n, k in ((3 * w, w), (w, w), (f, w), (w, f)))
        moved = layer + STREAMS * (synth.weight_bytes(LOCAL_VOCAB, w, storage) + batch * 4 * w)
        flops = 2 * batch * STREAMS * (4 * w * w + 2 * w * f + LOCAL_VOCAB * w)
        return {"bytes": moved, "flops": flops}
    if kind == "prefill":
        cfg = synth.encoder_config()
        L, w, f, t, size = cfg["layers"], cfg["width"], cfg["ffn"], case["tokens"], 2 if case["operands"] == "f16" else 4
        weights = L * (4 * w * w + 2 * f * w * case["taps"])
        pairs = t * (t + 1) // 2 if case["causal"] else t * t
        return {"bytes": weights * size + 2 * t * w * size + 4 * t * w, "flops": 2 * t * weights + 4 * L * w * pairs}
    if kind == "cross_kv":
        cfg = synth.decoder_config()
        L, w, t = cfg["layers"], cfg["width"], case["tokens"]
        return {"bytes": 4 * (L * 2 * w * w + t * w + L * 2 * t * w), "flops": 2 * L * 2 * w * w * t}
    channels, n = CODEC_CHANNELS, case["frames"]
    params, flops = channels * 32 * 7, 2 * channels * 32 * 7 * n
    for rate in RATES:
        half, longer = channels // 2, n * rate
        branch = sum(2 * len(DILATIONS) * half * half * k for k in KERNELS)
        params += branch + channels * 2 * rate
        flops += 2 * branch * longer + 2 * half * 2 * 2 * longer
        channels, n = half, longer
    params, flops = params + channels * 3, flops + 2 * channels * 3 * n
    return {"bytes": 4 * (params + 32 * case["frames"] + n), "flops": flops}


def tolerance(case):
    """A quantised step rounds its activations to int8: one that a last-bit difference moves across a rounding boundary moves a row
    by up to some 1e-2.  Tokens follow from such rows through a draw.  The f16 prefill rounds every product's operands.  The codec is some
    forty 32-bit sums deep."""
    kind = case["kind"]
    if kind == "local":
        return {"rel": 0.0, "differ": 0.01}
    if kind == "step":
        return {"rel": 1e-2 if case["storage"] in ("int8", "int4") else 1e-5}
    if kind == "prefill":
        return {"rel": 2e-3 if case["operands"] == "f16" else 1e-5}
    return {"rel": 2e-5 if kind == "codec" else 1e-5}

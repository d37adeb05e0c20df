"""GPU parity of the codec operators (mynah_hip_conv1d / _conv_transpose_dev / _snake_dev) against the oracle, through the
C ABI.  conv1d runs in three-piece form on the bf16 matrix cores and adds in a different order than the CPU: 1e-5 normalised.  The transposed
conv adds in the reference's order: bit-exact.  snake: the device sine against libm's, 1e-6 normalised."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _announce(msg):
    print("[gpu-case] " + msg, flush=True)


def _run_conv1d(backend, x, w, b, dilation):
    in_ch, length = x.shape
    out_ch, _, kernel = w.shape
    din = backend.alloc(x.size).write(x)
    dout = backend.alloc(out_ch * length)
    backend.conv1d(din.ptr, dout.ptr, in_ch, out_ch, length, kernel, dilation, w, b)
    got = dout.read().reshape(out_ch, length)
    din.free()
    dout.free()
    return got


def test_known_answer(backend):
    """gpu/metal/backend_metal_ops.m:1026-1027,1099-1106: input 1 2 3, taps 1 2, no bias -> 2 5 8."""
    _announce("conv1d known answer")
    got = _run_conv1d(backend, np.array([[1, 2, 3]], np.float32), np.array([[[1, 2]]], np.float32), None, 1)
    assert got.tolist() == [[2.0, 5.0, 8.0]]


# (in, out, length, kernel, dilation): the codec's pre-conv, its residual convs at three stages (kernels 3/7/11, dilations
# 1/3/5), the post-conv, and shapes that end inside a tile or are shorter than a tap's reach
SHAPES = [(32, 864, 75, 7, 1), (432, 432, 600, 3, 1), (216, 216, 700, 7, 3), (108, 108, 1000, 11, 5), (54, 54, 3000, 11, 1),
          (27, 27, 5000, 7, 5), (27, 1, 9000, 3, 1), (5, 70, 33, 1, 1), (9, 33, 20, 11, 5), (8, 64, 128, 2, 1),
          (40, 48, 300, 16, 8), (64, 40, 257, 5, 2), (33, 65, 129, 4, 1), (128, 96, 64, 1, 1),
          # channels split over the wavefronts from 32 on: a few positions, the last row count that splits and the first that does not
          (32, 864, 1, 7, 1), (32, 32, 200, 7, 1), (31, 864, 40, 7, 1), (33, 300, 2432, 3, 1), (33, 300, 2433, 3, 1)]   # generic tap counts, the largest reach, odd edges


@pytest.mark.parametrize("shape", SHAPES)
def test_conv1d_against_oracle(backend, orc, nerr, shape):
    in_ch, out_ch, length, kernel, dilation = shape
    _announce("conv1d in=%d out=%d length=%d kernel=%d dilation=%d" % shape)
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((in_ch, length)).astype(np.float32)
    w = (rng.standard_normal((out_ch, in_ch, kernel)) / np.sqrt(in_ch * kernel)).astype(np.float32)
    b = rng.standard_normal(out_ch).astype(np.float32)
    got = _run_conv1d(backend, x, w, b, dilation)
    want = orc.conv1d_causal(x, w, b, dilation)
    assert nerr(got, want) < 1e-5
    got_nobias = _run_conv1d(backend, x, w, None, dilation)
    assert nerr(got_nobias, want - b[:, None]) < 1e-5


@pytest.mark.parametrize("shape", [(864, 432, 75, 8), (432, 216, 600, 8), (54, 27, 3000, 2), (8, 4, 5, 4), (12, 4, 7, 3)])
def test_conv_transpose_bit_exact(backend, orc, shape):
    in_ch, out_ch, length, stride = shape
    _announce("conv_transpose in=%d out=%d length=%d stride=%d" % shape)
    kernel = 2 * stride
    groups = out_ch if in_ch % out_ch == 0 and shape != (12, 4, 7, 3) else 2
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((in_ch, length)).astype(np.float32)
    w = rng.standard_normal((in_ch, out_ch // groups, kernel)).astype(np.float32)
    b = rng.standard_normal(out_ch).astype(np.float32)
    want = orc.conv_transpose_causal(x, w, b, stride, groups)
    din = backend.alloc(x.size).write(x)
    dout = backend.alloc(want.size)
    backend.conv_transpose_dev(din.ptr, dout.ptr, in_ch, out_ch, length, want.shape[1], kernel, stride, groups, w, b)
    got = dout.read().reshape(want.shape)
    assert np.array_equal(got, want)
    din.free()
    dout.free()


def test_snake(backend, orc, nerr):
    _announce("snake 432 x 600")
    rng = np.random.default_rng(9)
    x = (rng.standard_normal((432, 600)) * 2).astype(np.float32)
    alpha = (np.abs(rng.standard_normal(216)) + 0.05).astype(np.float32)
    d = backend.alloc(x.size).write(x)
    backend.snake_dev(d.ptr, alpha, 432, 600, 216)
    got = d.read().reshape(x.shape)
    want = orc.snake(x, alpha, 216)
    assert nerr(got[:216], want[:216]) < 1e-6
    assert np.array_equal(got[216:], want[216:])
    d.free()


def test_res_block_chain(backend, orc, nerr):
    """snake -> conv -> snake -> conv -> residual add, as res_layer_device chains them (src/graph.c:2444-2491)."""
    _announce("residual block chain 108 x 800")
    rng = np.random.default_rng(10)
    C, L, K, D = 108, 800, 7, 3
    x = rng.standard_normal((C, L)).astype(np.float32)
    a1, a2 = [(np.abs(rng.standard_normal(C // 2)) + 0.1).astype(np.float32) for _ in range(2)]
    w1, w2 = [(rng.standard_normal((C, C, K)) / np.sqrt(C * K)).astype(np.float32) for _ in range(2)]
    b1, b2 = [rng.standard_normal(C).astype(np.float32) * np.float32(0.1) for _ in range(2)]
    cur = backend.alloc(x.size).write(x)
    act, res, br = backend.alloc(x.size), backend.alloc(x.size), backend.alloc(x.size)
    backend.copy_dev(act.ptr, cur.ptr, x.size)
    backend.snake_dev(act.ptr, a1, C, L, C // 2)
    backend.conv1d(act.ptr, res.ptr, C, C, L, K, D, w1, b1)
    backend.snake_dev(res.ptr, a2, C, L, C // 2)
    backend.conv1d(res.ptr, br.ptr, C, C, L, K, 1, w2, b2)
    backend.residual_inplace(cur.ptr, br.ptr, x.size)
    got = cur.read().reshape(C, L)
    want = x + orc.conv1d_causal(orc.snake(orc.conv1d_causal(orc.snake(x, a1, C // 2), w1, b1, D), a2, C // 2), w2, b2, 1)
    assert nerr(got, want) < 1e-5
    for d in (cur, act, res, br):
        d.free()


def _res_layer_inputs(C, L, seed, taps=(3, 7, 11)):
    rng = np.random.default_rng(seed)
    alpha = lambda: (np.abs(rng.standard_normal(C // 2)) + 0.1).astype(np.float32)
    conv = lambda k: ((rng.standard_normal((C, C, k)) / np.sqrt(C * k)).astype(np.float32), rng.standard_normal(C).astype(np.float32) * np.float32(0.1))
    blocks = [[(alpha(), conv(k), alpha(), conv(k), d) for d in (1, 3, 5)] for k in taps]
    return rng.standard_normal((C, L)).astype(np.float32), blocks


# channels x length: the 64 x 128 tiles, the channel-split small tiles in both widths, at most 32 output channels, ragged edges
@pytest.mark.parametrize("C,L", [(108, 1000), (432, 96), (216, 300), (54, 700), (28, 1300), (70, 33)])
def test_fused_res_layer_is_the_operator_sequence(pkg, backend, orc, nerr, C, L):
    """The residual layer from fused calls (conv1d_fused, snake_copy_dev) against the same layer from the seam's operators
    in res_layer_device's order (src/graph.c:2423-2498): every value bit for bit.  And, for one shape, both against the oracle."""
    import importlib
    codec = importlib.import_module(pkg.__name__ + ".codec")
    _announce("fused residual layer %d x %d" % (C, L))
    x, blocks = _res_layer_inputs(C, L, 20 + C)
    n = C * L
    din = backend.alloc(n).write(x)
    bufs = [backend.alloc(n) for _ in range(8)]
    out_a, out_b = bufs[0], bufs[1]
    codec.res_layer(backend, blocks, din.ptr, out_a.ptr, C, L, *(b.ptr for b in bufs[2:6]))
    codec.res_layer_fused(backend, blocks, din.ptr, out_b.ptr, C, L, *(b.ptr for b in bufs[5:8]))
    seq, fused = out_a.read().reshape(C, L), out_b.read().reshape(C, L)
    assert np.isfinite(seq).all()
    assert np.array_equal(seq.view(np.uint32), fused.view(np.uint32))
    assert np.array_equal(din.read().reshape(C, L), x), "the layer's input was written"
    # the three branches' convolutions of a block and position in one launch each (conv1d_fused_batch): the same bits again
    more = [backend.alloc(n) for _ in range(10)]
    codec.res_layer_batched(backend, blocks, din.ptr, more[0].ptr, C, L, [b.ptr for b in more[1:4]], [b.ptr for b in more[4:7]],
                            [b.ptr for b in more[7:10]])
    batched = more[0].read().reshape(C, L)
    assert np.array_equal(seq.view(np.uint32), batched.view(np.uint32))
    assert np.array_equal(din.read().reshape(C, L), x), "the layer's input was written"
    for d in more:
        d.free()
    if C == 70:
        total = np.zeros_like(x)
        for branch in blocks:
            cur = x.copy()
            for a_in, (w_in, b_in), a_skip, (w_skip, b_skip), d in branch:
                cur = cur + orc.conv1d_causal(orc.snake(orc.conv1d_causal(orc.snake(cur, a_in, C // 2), w_in, b_in, d), a_skip, C // 2), w_skip, b_skip, 1)
            total += cur
        assert nerr(fused, total * np.float32(1.0 / 3.0)) < 1e-5
    for d in bufs + [din]:
        d.free()


# a block as one launch up to 32 channels, two launches for the short rows above: rows and channels one off a tile's
@pytest.mark.parametrize("C,L", [(16, 1), (27, 54), (32, 55), (33, 53), (64, 109), (65, 107), (108, 641), (128, 54), (128, 700), (27, 20000)])
def test_res_layer_call(pkg, backend, orc, nerr, C, L):
    """mynah_hip_res_layer_dev is the operator sequence bit for bit, whatever follows (a half-snake or none), and refuses work rows
    that are the layer's input or each other's."""
    import importlib
    codec = importlib.import_module(pkg.__name__ + ".codec")
    _announce("residual layer call %d x %d" % (C, L))
    x, blocks = _res_layer_inputs(C, L, 90 + C)
    blocks[1][1][0][0] = blocks[2][2][2][-1] = np.float32(9000.0)   # a half-snake's argument beyond the fast range of its sine
    then = np.full(C // 2, 0.7, np.float32)
    n = C * L
    din = backend.alloc(n).write(x)
    bufs = [backend.alloc(n) for _ in range(11)]
    at = [b.ptr for b in bufs]
    codec.res_layer(backend, blocks, din.ptr, at[0], C, L, *at[1:5])
    want = bufs[0].read()
    codec.res_layer_batched(backend, blocks, din.ptr, at[1], C, L, at[2:5], at[5:8], at[8:11])
    assert np.array_equal(want.view(np.uint32), bufs[1].read().view(np.uint32))
    assert np.array_equal(din.read().reshape(C, L), x), "the layer's input was written"
    backend.snake_dev(at[0], then, C, L, C // 2)
    want = bufs[0].read()
    codec.res_layer_batched(backend, blocks, din.ptr, at[1], C, L, at[2:5], at[5:8], at[8:11], then_alpha=then)
    assert np.array_equal(want.view(np.uint32), bufs[1].read().view(np.uint32))
    if n < 8000:
        total = np.zeros_like(x)
        for branch in blocks:
            cur = x.copy()
            for a_in, (w_in, b_in), a_skip, (w_skip, b_skip), d in branch:
                cur = cur + orc.conv1d_causal(orc.snake(orc.conv1d_causal(orc.snake(cur, a_in, C // 2), w_in, b_in, d), a_skip, C // 2), w_skip, b_skip, 1)
            total += cur
        assert nerr(bufs[1].read().reshape(C, L), orc.snake(total * np.float32(1.0 / 3.0), then, C // 2)) < 1e-5
    for work in ([din.ptr] + at[3:11], at[2:10] + [at[2]]):
        with pytest.raises(pkg.BackendError):
            codec.res_layer_batched(backend, blocks, din.ptr, at[1], C, L, work[0:3], work[3:6], work[6:9])
    for d in bufs + [din]:
        d.free()


# (branches by their taps) each build of the one-launch block and the edges between it and its neighbours, on 256 CUs: at most 32 channels
# narrow and wide; to 64 two launches / split order / narrow and wide in the large order; to 128 (fewer branches) split tiles / one launch
@pytest.mark.parametrize("C,L,taps", [(27, 20780, (3, 7, 11)), (27, 20786, (3, 7, 11)), (32, 30300, (3, 11)), (64, 3392, (3, 7, 11)), (64, 3393, (3, 7, 11)),
                                      (33, 4609, (3, 7, 11)), (50, 8193, (7,)), (50, 10300, (7,)), (54, 12160, (11, 3, 3, 7)), (54, 12161, (3, 7, 11)), (64, 20741, (3, 7, 11)),
                                      (54, 20800, (3, 7, 11)), (108, 6016, (11,)), (108, 6017, (11,)), (65, 6017, (3, 11)), (128, 6090, (7, 3)),
                                      (113, 13824, (11,)), (113, 13825, (11,)), (216, 3456, (3, 7)), (216, 3585, (3, 7))])
def test_res_layer_builds(pkg, backend, C, L, taps):
    """mynah_hip_res_layer_dev is the operator sequence bit for bit whichever way its blocks are launched."""
    import importlib
    codec = importlib.import_module(pkg.__name__ + ".codec")
    _announce("residual layer builds %d x %d taps %s" % (C, L, taps))
    x, blocks = _res_layer_inputs(C, L, 200 + C, taps)
    n, b = C * L, len(taps)
    din = backend.alloc(n).write(x)
    bufs = [backend.alloc(n) for _ in range(2 + max(4, 3 * b))]
    at = [d.ptr for d in bufs]
    codec.res_layer(backend, blocks, din.ptr, at[0], C, L, *at[2:6])
    codec.res_layer_batched(backend, blocks, din.ptr, at[1], C, L, at[2:2 + b], at[2 + b:2 + 2 * b], at[2 + 2 * b:2 + 3 * b])
    want, got = bufs[0].read(), bufs[1].read()
    assert np.isfinite(want).all()
    assert np.array_equal(want.view(np.uint32), got.view(np.uint32))
    for d in bufs + [din]:
        d.free()


# which of three positions leave the one launch, by a reach above 64 positions or by five taps in one branch
@pytest.mark.parametrize("leave", [(0,), (1,), (2,), (0, 1), (0, 2), (1, 2)])
@pytest.mark.parametrize("C,L,five", [(27, 700, False), (32, 130, True), (54, 3500, True)])
def test_res_layer_mixed_positions(pkg, backend, C, L, five, leave):
    """A layer some of whose positions are one launch and some two (the row sets change places between them): the operator sequence bit for bit."""
    import importlib
    codec = importlib.import_module(pkg.__name__ + ".codec")
    _announce("residual layer mixed positions %d x %d %s %s" % (C, L, leave, five))
    x, blocks = _res_layer_inputs(C, L, 400 + C)
    rng = np.random.default_rng(C)
    for p in leave:
        a_in, (w_in, b_in), a_skip, (w_skip, b_skip), d = blocks[0 if five else 2][p]
        if five:
            w_in, w_skip = ((rng.standard_normal((C, C, 5)) / np.sqrt(5 * C)).astype(np.float32) for _ in range(2))
        blocks[0 if five else 2][p] = (a_in, (w_in, b_in), a_skip, (w_skip, b_skip), d if five else 7)
    n = C * L
    din = backend.alloc(n).write(x)
    bufs = [backend.alloc(n) for _ in range(11)]
    at = [d.ptr for d in bufs]
    codec.res_layer(backend, blocks, din.ptr, at[0], C, L, *at[1:5])
    want = bufs[0].read()
    codec.res_layer_batched(backend, blocks, din.ptr, at[1], C, L, at[2:5], at[5:8], at[8:11])
    assert np.isfinite(want).all()
    assert np.array_equal(want.view(np.uint32), bufs[1].read().view(np.uint32))
    assert np.array_equal(din.read().reshape(C, L), x), "the layer's input was written"
    for d in bufs + [din]:
        d.free()


@pytest.mark.parametrize("C,L", [(27, 130), (108, 200), (216, 90)])
def test_res_layer_output_and_branch_forms(pkg, backend, C, L):
    """The layer's output may be its input or any of the work rows, in one launch a block or several; a single branch may grow in its
    input; blocks that the first branch does not have are not looked at, and a branch with fewer, or too few work rows, is an error."""
    import importlib
    codec = importlib.import_module(pkg.__name__ + ".codec")
    _announce("residual layer output forms %d x %d" % (C, L))
    x, blocks = _res_layer_inputs(C, L, 140 + C)
    n = C * L
    bufs = [backend.alloc(n) for _ in range(11)]
    at = [b.ptr for b in bufs]

    def layer(blocks, dout, work):
        bufs[0].write(x.ravel())
        codec.res_layer_batched(backend, blocks, at[0], dout, C, L, work[0:3], work[3:6], work[6:9])
        return next(b for b in bufs if b.ptr == dout).read().view(np.uint32)

    want = layer(blocks, at[1], at[2:11])
    for dout in (at[0], at[2], at[6], at[10]):
        assert np.array_equal(layer(blocks, dout, at[2:11]), want), at.index(dout)
    assert np.array_equal(layer([blocks[0], blocks[1] + blocks[2], blocks[2]], at[1], at[2:11]), want)
    with pytest.raises(IndexError):
        layer([blocks[0], blocks[1][:2], blocks[2]], at[1], at[2:11])
    with pytest.raises(ValueError):
        backend.res_layer_dev(blocks, at[0], at[1], C, L, at[2:10])
    one = layer(blocks[2:], at[1], at[2:11])
    assert np.array_equal(layer(blocks[2:], at[1], [at[0]] + at[3:11]), one)
    for d in bufs:
        d.free()


def test_conv_batch_members_and_refusals(pkg, backend):
    """conv1d_fused_batch, two to four members: with tap counts outside 3 / 7 / 11 (run one after the other) and with them
    (one launch) every member gets its own conv1d_fused result bit for bit; a member that writes what another reads is refused."""
    _announce("conv1d_fused_batch members")
    rng = np.random.default_rng(77)
    C, O, L = 40, 72, 210
    x = rng.standard_normal((4, C, L)).astype(np.float32)
    r = rng.standard_normal((O, L)).astype(np.float32)
    alpha = (np.abs(rng.standard_normal(O // 2)) + 0.1).astype(np.float32)
    dins = [backend.alloc(C * L).write(x[i]) for i in range(4)]
    dres = backend.alloc(O * L).write(r)
    for taps in ((3, 7, 11), (11, 11, 3), (5, 7, 11), (7, 3), (11, 3, 7, 11)):
        ws = [(rng.standard_normal((O, C, k)) / np.sqrt(C * k)).astype(np.float32) for k in taps]
        bs = [rng.standard_normal(O).astype(np.float32) for _ in taps]
        single = [backend.alloc(O * L) for _ in taps]
        together = [backend.alloc(O * L) for _ in taps]
        acts = [backend.alloc(O * L) for _ in range(2)]
        extras = [dict(residual=dres.ptr, scale=0.5), dict(alpha=alpha, activated=acts[0].ptr), dict(), dict(alpha=alpha)][:len(taps)]
        for i, k in enumerate(taps):
            e = dict(extras[i])
            if "activated" in e:
                e["activated"] = acts[1].ptr
            backend.conv1d_fused(dins[i].ptr, single[i].ptr, C, O, L, k, 1 + i, ws[i], bs[i], **e)
        backend.conv1d_fused_batch([dict(din=dins[i].ptr, dout=together[i].ptr, kernel=k, dilation=1 + i, weight=ws[i], bias=bs[i], **extras[i])
                                    for i, k in enumerate(taps)], C, O, L)
        for a, b in zip(single, together):
            assert np.array_equal(a.read().view(np.uint32), b.read().view(np.uint32)), taps
        assert np.array_equal(acts[0].read().view(np.uint32), acts[1].read().view(np.uint32)), taps
        with pytest.raises(pkg.BackendError, match="another member"):
            backend.conv1d_fused_batch([dict(din=dins[0].ptr, dout=together[0].ptr, kernel=taps[0], dilation=1, weight=ws[0]),
                                        dict(din=together[0].ptr, dout=together[1].ptr, kernel=taps[1], dilation=1, weight=ws[1])], C, O, L)
        for d in single + together + acts:
            d.free()
    with pytest.raises(pkg.BackendError, match="one to four"):
        backend.conv1d_fused_batch([], C, O, L)
    for d in dins + [dres]:
        d.free()


# channels shared between workgroups (more than 128, few short rows): one position, either side of the narrow and the wide tile, either side of
# each line between fewer workgroups (216 channels: 4 to 320 positions, 2 to 704, then one; 432: 7 to 64, 4 to 128, 3 to 192, 2 to 320), a last
# workgroup without a block of its own, any tap count; and two rows that one workgroup a tile takes
@pytest.mark.parametrize("C,O,L", [(432, 432, 1), (432, 400, 32), (432, 432, 33), (129, 70, 64), (216, 216, 320), (216, 216, 321), (216, 216, 704), (216, 216, 705),
                                   (432, 432, 129), (432, 432, 192), (432, 432, 193), (216, 216, 1408), (216, 216, 1409), (600, 30, 65), (144, 31, 130)])
def test_channels_shared_between_workgroups(backend, orc, nerr, C, O, L):
    """Against the oracle, single calls and members side by side (the same bits), with everything the epilogue can do."""
    _announce("shared channels %d -> %d x %d" % (C, O, L))
    rng = np.random.default_rng(C + O + L)
    x, r = rng.standard_normal((C, L)).astype(np.float32), rng.standard_normal((O, L)).astype(np.float32)
    alpha = (np.abs(rng.standard_normal(O // 2)) + 0.1).astype(np.float32)
    din, dres = backend.alloc(C * L).write(x), backend.alloc(O * L).write(r)
    taps = (3, 7, 11, 5)
    ws = [(rng.standard_normal((O, C, k)) / np.sqrt(C * k)).astype(np.float32) for k in taps]
    bs = [rng.standard_normal(O).astype(np.float32) for _ in taps]
    bufs = [backend.alloc(O * L) for _ in range(8)]
    extras = [dict(residual=dres.ptr, scale=0.5), dict(alpha=alpha, activated=bufs[7].ptr), dict(alpha=alpha), dict()]
    plain = [orc.conv1d_causal(x, w, b, 1 + 2 * i) for i, (w, b) in enumerate(zip(ws, bs))]
    want = [(plain[0] + r) * np.float32(0.5), plain[1], orc.snake(plain[2], alpha, O // 2), plain[3]]
    for i, k in enumerate(taps):
        backend.conv1d_fused(din.ptr, bufs[i].ptr, C, O, L, k, 1 + 2 * i, ws[i], bs[i], **extras[i])
        assert nerr(bufs[i].read().reshape(O, L), want[i]) < 1e-5, k
    assert nerr(bufs[7].read().reshape(O, L), orc.snake(plain[1], alpha, O // 2)) < 1e-5
    backend.conv1d_fused_batch([dict(din=din.ptr, dout=bufs[4 + i].ptr, kernel=taps[i], dilation=1 + 2 * i, weight=ws[i], bias=bs[i], **extras[i])
                                for i in range(3)], C, O, L)
    for a, b in zip(bufs[:3], bufs[4:7]):
        assert np.array_equal(a.read().view(np.uint32), b.read().view(np.uint32))
    for d in bufs + [din, dres]:
        d.free()


def test_conv_batch_on_the_wider_split_tiles(backend):
    """432 channels x 512 positions: alone a convolution takes the channel-split kernel's 32 x 32 tiles, three side by side
    its 32 x 64 tiles.  The tile's width is not part of a value's arithmetic: every member keeps its single call's bits."""
    _announce("conv1d_fused_batch on 432 x 512")
    rng = np.random.default_rng(78)
    C, L, taps = 432, 512, (3, 7, 11)
    x = rng.standard_normal((C, L)).astype(np.float32)
    din = backend.alloc(C * L).write(x)
    ws = [(rng.standard_normal((C, C, k)) / np.sqrt(C * k)).astype(np.float32) for k in taps]
    bs = [rng.standard_normal(C).astype(np.float32) for _ in taps]
    single = [backend.alloc(C * L) for _ in taps]
    together = [backend.alloc(C * L) for _ in taps]
    for i, k in enumerate(taps):
        backend.conv1d_fused(din.ptr, single[i].ptr, C, C, L, k, 1 + 2 * i, ws[i], bs[i], residual=din.ptr)
    backend.conv1d_fused_batch([dict(din=din.ptr, dout=together[i].ptr, kernel=k, dilation=1 + 2 * i, weight=ws[i], bias=bs[i], residual=din.ptr)
                                for i, k in enumerate(taps)], C, C, L)
    for a, b in zip(single, together):
        got = b.read()
        assert np.isfinite(got).all()
        assert np.array_equal(a.read().view(np.uint32), got.view(np.uint32))
    for d in single + together + [din]:
        d.free()


def test_rows_combine_is_the_operator_sequence(pkg, backend):
    """rows_combine_dev against residual_inplace per addend, scale_dev and snake_dev / snake_copy_dev: bit for bit."""
    _announce("rows_combine_dev")
    rng = np.random.default_rng(91)
    C, L = 54, 333
    rows = (rng.standard_normal((3, C, L)) * 3).astype(np.float32)
    alphas = [(np.abs(rng.standard_normal(C // 2)) + 0.1).astype(np.float32) for _ in range(3)]
    dins = [backend.alloc(C * L).write(rows[i]) for i in range(3)]
    outs = [backend.alloc(C * L) for _ in range(3)]
    want = backend.alloc(C * L)
    bits = lambda d: d.read().view(np.uint32)
    # one input, three activated outputs
    backend.rows_combine_dev([dins[0].ptr], 1.0, [o.ptr for o in outs], alphas, C, L)
    for o, al in zip(outs, alphas):
        backend.snake_copy_dev(dins[0].ptr, want.ptr, al, C, L, C // 2)
        assert np.array_equal(bits(o), bits(want))
    # three inputs summed in order, scaled, one output plain and one activated
    backend.rows_combine_dev([d.ptr for d in dins], 1.0 / 3.0, [outs[0].ptr, outs[1].ptr], [None, alphas[1]], C, L)
    backend.copy_dev(want.ptr, dins[0].ptr, C * L)
    backend.residual_inplace(want.ptr, dins[1].ptr, C * L)
    backend.residual_inplace(want.ptr, dins[2].ptr, C * L)
    backend.scale_dev(want.ptr, C * L, 1.0 / 3.0)
    assert np.array_equal(bits(outs[0]), bits(want))
    backend.snake_dev(want.ptr, alphas[1], C, L, C // 2)
    assert np.array_equal(bits(outs[1]), bits(want))
    # an output that is also the first input
    backend.rows_combine_dev([d.ptr for d in dins], 1.0 / 3.0, [dins[0].ptr], [alphas[1]], C, L)
    assert np.array_equal(bits(dins[0]), bits(want))
    with pytest.raises(pkg.BackendError, match="named twice"):
        backend.rows_combine_dev([dins[1].ptr], 1.0, [outs[0].ptr, outs[0].ptr], [None, None], C, L)
    with pytest.raises(pkg.BackendError, match="one to four"):
        backend.rows_combine_dev([], 1.0, [outs[0].ptr], [None], C, L)
    for d in dins + outs + [want]:
        d.free()


def test_fused_conv_pieces(backend, orc, nerr):
    """Each optional step of conv1d_fused alone against the operator it stands for, bit for bit."""
    _announce("conv1d_fused steps")
    rng = np.random.default_rng(31)
    C, O, L, K, D = 40, 72, 210, 7, 3
    x = rng.standard_normal((C, L)).astype(np.float32)
    w = (rng.standard_normal((O, C, K)) / np.sqrt(C * K)).astype(np.float32)
    b = rng.standard_normal(O).astype(np.float32)
    r1, r2 = rng.standard_normal((2, O, L)).astype(np.float32)
    alpha = (np.abs(rng.standard_normal(O // 2)) + 0.1).astype(np.float32)
    din, dr1, dr2 = backend.alloc(x.size).write(x), backend.alloc(r1.size).write(r1), backend.alloc(r2.size).write(r2)
    plain, got, act = backend.alloc(O * L), backend.alloc(O * L), backend.alloc(O * L)
    bits = lambda d: d.read().view(np.uint32)

    backend.conv1d(din.ptr, plain.ptr, C, O, L, K, D, w, b)
    backend.conv1d_fused(din.ptr, got.ptr, C, O, L, K, D, w, b)                       # nothing added: the plain operator
    assert np.array_equal(bits(got), bits(plain))

    backend.conv1d_fused(din.ptr, got.ptr, C, O, L, K, D, w, b, residual=dr1.ptr, residual2=dr2.ptr, scale=0.25)
    backend.residual_inplace(dr1.ptr, plain.ptr, O * L)                                # dr1 += conv
    backend.residual_inplace(dr2.ptr, dr1.ptr, O * L)                                  # dr2 += that
    backend.scale_dev(dr2.ptr, O * L, 0.25)
    assert np.array_equal(bits(got), bits(dr2))

    backend.conv1d_fused(din.ptr, got.ptr, C, O, L, K, D, w, b, alpha=alpha, snake_channels=O // 2, activated=act.ptr)
    assert np.array_equal(bits(got), bits(plain)), "the plain value must stay beside the activated one"
    backend.snake_dev(plain.ptr, alpha, O, L, O // 2)
    assert np.array_equal(bits(act), bits(plain))
    backend.conv1d_fused(din.ptr, got.ptr, C, O, L, K, D, w, b, alpha=alpha, snake_channels=O // 2)
    assert np.array_equal(bits(got), bits(plain))

    # sine arguments beyond the short routine's range take the epilogue's other path (and the library's sine in both kernels)
    big = (alpha * np.float32(3.0e4)).astype(np.float32)
    backend.conv1d(din.ptr, plain.ptr, C, O, L, K, D, w, b)
    backend.snake_dev(plain.ptr, big, O, L, O // 2)
    backend.conv1d_fused(din.ptr, got.ptr, C, O, L, K, D, w, b, alpha=big, snake_channels=O // 2)
    assert np.array_equal(bits(got), bits(plain))
    conv = _run_conv1d(backend, x, w, b, D)
    assert nerr(got.read().reshape(O, L), orc.snake(conv, big, O // 2)) < 1e-6

    backend.snake_copy_dev(din.ptr, got.ptr, alpha[:C // 2], C, L, C // 2)
    assert nerr(got.read(x.size).reshape(C, L), orc.snake(x, alpha[:C // 2], C // 2)) < 1e-6
    assert np.array_equal(din.read().reshape(C, L), x)
    for d in (din, dr1, dr2, plain, got, act):
        d.free()


def test_error_paths(pkg, backend):
    _announce("codec error paths")
    d = backend.alloc(64)
    w = np.zeros((1, 1, 17), np.float32)
    with pytest.raises(pkg.BackendError, match="kernel above 16 taps"):
        backend.conv1d(d.ptr, d.ptr, 1, 1, 8, 17, 1, w)
    with pytest.raises(pkg.BackendError, match="invalid conv1d arguments"):
        backend.conv1d(d.ptr, d.ptr, 1, 1, 0, 3, 1, w)
    with pytest.raises(pkg.BackendError, match="invalid conv_transpose arguments"):
        backend.conv_transpose_dev(d.ptr, d.ptr, 3, 2, 4, 8, 4, 2, 2, w)
    with pytest.raises(pkg.BackendError, match="invalid snake arguments"):
        backend.snake_dev(d.ptr, np.ones(4, np.float32), 2, 8, 3)
    e = backend.alloc(64)
    w3 = np.zeros((1, 1, 3), np.float32)
    with pytest.raises(pkg.BackendError, match="conv1d_fused"):      # the activated copy may not be the output itself
        backend.conv1d_fused(d.ptr, e.ptr, 1, 1, 8, 3, 1, w3, alpha=np.ones(1, np.float32), snake_channels=1, activated=e.ptr)
    with pytest.raises(pkg.BackendError, match="conv1d_fused"):      # more snake channels than output channels
        backend.conv1d_fused(d.ptr, e.ptr, 1, 1, 8, 3, 1, w3, alpha=np.ones(2, np.float32), snake_channels=2)
    e.free()
    d.free()


def _conv_multiply_adds(x, w, b, dilation):
    """The convolution as f32 multiply-adds (eight channels, the taps, the next eight), taps in front of the row left out."""
    out_ch, in_ch, kernel = w.shape
    length = x.shape[1]
    want = np.zeros((out_ch, length), np.float32) + b[:, None]
    for c0 in range(0, in_ch, 8):
        for k in range(kernel):
            back = min((kernel - 1 - k) * dilation, length)
            for c in range(c0, min(c0 + 8, in_ch)):
                want[:, back:] = want[:, back:].astype(np.float64) + w[:, c, k].astype(np.float64)[:, None] * x[c, :length - back].astype(np.float64)[None]
    return want


# large tiles (two shapes), channels split over the wavefronts, and over workgroups, each with straight-line taps and any
@pytest.mark.parametrize("C,O,L,K,D", [(20, 70, 300, 7, 3), (27, 27, 500, 11, 1), (27, 30, 90, 4, 2), (40, 48, 300, 3, 5), (33, 65, 129, 4, 1), (432, 100, 32, 3, 1),
                                       (150, 70, 70, 5, 2)])
def test_conv1d_extremes(backend, C, O, L, K, D):
    """Infinite, NaN and largest operands, in the rows and in the weights: what f32 multiply-adds give, and only in the outputs they enter.
    (An input channel that the last block of sixteen repeats, the first and the last position and output channel are among them.)"""
    _announce("conv1d extremes %d -> %d x %d, %d taps" % (C, O, L, K))
    rng = np.random.default_rng(C + L)
    x = rng.standard_normal((C, L)).astype(np.float32)
    w = (rng.standard_normal((O, C, K)) / np.sqrt(C * K)).astype(np.float32)
    b = rng.standard_normal(O).astype(np.float32)
    x[C - 1, 3], x[2, L // 2], x[0, L // 2 + 5], x[1, L - 1] = np.inf, -np.inf, np.nan, 3.4e38
    x[C - 1, 0], x[3, L // 3] = 3.4e38, -3.4028235e38
    w[4, 5, K - 1], w[5, C - 1, 0], w[O - 1, 7, K // 2], b[6] = np.inf, np.nan, 3.4e38, -np.inf
    with np.errstate(invalid="ignore", over="ignore"):
        want = _conv_multiply_adds(x, w, b, D).astype(np.float64)
        size = _conv_multiply_adds(np.abs(np.nan_to_num(x, posinf=0, neginf=0)), np.abs(np.nan_to_num(w, posinf=0)), np.abs(np.nan_to_num(b, neginf=0)), D).astype(np.float64)
    got = _run_conv1d(backend, x, w, b, D).astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    finite = np.isfinite(want)
    assert finite.mean() > 0.5 and (np.abs(want[finite]) > 1e36).any()
    assert (np.abs(got[finite] - want[finite]) <= 1e-5 * np.minimum(size[finite], 3.4e38)).all()
    # with an epilogue: the separate operators on the same values, the residual in place
    n = O * L
    r, alpha = rng.standard_normal((O, L)).astype(np.float32), (np.abs(rng.standard_normal(O // 2)) + 0.1).astype(np.float32)
    din, plain, fused, act = backend.alloc(x.size).write(x), backend.alloc(n), backend.alloc(n).write(r), backend.alloc(n)
    backend.conv1d(din.ptr, plain.ptr, C, O, L, K, D, w, b)
    dres = backend.alloc(n).write(r)
    backend.residual_inplace(dres.ptr, plain.ptr, n)
    backend.conv1d_fused(din.ptr, fused.ptr, C, O, L, K, D, w, b, residual=fused.ptr, alpha=alpha, snake_channels=O // 2, activated=act.ptr)
    assert np.array_equal(fused.read(), dres.read(), equal_nan=True)
    fused.write(r)
    backend.conv1d_fused(din.ptr, fused.ptr, C, O, L, K, D, w, b, residual=fused.ptr)
    assert np.array_equal(fused.read(), dres.read(), equal_nan=True)
    backend.snake_dev(dres.ptr, alpha, O, L, O // 2)
    assert np.array_equal(act.read(), dres.read(), equal_nan=True)
    for d in (din, plain, fused, act, dres):
        d.free()


# each build of the one-launch block, and a layer of two launches a position
@pytest.mark.parametrize("C,L,taps", [(27, 700, (3, 7, 11)), (27, 20786, (3, 7, 11)), (64, 3400, (3, 7, 11)), (54, 12161, (3, 7, 11)), (108, 6017, (11,)), (108, 500, (3, 7, 11))])
def test_res_layer_extremes(pkg, backend, C, L, taps):
    """Infinite, NaN and largest values in a layer's input, weights and (by a weight of one) in its inner rows, which the one-launch block
    keeps in three pieces alone: the operator sequence's values still."""
    import importlib
    codec = importlib.import_module(pkg.__name__ + ".codec")
    _announce("residual layer extremes %d x %d taps %s" % (C, L, taps))
    x, blocks = _res_layer_inputs(C, L, 300 + C, taps)
    leaky = C - 2                                            # a channel without a sine
    x[leaky, 40], x[1, 90], x[C - 1, 200], x[leaky, L - 1], x[leaky, 0] = 3.4e38, np.inf, np.nan, 3.4028235e38, -np.inf
    for branch in blocks:
        branch[0][1][0][leaky, leaky, :] = 1.0               # inner rows as large as the input's
    blocks[0][2][3][0][2, 3, 0], blocks[-1][2][3][0][C - 1, 0, 1] = 3.399e38, np.inf
    n, b = C * L, len(taps)
    din = backend.alloc(n).write(x)
    bufs = [backend.alloc(n) for _ in range(2 + max(4, 3 * b))]
    at = [d.ptr for d in bufs]
    for part in ([branch[:1] for branch in blocks], blocks):
        codec.res_layer(backend, part, din.ptr, at[0], C, L, *at[2:6])
        codec.res_layer_batched(backend, part, din.ptr, at[1], C, L, at[2:2 + b], at[2 + b:2 + 2 * b], at[2 + 2 * b:2 + 3 * b])
        want, got = bufs[0].read().reshape(C, L), bufs[1].read().reshape(C, L)
        assert np.array_equal(got, want, equal_nan=True)
        assert np.isfinite(want).any() and not np.isfinite(want).all()
    one = codec.res_layer(backend, [blocks[0][:1]], din.ptr, at[0], C, L, *at[2:6]) or bufs[0].read().reshape(C, L)
    assert np.isfinite(one[:, 40:60]).any() and np.abs(one[:, 40:60][np.isfinite(one[:, 40:60])]).max() > 1e36   # (the large values are values)
    for d in bufs + [din]:
        d.free()


# large tiles (two shapes), channels split over the wavefronts (both widths) and over workgroups, each with straight-line taps and any
UNEVEN = [(20, 70, 300, 7, 3), (27, 27, 900, 3, 1), (27, 30, 90, 4, 2), (40, 48, 300, 5, 5), (216, 216, 320, 11, 1), (432, 64, 33, 3, 1), (432, 100, 130, 7, 3)]


def _uneven_rows(rng, channels, length, sizes):
    """Rows in stretches of 1 to 40 positions, each of one of the sizes."""
    x = rng.uniform(-1, 1, size=(channels, length)).astype(np.float32)
    size, t = np.empty(length, np.float32), 0
    while t < length:
        n = int(rng.integers(1, 41))
        size[t:t + n] = rng.choice(sizes)
        t += n
    return x * size, size


@pytest.mark.parametrize("C,O,L,K,D", UNEVEN)
def test_conv1d_input_sizes(backend, C, O, L, K, D):
    """Positions from 2^-40 to 2^24 beside each other in a tile, output channels from 2^-60 to 2^60, and input channels of 2^-20 under weights that
    make up for it: f32's accuracy at every position."""
    _announce("conv1d input sizes %d -> %d x %d, %d taps" % (C, O, L, K))
    rng = np.random.default_rng(C + L)
    x, size = _uneven_rows(rng, C, L, np.exp2([-40, -30, -24, -20, -12, -9, 0, 15, 17, 24]).astype(np.float32))
    w = (rng.standard_normal((O, C, K)) / np.sqrt(C * K)).astype(np.float32)
    quiet = np.exp2(-20 * rng.integers(0, 2, size=(C, 1))).astype(np.float32)
    scale = np.exp2(rng.integers(-60, 60, size=(O, 1))).astype(np.float32)
    got = _run_conv1d(backend, x * quiet, w / quiet.reshape(1, C, 1) * scale[:, :, None], None, D).astype(np.float64) / scale
    want = np.zeros((O, L))
    for k in range(K):
        back = min((K - 1 - k) * D, L)
        want[:, back:] += w[:, :, k].astype(np.float64) @ x[:, :L - back].astype(np.float64)
    # operands in full; a term's products that are left out are 2^-26 of it in the mean, one of at most 900 additions in a row rounds 2^-25 of the running
    # sum in the mean, all of either sign: some 30 * 2^-25 of the result
    assert (np.linalg.norm(got - want, axis=0) <= 1e-6 * np.linalg.norm(want, axis=0)).all()


@pytest.mark.parametrize("C,O,L,K,D", UNEVEN)
def test_conv1d_neighbours_do_not_count(backend, C, O, L, K, D):
    """A position's bits follow from the inputs it reads alone, whatever else its tile reads (nothing, ordinary values, 2^24, f32's largest, an
    infinity, NaN), and a power of two in every input is one in every output."""
    _announce("conv1d neighbours %d -> %d x %d, %d taps" % (C, O, L, K))
    rng = np.random.default_rng(2 * C + L)
    x, _ = _uneven_rows(rng, C, L, np.exp2([-30, -20, -13]).astype(np.float32))
    w, b = (rng.standard_normal((O, C, K)) / np.sqrt(C * K)).astype(np.float32), np.zeros(O, np.float32)
    loud = rng.choice(L, size=max(1, L // 60), replace=False)
    free = np.ones(L, bool)
    for t in loud:
        for k in range(K):
            if t + k * D < L:
                free[t + k * D] = False
    assert free.any()
    want = _run_conv1d(backend, x, w, b, D)
    for value in (0.0, 2.0 ** -9, 1.0, 65521.0, 2.0 ** 24, 3.4028235e38, np.inf, np.nan):
        y = x.copy()
        y[rng.integers(0, C, size=loud.size), loud] = value
        assert np.array_equal(_run_conv1d(backend, y, w, b, D)[:, free].view(np.uint32), want[:, free].view(np.uint32)), value
    for power in (-30, -9, 13, 40):
        assert np.array_equal(_run_conv1d(backend, x * np.float32(2.0 ** power), w, b, D), want * np.float32(2.0 ** power)), power


# every way in which a position is launched (test_res_layer_builds): tiles of all widths, shared channels, each one-launch block
@pytest.mark.parametrize("C,L,taps", [(432, 40, (3, 7, 11)), (432, 300, (3, 7, 11)), (216, 320, (3, 7, 11)), (216, 1000, (3, 7)), (216, 4700, (3, 11)), (108, 1000, (3, 7, 11)),
                                      (108, 6300, (11,)), (27, 1300, (3, 7, 11)), (27, 42000, (3, 7)), (54, 2000, (3, 7, 11)), (54, 8000, (3, 7, 11)), (54, 13000, (3, 7, 11)),
                                      (64, 20700, (3, 7, 11))])
def test_res_layer_uneven_rows(pkg, backend, C, L, taps):
    """Rows with stretches and blocks of sixteen channels of 2^-24 to 2^17 beside each other and biases as small, so that tiles of every size
    meet values on both sides of any line: all forms of the layer still give the operator sequence's bits."""
    import importlib
    codec = importlib.import_module(pkg.__name__ + ".codec")
    _announce("residual layer uneven rows %d x %d taps %s" % (C, L, taps))
    x, blocks = _res_layer_inputs(C, L, 500 + C, taps)
    rng = np.random.default_rng(C + L)
    x, _ = _uneven_rows(rng, C, L, np.exp2([-24, -13, -12, -11, -9, 0, 17]).astype(np.float32))
    x *= np.repeat(np.exp2(-rng.integers(0, 14, size=(C + 15) // 16)), 16)[:C, None].astype(np.float32)
    for branch in blocks:
        for _, (_, b_in), _, (_, b_skip), _ in branch:
            b_in *= np.float32(1e-4)
            b_skip *= np.float32(1e-4)
    n, b = C * L, len(taps)
    din = backend.alloc(n).write(x)
    bufs = [backend.alloc(n) for _ in range(2 + max(4, 3 * b))]
    at = [d.ptr for d in bufs]
    codec.res_layer(backend, blocks, din.ptr, at[0], C, L, *at[2:6])
    want = bufs[0].read()
    assert np.isfinite(want).all()
    codec.res_layer_fused(backend, blocks, din.ptr, at[1], C, L, *at[2:5])
    assert np.array_equal(want.view(np.uint32), bufs[1].read().view(np.uint32))
    codec.res_layer_batched(backend, blocks, din.ptr, at[1], C, L, at[2:2 + b], at[2 + b:2 + 2 * b], at[2 + 2 * b:2 + 3 * b])
    assert np.array_equal(want.view(np.uint32), bufs[1].read().view(np.uint32))
    for d in bufs + [din]:
        d.free()


def test_conv_batch_members_uneven_rows(pkg, backend):
    """One call alone and two to four side by side, whose tiles differ in width: the same bits where the second half of a tile is the larger one."""
    _announce("conv1d_fused_batch members, uneven rows")
    rng = np.random.default_rng(78)
    for C, O, L in ((432, 432, 64), (432, 432, 256), (216, 216, 700), (40, 72, 210)):
        x, _ = _uneven_rows(rng, C, L, np.exp2([-13.0]).astype(np.float32))
        x[rng.integers(0, C, size=L // 32), np.arange(32, L + 32, 32)[:L // 32] % L] = 2.0 ** -9
        ws = [(rng.standard_normal((O, C, k)) / np.sqrt(C * k)).astype(np.float32) for k in (3, 7, 11, 3)]
        din, outs = backend.alloc(C * L).write(x), [backend.alloc(O * L) for _ in ws]
        alone = []
        for w in ws:
            backend.conv1d(din.ptr, outs[0].ptr, C, O, L, w.shape[2], 1, w, None)
            alone.append(outs[0].read().view(np.uint32))
        for members in (2, 3, 4):
            backend.conv1d_fused_batch([dict(din=din.ptr, dout=outs[i].ptr, kernel=ws[i].shape[2], dilation=1, weight=ws[i]) for i in range(members)], C, O, L)
            for i in range(members):
                assert np.array_equal(outs[i].read().view(np.uint32), alone[i]), (C, O, L, members, i)
        for d in [din] + outs:
            d.free()


@pytest.mark.parametrize("stride,kernel", [(2, 4), (4, 8), (8, 16), (2, 2), (2, 3), (4, 5), (8, 11), (4, 9), (8, 5), (3, 6), (1, 2)])
def test_conv_transpose_forms(backend, stride, kernel):
    """Strides and kernels on both sides of the vector form's rule, outputs that end before, at and behind the inputs' reach, rows at any
    alignment: bit for bit the sums in the reference's order (input channel, then input position), guard values around the output."""
    rng = np.random.default_rng(10 * stride + kernel)
    for in_ch, out_ch, groups in ((4, 2, 2), (3, 1, 1), (6, 4, 2)):
        for length in (1, 2, 37, 300):
            for output in sorted({1, max(1, length * stride - 1), length * stride, (length - 1) * stride + kernel, length * stride + stride + 1}):
                _announce("conv_transpose stride=%d kernel=%d %d -> %d in %d groups, %d -> %d" % (stride, kernel, in_ch, out_ch, groups, length, output))
                ipg, opg = in_ch // groups, out_ch // groups
                x = rng.standard_normal((in_ch, length)).astype(np.float32)
                w, b = rng.standard_normal((in_ch, opg, kernel)).astype(np.float32), rng.standard_normal(out_ch).astype(np.float32)
                want = np.zeros((out_ch, output), np.float32) + b[:, None]
                position = np.arange(output)
                for o in range(out_ch):
                    for i in range((o // opg) * ipg, (o // opg + 1) * ipg):
                        for back in range(-(-kernel // stride) - 1, -1, -1):         # earlier inputs first
                            t = position // stride - back
                            k = position - t * stride
                            ok = (t >= 0) & (t < length) & (k < kernel)
                            want[o, ok] = want[o, ok] + x[i, t[ok]] * w[i, o % opg, k[ok]]
                        reach = (position // stride > length - 1)                   # (behind the last input: counted from the last)
                        assert not (reach & (position - (length - 1) * stride < kernel) & (position // stride - (length - 1) >= -(-kernel // stride))).any()
                for lead in (0, 1):
                    din = backend.alloc(x.size).write(x)
                    dout = backend.alloc(out_ch * output + 3).write(np.full(out_ch * output + 3, 7.0, np.float32))
                    backend.conv_transpose_dev(din.ptr, dout.ptr + 4 * lead, in_ch, out_ch, length, output, kernel, stride, groups, w, b)
                    got = dout.read()
                    assert np.array_equal(got[lead:lead + want.size].reshape(want.shape), want)
                    assert (got[:lead] == 7.0).all() and (got[lead + want.size:] == 7.0).all()
                    din.free()
                    dout.free()


# (branches of 3, 7 and 11 taps, 256 CUs) the last and the first length of each one-launch build: at most 32 channels narrow / wide / narrow again; to 64
# two launches / one, the two orders, narrow / wide; more channels: split and large tiles
@pytest.mark.parametrize("C,L", [(27, 31152), (27, 31153), (27, 42558), (27, 42559), (40, 1), (50, 4096), (50, 4097), (50, 5440), (50, 5441), (54, 12160), (54, 12161), (54, 14790), (54, 14791), (64, 20768), (64, 20769),
                                 (33, 34510), (33, 34511), (216, 4608), (216, 4609)])
def test_res_layer_build_lines(pkg, backend, C, L):
    test_res_layer_builds(pkg, backend, C, L, (3, 7, 11))

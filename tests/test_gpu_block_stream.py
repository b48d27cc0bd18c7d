"""One token through Q8_0 / Q4_0 matrices as a row stream (block_stream.hip).

Outputs are held to a 64-bit product of the oracle's dequantized weights.  With S = sum |w| |x|, an
output passes at most 34 f32 roundings of partial sums of S: 16 of a block's chain, the two chains'
sum, the scale, a lane's two blocks, 6 of the lanes, 8 of the waves.  (Q4_0's q - 8 is exact.)
Over many rows such a rounding is at most 2^-24 / sqrt(3) of its sum's root mean square, which is no
larger than the result's, and 34 of them add to NORM (2-norm over the result's), which a sum less 8
times another (Q4_0 on the team kernels) passes: 2e-7 to 5e-7, through an FFN up to 9e-7.
"""
import numpy as np
import pytest

import hayai_amd
import oracle
from hayai_amd import synth

pytestmark = pytest.mark.gpu
Q4_0, Q8_0 = 2, 8
NORM = 34 ** 0.5 * 2.0 ** -24 / 3 ** 0.5  # 2.0e-7; measured 0.8e-7 to 1.2e-7


@pytest.fixture(scope="module")
def stream():
    import os
    os.environ["HAYAI_HIP_BLOCK_STREAM_MIN"] = "0"  # the smallest matrices too
    try:
        eng = hayai_amd.HipEngine(0)
    finally:
        del os.environ["HAYAI_HIP_BLOCK_STREAM_MIN"]
    yield eng
    eng.close()


# one row; fewer rows than workgroups; slices of one 8-block run, up to 64 blocks (two rows at a
# time, an odd last one), 65..128 blocks, several waves per row with a short or an empty last slice
@pytest.mark.parametrize("m,n", [(1, 256), (255, 512), (257, 768), (5000, 1024), (9000, 2048), (700, 2304),
                                 (513, 4096), (3000, 4352), (300, 8192), (260, 8448), (100, 14336), (40, 16640),
                                 (20, 25600), (1, 32), (3, 96), (300, 576), (1000, 1056), (515, 2080), (77, 4128),
                                 (33, 11008 + 32)])
@pytest.mark.parametrize("t", [Q4_0, Q8_0])
def test_gemv(stream, t, m, n):
    print(f"[case] block stream type={t} m={m} n={n}", flush=True)
    w = synth.matrix(t, m, n, synth.seed_for(71, m, n))
    x = synth.normal(synth.seed_for(72, m, n), n)
    y = stream.ggml_gemv_dispatch(t, m, n, w, x)
    W = oracle.dequant(t, w, m * n).reshape(m, n).astype(np.float64)
    ax = np.abs(x.astype(np.float64))
    err, exact = y - W @ x.astype(np.float64), W @ x.astype(np.float64)
    worst = float(np.max(np.abs(err) / (np.abs(W) @ ax * 34 * 2.0 ** -24)))
    norm = float(np.linalg.norm(err) / np.linalg.norm(exact))
    print(f"  worst error / bound {worst:.3e}, 2-norm {norm:.3e}", flush=True)
    assert np.isfinite(y).all() and worst <= 1.0 and (m < 64 or norm <= NORM)


@pytest.mark.parametrize("t,d_model,d_ff,act", [(Q8_0, 256, 768, 0), (Q4_0, 512, 2304, 1), (Q8_0, 2048, 5632, 0),
                                                (Q4_0, 4096, 4352, 0), (Q8_0, 8448, 256, 0), (Q4_0, 2080, 4128, 0),
                                                (Q8_0, 1056, 5664, 1)])
def test_ffn_and_block(stream, t, d_model, d_ff, act):
    print(f"[case] block stream ffn type={t} {d_model}x{d_ff} act={act}", flush=True)
    shapes = [(d_ff, d_model), (d_ff, d_model), (d_model, d_ff)]
    mats = [hayai_amd.QuantMatrix("m", c, r, t) for r, c in shapes]
    lay = hayai_amd.LayerPackLayout.ffn_only(*mats)
    ws = [synth.matrix(t, r, c, synth.seed_for(73, d_ff, i)) for i, (r, c) in enumerate(shapes)]
    pack = stream.alloc(lay.total)
    for w, off in zip(ws, (lay.gate_off, lay.up_off, lay.down_off)):
        pack.write(w, off)
    desc = stream.ffn_desc((t,) * 3, d_model, d_ff, lay, act)
    x = synth.normal(74, d_model)
    norm = (1 + 0.1 * synth.normal(75, d_model)).astype(np.float32)
    ref = oracle.ffn((t,) * 3, d_model, d_ff, *ws, x, act=act)
    y = stream.ffn(desc, pack, 0, x)
    print(f"  ffn {np.max(np.abs(y - ref)) / np.max(np.abs(ref)):.3e}", flush=True)
    # f32 sums on both sides: 1e-6 each at these widths
    assert np.max(np.abs(y - ref)) <= 1e-5 * np.max(np.abs(ref))
    # and against 64 bits the three products' errors, independent
    g, u, dn = (oracle.dequant(t, w, r * c).reshape(r, c).astype(np.float64) for w, (r, c) in zip(ws, shapes))
    gate = g @ x.astype(np.float64)
    f = 0.5 * gate * (1 + np.tanh(np.sqrt(2 / np.pi) * (gate + 0.044715 * gate ** 3))) if act else gate / (1 + np.exp(-gate))
    exact = dn @ (f * (u @ x.astype(np.float64)))
    err = float(np.linalg.norm(y - exact) / np.linalg.norm(exact))
    print(f"  ffn against 64 bits {err:.3e}", flush=True)
    assert err <= 3 ** 0.5 * NORM
    ref = oracle.ffn_block((t,) * 3, d_model, d_ff, *ws, norm, 1e-5, x, act=act)
    y = stream.ffn_block(desc, pack, 0, norm, 1e-5, x)
    assert np.max(np.abs(y - ref)) <= 1e-5 * np.max(np.abs(ref))
    # the block's two calls are its kernels
    xb, nb, yb = stream.upload(x), stream.upload(norm), stream.alloc(4 * d_model)
    stream.ffn_block_begin_dev(desc, pack, 0, nb, 0, 1e-5, xb, 0)
    stream.ffn_block_finish_dev(desc, pack, 0, xb, 0, yb, 0)
    if d_model > 2048 or d_ff > 2048:  # smaller layers: the one-launch FFN
        np.testing.assert_array_equal(yb.read(np.float32, d_model), y)


def test_ends_of_the_buffer(stream):
    # a matrix that ends with its buffer and starts at an odd multiple of 2: the last row's bytes
    # past the whole 16-byte pieces, and nothing past the end
    for t, bb in ((Q8_0, 34), (Q4_0, 18)):
        for m, n, at in ((5, 32, 0), (7, 96, 2), (300, 1056, 14), (260, 4128, 6)):
            w = synth.matrix(t, m, n, 78)
            x = synth.normal(79, n)
            buf = stream.alloc(at + w.nbytes)
            buf.write(w, at)
            xb, yb = stream.upload(x), stream.alloc(4 * m)
            stream.gemv_dev(t, m, n, buf, at, xb, 0, yb, 0)
            ref = oracle.gemv(t, m, n, w, x)
            assert np.max(np.abs(yb.read(np.float32, m) - ref)) <= 1e-5 * np.max(np.abs(ref)), (t, m, n, at)


def test_zero_scale_past_the_slice(stream):
    # lanes past a slice reread its last block with scale 0: an infinite d there stays in its row
    t, m, n = Q8_0, 6, 256
    w = synth.matrix(t, m, n, 76).reshape(m, -1).copy()
    w[3, -34:-32] = np.array([0x7C00], np.uint16).view(np.uint8)
    y = stream.ggml_gemv_dispatch(t, m, n, w, synth.normal(77, n))
    assert not np.isfinite(y[3]) and np.isfinite(np.delete(y, 3)).all()


@pytest.mark.parametrize("m,n", [(40, 256), (5, 4096), (40, 5632), (9, 14336)])
@pytest.mark.parametrize("t", [Q4_0, Q8_0])
def test_infinite_element_in_the_last_block(stream, t, m, n):
    # lanes past a slice hold its last block of x: an infinity there counts once, as in IEEE sums
    print(f"[case] block stream infinity type={t} m={m} n={n}", flush=True)
    w = synth.matrix(t, m, n, 80)
    x = synth.normal(81, n)
    x[n - 3] = -np.inf
    y = stream.ggml_gemv_dispatch(t, m, n, w, x)
    W = oracle.dequant(t, w, m * n).reshape(m, n).astype(np.float64)
    with np.errstate(invalid="ignore"):
        np.testing.assert_array_equal(y, (W * x.astype(np.float64)).sum(axis=1).astype(np.float32))


@pytest.mark.parametrize("t", [Q4_0, Q8_0])
def test_captured_blocks_replay(engine, t):
    # two residual blocks and a product on the row stream in one graph: every replay, with eager
    # calls between them, gives the eager bits
    d_model, d_ff = 2048, 5632
    shapes = [(d_ff, d_model), (d_ff, d_model), (d_model, d_ff)]
    lay = hayai_amd.LayerPackLayout.ffn_only(*[hayai_amd.QuantMatrix("m", c, r, t) for r, c in shapes])
    ws = [synth.matrix(t, r, c, synth.seed_for(82, t, i)) for i, (r, c) in enumerate(shapes)]
    pack = engine.alloc(lay.total)
    for w, off in zip(ws, (lay.gate_off, lay.up_off, lay.down_off)):
        pack.write(w, off)
    desc = engine.ffn_desc((t,) * 3, d_model, d_ff, lay)
    x, norm = engine.upload(synth.normal(83, d_model)), engine.upload(np.ones(d_model, np.float32))
    y, z = engine.alloc(4 * d_model), engine.alloc(4 * d_ff)

    def step():
        engine.ffn_block_dev(desc, pack, 0, norm, 0, 1e-5, x, 0, y, 0)
        engine.ffn_block_dev(desc, pack, 0, norm, 0, 1e-5, y, 0, y, 0)
        engine.gemv_dev(t, d_ff, d_model, pack, lay.gate_off, y, 0, z, 0)

    step()
    engine.sync()
    want = y.read(np.float32, d_model), z.read(np.float32, d_ff)
    g = engine.capture(step)
    for k in range(4):
        x.write(synth.normal(84 + k, d_model), 0)  # other inputs in the same buffer
        step()
        engine.sync()
        eager = y.read(np.float32, d_model), z.read(np.float32, d_ff)
        assert not np.array_equal(eager[0], want[0])
        y.write(np.zeros(d_model, np.float32), 0)
        g.launch()
        engine.sync()
        np.testing.assert_array_equal(y.read(np.float32, d_model), eager[0])
        np.testing.assert_array_equal(z.read(np.float32, d_ff), eager[1])
    g.free()

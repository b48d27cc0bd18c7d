"""Many tokens through one matrix on the matrix cores, every quantized format (mmg.hip).

Held to a 64-bit product of the oracle's dequantized weights.  Bound per output, with
S = sum |w| |x|: the two-f16 split of x leaves at most 2^-22 of each |x|, and every f32
addition of the matrix cores (n / 16 steps, hi and lo) and of the running sum (at most n / 32)
at most 2^-23 of S.
"""
import numpy as np
import pytest

import hayai_amd
import oracle
from hayai_amd import synth

pytestmark = pytest.mark.gpu
Q4_0, Q8_0, Q4_K, Q6_K, IQ2, IQ3 = 2, 8, 12, 14, 16, 18
FORMATS = [Q4_0, Q8_0, Q6_K, IQ2, IQ3]


def check(t, m, n, w, X, Y):
    W = oracle.dequant(t, w, m * n).reshape(m, n).astype(np.float64)
    X = X.astype(np.float64)
    bound = (np.abs(X) @ np.abs(W).T) * (2.0 ** -22 + (n / 8 + n / 32) * 2.0 ** -23) + 1e-300
    worst = float(np.max(np.abs(Y - X @ W.T) / bound))
    print(f"  worst error / bound {worst:.3e}", flush=True)
    assert np.isfinite(Y).all() and worst <= 1.0


# rows and tokens around the tiles (256 rows a workgroup, 64 a wave; 16, 32 and 64 tokens),
# columns of one block, odd block counts, a partial 128-column chunk, and split columns
SHAPES = [(1, 256, 4), (33, 256, 16), (255, 768, 17), (257, 512, 32), (300, 1280, 33), (64, 2048, 64),
          (1000, 256, 65), (512, 2304, 97), (100, 14336, 5)]


@pytest.mark.parametrize("m,n,batch", SHAPES)
@pytest.mark.parametrize("t", FORMATS)
def test_products(engine, t, m, n, batch):
    print(f"[case] many tokens type={t} m={m} n={n} batch={batch}", flush=True)
    w = synth.matrix(t, m, n, synth.seed_for(51, batch, t))
    X = synth.normal(synth.seed_for(51, n, m), batch * n).reshape(batch, n)
    Y = engine.ggml_gemv_batched(t, m, n, w, X, batch).reshape(batch, m)
    check(t, m, n, w, X, Y)


@pytest.mark.parametrize("n", [32, 96, 576, 1056])
@pytest.mark.parametrize("t", [Q4_0, Q8_0])
def test_short_blocks_end_inside_a_chunk(engine, t, n):
    print(f"[case] many tokens type={t} n={n}", flush=True)
    m, batch = 70, 21
    w = synth.matrix(t, m, n, 52)
    X = synth.normal(53, batch * n).reshape(batch, n)
    check(t, m, n, w, X, engine.ggml_gemv_batched(t, m, n, w, X, batch).reshape(batch, m))


@pytest.mark.parametrize("t", FORMATS)
def test_tokens_of_any_size(engine, t):
    # each token has its own power of two: tiny, huge, zero and mixed tokens do not disturb
    # one another, and an infinite one only itself
    print(f"[case] token sizes type={t}", flush=True)
    m, n = 96, 512
    w = synth.matrix(t, m, n, 54)
    X = synth.normal(55, 6 * n).reshape(6, n)
    X[0] *= np.float32(1e-30)
    X[1] *= np.float32(1e30)
    X[2] = 0
    X[3, ::2] *= np.float32(1e-6)
    X[4, 7] = np.inf
    Y = engine.ggml_gemv_batched(t, m, n, w, X, 6).reshape(6, m)
    fine = [0, 1, 2, 3, 5]
    check(t, m, n, w, X[fine], Y[fine])
    assert not np.isfinite(Y[4]).any()


@pytest.mark.parametrize("batch", [7, 24, 64])  # the three tilings
@pytest.mark.parametrize("t", FORMATS)
def test_infinities_and_nan(engine, t, batch):
    # as the sum of the products in IEEE arithmetic: an infinite element makes an output infinite, or
    # NaN where its weight is 0, whatever its token's finite elements are
    print(f"[case] infinities type={t} batch={batch}", flush=True)
    m, n = 96, 768
    w = synth.matrix(t, m, n, 56)
    X = synth.normal(57, batch * n).reshape(batch, n)
    X[1, n - 1] = np.inf
    X[2, 5] = -np.inf
    X[2, 300:] *= np.float32(1e9)  # finite, far above f16
    X[3, 40] = np.nan
    X[4, 9], X[4, 700] = np.inf, -np.inf
    Y = engine.ggml_gemv_batched(t, m, n, w, X, batch).reshape(batch, m)
    W = oracle.dequant(t, w, m * n).reshape(m, n).astype(np.float64)
    fine = [0, 5, 6]
    check(t, m, n, w, X[fine], Y[fine])
    with np.errstate(invalid="ignore"):
        for b in (1, 2, 3, 4):
            np.testing.assert_array_equal(Y[b], (W * X[b].astype(np.float64)).sum(axis=1).astype(np.float32), str(b))


def make_pack(engine, types, d_model, d_ff, cfg):
    shapes = [(d_ff, d_model), (d_ff, d_model), (d_model, d_ff)]
    mats = [hayai_amd.QuantMatrix("m", c, r, t) for t, (r, c) in zip(types, shapes)]
    lay = hayai_amd.LayerPackLayout.ffn_only(*mats)
    ws = [synth.matrix(t, r, c, synth.seed_for(cfg, 0, i)) for i, (t, (r, c)) in enumerate(zip(types, shapes))]
    pack = engine.alloc(lay.total)
    for w, off in zip(ws, (lay.gate_off, lay.up_off, lay.down_off)):
        pack.write(w, off)
    return lay, ws, pack


def rms(err):
    return float(np.sqrt(np.mean(err ** 2)))


@pytest.fixture(scope="module")
def team_kernels():
    import os
    os.environ["HAYAI_HIP_BLOCK_STREAM"] = "0"  # Q8_0 / Q4_0 too
    try:
        eng = hayai_amd.HipEngine(0)
    finally:
        del os.environ["HAYAI_HIP_BLOCK_STREAM"]
    yield eng
    eng.close()


# where the team kernels' one token at a time is f32 products summed in f32 (Q8_0, Q4_0; Q6_K and IQ
# in rows of an odd number of blocks): long and split columns, one workgroup's whole row, each tiling; and where it is
# 16-bit digits (the last three), which a lost lo operand, 2^-12 of x, would pass by ten times
@pytest.mark.parametrize("t,m,n,batch", [
    (Q8_0, 4160, 4096, 1000), (Q8_0, 2048, 8192, 24), (Q8_0, 2048, 4096, 8), (Q6_K, 2048, 3840, 24),
    (Q6_K, 2048, 768, 40), (IQ2, 2048, 3840, 12), (IQ2, 2048, 2304, 64), (IQ3, 2048, 3840, 24),
    (Q4_0, 2048, 4096, 24), (Q4_0, 2048, 8192, 8), (Q6_K, 2048, 4096, 64), (IQ2, 2048, 4096, 24), (IQ3, 2048, 2048, 9),
])
def test_as_accurate_as_one_token(engine, team_kernels, t, m, n, batch):
    print(f"[case] accuracy type={t} m={m} n={n} batch={batch}", flush=True)
    w = synth.matrix(t, m, n, 74)
    X = synth.normal(75, batch * n).reshape(batch, n)
    rows = w.reshape(m, -1)[:2048]
    Y = engine.ggml_gemv_batched(t, m, n, w, X, batch).reshape(batch, m)[:8, :2048]
    one = np.stack([team_kernels.ggml_gemv_dispatch(t, len(rows), n, rows.reshape(-1), x) for x in X[:8]])
    ref = X[:8].astype(np.float64) @ oracle.dequant(t, rows.reshape(-1), rows.shape[0] * n).reshape(-1, n).T.astype(np.float64)
    ours, theirs = rms(Y - ref), rms(one - ref)
    print(f"  batch {ours:.3e} one at a time {theirs:.3e}", flush=True)
    # 16384 outputs a side: the root mean squares of two equal errors are within 2 %
    assert ours <= 1.04 * theirs


@pytest.mark.parametrize("types,d_model,d_ff,batch", [((Q8_0,) * 3, 2048, 5632, 77), ((Q8_0,) * 3, 2048, 5632, 400),
                                                      ((IQ3,) * 3, 2304, 3328, 40), ((Q6_K,) * 3, 2304, 3328, 70)])
def test_ffn_as_accurate_as_one_token(engine, team_kernels, types, d_model, d_ff, batch):
    print(f"[case] ffn accuracy {types} {d_model}x{d_ff} batch={batch}", flush=True)
    lay, ws, pack = make_pack(engine, types, d_model, d_ff, 76)
    desc = engine.ffn_desc(types, d_model, d_ff, lay)
    X = synth.normal(77, batch * d_model).reshape(batch, d_model)
    Y = engine.ffn_batched(desc, pack, 0, X)[:8]
    _, _, own = make_pack(team_kernels, types, d_model, d_ff, 76)
    one = np.stack([team_kernels.ffn(desc, own, 0, x) for x in X[:8]])
    g, u, d = (oracle.dequant(t, w, r * c).reshape(r, c).astype(np.float64)
               for t, w, (r, c) in zip(types, ws, [(d_ff, d_model), (d_ff, d_model), (d_model, d_ff)]))
    x = X[:8].astype(np.float64)
    gate = x @ g.T
    ref = (gate / (1 + np.exp(-gate)) * (x @ u.T)) @ d.T
    ours, theirs = rms(Y - ref), rms(one - ref)
    print(f"  batch {ours:.3e} one at a time {theirs:.3e}", flush=True)
    # the sums lose what the one-token ones do, about 1e-7 a product; the 22 bits of x and of h add 4e-8
    # each, independently: sqrt(1 + 0.4 ** 2) = 1.08, and 2 % between samples as above
    assert ours <= 1.1 * theirs


@pytest.mark.parametrize("types,d_model,d_ff,batch,act", [
    ((Q4_0,) * 3, 576, 1536, 5, 0), ((Q8_0,) * 3, 96, 160, 40, 0), ((Q6_K,) * 3, 768, 1280, 33, 1),
    ((Q4_K, Q4_K, Q6_K), 512, 1536, 70, 0), ((IQ2,) * 3, 512, 768, 16, 0), ((IQ3, IQ3, Q8_0), 256, 512, 17, 0),
    ((Q4_K, Q4_K, Q6_K), 256, 512, 1029, 0),  # more than one pass, the last of five tokens
])
def test_ffn(engine, types, d_model, d_ff, batch, act):
    print(f"[case] many tokens ffn {types} {d_model}x{d_ff} batch={batch}", flush=True)
    lay, ws, pack = make_pack(engine, types, d_model, d_ff, 56)
    desc = engine.ffn_desc(types, d_model, d_ff, lay, act)
    X = synth.normal(57, batch * d_model).reshape(batch, d_model)
    Y = engine.ffn_batched(desc, pack, 0, X)
    for b in list(range(min(batch, 40))) + list(range(max(40, batch - 8), batch)):
        ref = oracle.ffn(types, d_model, d_ff, *ws, X[b], act=act)
        # the oracle sums in f32 itself; both are within 1e-5 of max |y| at these widths
        assert np.max(np.abs(Y[b] - ref)) <= 2e-5 * np.max(np.abs(ref)), b


@pytest.mark.parametrize("d_model,d_ff,batch", [(256, 256, 4), (512, 768, 17), (2304, 512, 16), (1280, 1792, 31),
                                                (4096, 256, 70)])
def test_q4_k_rows_through_lds(engine, d_model, d_ff, batch):
    # gate/up with one token tile: one superblock, a short and a long run of them, splits of
    # unequal length, 16- and 32-token tiles
    types = (Q4_K, Q4_K, Q8_0)
    print(f"[case] q4_k rows through lds {d_model}x{d_ff} batch={batch}", flush=True)
    lay, ws, pack = make_pack(engine, types, d_model, d_ff, 66)
    desc = engine.ffn_desc(types, d_model, d_ff, lay)
    X = synth.normal(67, batch * d_model).reshape(batch, d_model)
    Y = engine.ffn_batched(desc, pack, 0, X)
    for b in range(batch):
        ref = oracle.ffn(types, d_model, d_ff, *ws, X[b])
        # as test_ffn
        assert np.max(np.abs(Y[b] - ref)) <= 2e-5 * np.max(np.abs(ref)), b


def test_in_place_and_unaligned_activations(engine):
    # x read and y written at 4-byte offsets, and y over x
    t, d_model, d_ff, batch = Q8_0, 160, 96, 9
    lay, ws, pack = make_pack(engine, (t,) * 3, d_model, d_ff, 58)
    desc = engine.ffn_desc((t,) * 3, d_model, d_ff, lay)
    X = synth.normal(59, batch * d_model).reshape(batch, d_model)
    want = engine.ffn_batched(desc, pack, 0, X)
    buf = engine.alloc(4 + X.nbytes)
    buf.write(X, 4)
    engine.ffn_batched_dev(desc, pack, 0, buf, 4, batch, buf, 4)
    np.testing.assert_array_equal(buf.read(np.float32, X.size, 4).reshape(X.shape), want)


# ---- all-Q4_K batches past 64 tokens: one f16 per activation -----------------------------


@pytest.fixture(scope="module")
def f16_engine():
    import os
    os.environ["HAYAI_HIP_MMF_MIN"] = "65"  # small shapes too
    try:
        eng = hayai_amd.HipEngine(0)
    finally:
        del os.environ["HAYAI_HIP_MMF_MIN"]
    yield eng
    eng.close()


def parts(w, m, n):
    """Q4_K weights in 64 bits, and per weight the error that a product with |x| may have: over
    |d sc q| and |dmin m| apart (they cancel in w), f16 rounds x by at most 2^-11 of it, the
    minima's 16-bit factors and sums of 32 x by 2^-14; f32 additions and unit changes as above."""
    W = oracle.dequant(Q4_K, w, m * n).reshape(m, n).astype(np.float64)
    nomin = w.reshape(-1, 144).copy()
    nomin[:, 2:4] = 0
    A = oracle.dequant(Q4_K, nomin.reshape(-1), m * n).reshape(m, n).astype(np.float64)
    a, b = np.abs(A), np.abs(A - W)
    return W, a * 2.0 ** -11 + b * 2.0 ** -14 + (a + b) * (n / 8) * 2.0 ** -23


@pytest.mark.parametrize("m,n,batch", [(1, 256, 65), (300, 256, 128), (257, 768, 129), (512, 2304, 200),
                                       (40, 14336, 97), (256, 512, 1100)])
@pytest.mark.parametrize("blocks", ["plain", "zero d", "small d"])
def test_f16_products(f16_engine, m, n, batch, blocks):
    print(f"[case] f16 tokens m={m} n={n} batch={batch} {blocks}", flush=True)
    w = synth.matrix(Q4_K, m, n, 61).reshape(-1, 144).copy()
    some = np.random.default_rng(62).random(len(w)) < 0.4
    if blocks == "zero d":  # the accumulator's unit stays the one before (or 1)
        w[some, 0:2] = 0
    if blocks == "small d":  # units 2^-24 beside ordinary ones, the minima as they were
        w[some, 0:2] = [1, 0]
    w = w.reshape(-1)
    X = synth.normal(63, batch * n).reshape(batch, n)
    X[1] *= np.float32(1e20)
    X[2] = 0
    Y = f16_engine.ggml_gemv_batched_q4_k(m, n, w, X, batch).reshape(batch, m)
    W, wide = parts(w, m, n)
    X = X.astype(np.float64)
    bound = np.abs(X) @ wide.T + 1e-300
    worst = float(np.max(np.abs(Y - X @ W.T) / bound))
    print(f"  worst error / bound {worst:.3e}", flush=True)
    assert np.isfinite(Y).all() and worst <= 1.0


@pytest.mark.parametrize("d_model,d_ff,batch,act", [(256, 512, 65, 0), (512, 768, 130, 1), (768, 1280, 257, 0)])
def test_f16_ffn(f16_engine, d_model, d_ff, batch, act):
    print(f"[case] f16 tokens ffn {d_model}x{d_ff} batch={batch}", flush=True)
    lay, ws, pack = make_pack(f16_engine, (Q4_K,) * 3, d_model, d_ff, 64)
    desc = f16_engine.ffn_desc((Q4_K,) * 3, d_model, d_ff, lay, act)
    X = synth.normal(65, batch * d_model).reshape(batch, d_model)
    Y = f16_engine.ffn_batched(desc, pack, 0, X)
    # the products' bounds carried through: |act'| <= 1.13, h's own rounding is in the last
    (G, eg), (U, eu), (D, ed) = (parts(w, r, c) for w, (r, c) in
                                 zip(ws, [(d_ff, d_model), (d_ff, d_model), (d_model, d_ff)]))
    X = X.astype(np.float64)
    g, u, ax = X @ G.T, X @ U.T, np.abs(X)
    inner = np.sqrt(2 / np.pi) * (g + 0.044715 * g ** 3)
    f = 0.5 * g * (1 + np.tanh(inner)) if act else g / (1 + np.exp(-g))
    dg, du = ax @ eg.T, ax @ eu.T
    dh = 1.13 * dg * (np.abs(u) + du) + np.abs(f) * du
    bound = dh @ np.abs(D).T + (np.abs(f * u) + dh) @ ed.T
    worst = float(np.max(np.abs(Y - (f * u) @ D.T) / bound))
    print(f"  worst error / bound {worst:.3e}", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("m,n,batch", [(300, 512, 65), (257, 768, 66), (256, 2304, 80), (512, 512, 139)])
def test_f16_leaves_a_short_last_pass(f16_engine, m, n, batch):
    # the 1..16 tokens over a multiple of 64 are computed as in a batch of their own
    print(f"[case] f16 tokens, last pass m={m} n={n} batch={batch}", flush=True)
    at = batch // 64 * 64
    w = synth.matrix(Q4_K, m, n, 68)
    X = synth.normal(69, batch * n).reshape(batch, n)
    Y = f16_engine.ggml_gemv_batched_q4_k(m, n, w, X, batch).reshape(batch, m)
    last = f16_engine.ggml_gemv_batched_q4_k(m, n, w, X[at:], batch - at).reshape(-1, m)
    np.testing.assert_array_equal(Y[at:], last)
    lay, ws, pack = make_pack(f16_engine, (Q4_K,) * 3, n, 512, 70)
    desc = f16_engine.ffn_desc((Q4_K,) * 3, n, 512, lay)
    Y = f16_engine.ffn_batched(desc, pack, 0, X)
    np.testing.assert_array_equal(Y[at:], f16_engine.ffn_batched(desc, pack, 0, X[at:]))


def test_f16_starts_at_a_full_pass(f16_engine):
    # 81 tokens: the last pass has 17, which would be 8-bit ones, and is f16 with the others
    m, n, batch = 64, 512, 81
    w = synth.matrix(Q4_K, m, n, 71)
    X = synth.normal(72, batch * n).reshape(batch, n)
    Y = f16_engine.ggml_gemv_batched_q4_k(m, n, w, X, batch).reshape(batch, m)
    W, wide = parts(w, m, n)
    X = X.astype(np.float64)
    assert np.all(np.abs(Y - X @ W.T) <= np.abs(X) @ wide.T)

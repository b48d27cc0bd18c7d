"""What a user of this framework has it do, as measured cases.

The framework runs the feed-forward half of GGUF language models on one GPU, so its work is:
one token at a time through the FFN blocks of a resident model (decode), a prompt's tokens
through an FFN at once (prompt), a mixture-of-experts layer for one or many tokens (moe), and
the output projection (head).  Activations and weights stay on the device, as they do between
the calls of a decode loop, and every call goes through HipEngine's enqueue-only entry points.

Host-link work (the pinned-host streamer, the file reader) is bound by the link and not listed.
"""
import ctypes
import math
import os
import re

import numpy as np
import torch

import hayai_amd
from hayai_amd.engine import HipEngine, LayerPackLayout, QuantMatrix

# format: GGML type, columns and bytes per block, byte offset of the f16 scale, std of the
# uniform codes' weights in units of that scale (weights get a std of 1 / sqrt(columns), so
# activations keep their size through an FFN as they do in a trained model)
FORMATS = {
    "q4_0": (hayai_amd.Q4_0, 32, 18, 0, 4.64),
    "q8_0": (hayai_amd.Q8_0, 32, 34, 0, 73.9),
    "q4_k": (hayai_amd.Q4_K, 256, 144, 0, 258.0),
    "q6_k": (hayai_amd.Q6_K, 256, 210, 208, 1366.0),
    "iq2_xxs": (hayai_amd.IQ2_XXS, 256, 66, 0, 48.0),
    "iq3_xxs": (hayai_amd.IQ3_XXS, 256, 98, 0, 128.0),
}
# a layer's (gate, up, down) formats: the mixed Q4_K_M files keep down in Q6_K
LAYERS = {f: (f, f, f) for f in FORMATS}
LAYERS["q4_k_m"] = ("q4_k", "q4_k", "q6_k")

EPS = 1e-5


def listed():
    return [
        # the smallest call: one FFN of a 135M-parameter model, launch and latency bound
        {"name": "decode 135m q4_0", "kind": "ffn", "fmt": "q4_0", "d_model": 576, "d_ff": 1536, "layers": 1},
        # decode of the models people run: a token through resident FFN residual blocks
        {"name": "decode 8b q4_k", "kind": "block", "fmt": "q4_k", "d_model": 4096, "d_ff": 14336, "layers": 4},
        {"name": "decode 8b q4_k_m", "kind": "block", "fmt": "q4_k_m", "d_model": 4096, "d_ff": 14336, "layers": 3},
        {"name": "decode 8b q8_0", "kind": "block", "fmt": "q8_0", "d_model": 4096, "d_ff": 14336, "layers": 2},
        {"name": "decode 70b iq2_xxs", "kind": "block", "fmt": "iq2_xxs", "d_model": 8192, "d_ff": 28672, "layers": 2},
        # the output projection of a 128k-word vocabulary, one token
        {"name": "head q6_k", "kind": "head", "fmt": "q6_k", "m": 128256, "n": 4096, "tokens": 1},
        # a few sequences decoded together
        {"name": "prompt 8b q4_k 16", "kind": "prompt", "fmt": "q4_k", "d_model": 4096, "d_ff": 14336, "tokens": 16},
        # prompts: a whole chunk, and lengths that are no multiple of anything
        {"name": "prompt 8b q4_k 512", "kind": "prompt", "fmt": "q4_k", "d_model": 4096, "d_ff": 14336, "tokens": 512},
        {"name": "prompt 8b q4_k_m 203", "kind": "prompt", "fmt": "q4_k_m", "d_model": 4096, "d_ff": 14336,
         "tokens": 203},
        {"name": "prompt 1b q8_0 77", "kind": "prompt", "fmt": "q8_0", "d_model": 2048, "d_ff": 5632, "tokens": 77},
        # a mixture-of-experts layer (128 experts, 8 per token): a decode batch and a prompt
        {"name": "moe q4_k 32", "kind": "moe", "experts": 128, "top_k": 8, "d_model": 2048, "d_ff": 768, "tokens": 32},
        {"name": "moe q4_k 512", "kind": "moe", "experts": 128, "top_k": 8, "d_model": 2048, "d_ff": 768,
         "tokens": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["ffn", "block", "prompt", "prompt", "moe", "head"])
        fmt = rng.choice(sorted(LAYERS))
        if kind == "moe":
            case = {"kind": kind, "experts": rng.choice([16, 64, 128]), "top_k": rng.randint(2, 8),
                    "d_model": rng.choice([1024, 2048]), "d_ff": 256 * rng.randint(2, 6), "tokens": _log(rng, 1, 512)}
        elif kind == "head":
            fmt = rng.choice(sorted(FORMATS))
            b = FORMATS[fmt][1]
            case = {"kind": kind, "fmt": fmt, "m": _log(rng, 300, 128256), "n": b * _log(rng, 512 // b, 8192 // b),
                    "tokens": rng.choice([1, _log(rng, 2, 64)])}
        else:
            b = max(FORMATS[f][1] for f in LAYERS[fmt])
            d_model = b * _log(rng, 512 // b, 8192 // b)
            case = {"kind": kind, "fmt": fmt, "d_model": d_model,
                    "d_ff": b * max(1, int(d_model * rng.uniform(2.0, 3.6)) // b)}
            if kind == "prompt":
                case["tokens"] = _log(rng, 2, 512)
            else:
                case["layers"] = rng.randint(1, 4)
        w = work(case)
        # no dearer than the listed 8B prompt of 512 tokens or the listed decodes' weights
        if w["flops"] <= 180.4e9 and w["bytes"] <= 395e6:
            return case


def _row_bytes(fmt, n):
    _, block, size, _, _ = FORMATS[fmt]
    return n // block * size


def work(case):
    kind = case["kind"]
    if kind == "moe":
        # the experts that random routing reaches, each read once
        e, k, t = case["experts"], min(case["top_k"], case["experts"]), case["tokens"]
        reached = e * (1.0 - (1.0 - k / e) ** t)
        dm, df = case["d_model"], case["d_ff"]
        per = 2 * df * _row_bytes("q4_k", dm) + dm * _row_bytes("q4_k", df)
        return {"bytes": reached * per + 4.0 * t * (2 * dm + e), "flops": 2.0 * t * k * 3 * dm * df}
    if kind == "head":
        m, n, t = case["m"], case["n"], case["tokens"]
        return {"bytes": m * _row_bytes(case["fmt"], n) + 4.0 * t * (m + n), "flops": 2.0 * t * m * n}
    dm, df = case["d_model"], case["d_ff"]
    t, layers = case.get("tokens", 1), case.get("layers", 1)
    g, u, d = LAYERS[case["fmt"]]
    per = df * (_row_bytes(g, dm) + _row_bytes(u, dm)) + dm * _row_bytes(d, df)
    norm = 4 * dm if kind == "block" else 0
    return {"bytes": layers * (per + norm) + 8.0 * t * dm, "flops": 2.0 * t * layers * 3 * dm * df}


def tolerance(case):
    """About four times the largest distance from exact() that was measured over these ranges."""
    kind, fmt, tokens = case["kind"], case.get("fmt"), case.get("tokens", 1)
    if kind == "moe":
        return {"rel": 4e-4}  # activations of 16 bits in the integer kernels, 1e-4 measured
    if fmt == "q4_k" and kind == "prompt" and tokens >= 17:
        return {"rel": 0.03, "max": 0.4}  # 8-bit activations and intermediates: 1.2e-2, max 8e-2
    if fmt == "q4_k" and kind == "head" and tokens >= 17:
        return {"rel": 0.02, "max": 0.2}  # 8-bit activations: 5e-3
    if fmt == "q4_k" and kind == "prompt":
        return {"rel": 1e-3}  # an f16 intermediate: 2.6e-4
    chain = kind == "ffn" and case["layers"] > 1  # x -> FFN -> FFN: errors double at each product
    if fmt in ("q4_0", "q8_0"):
        return {"rel": 1.2e-4 if chain else 4e-6}  # 32-bit sums: 3e-5 through a chain, else 1e-6
    return {"rel": 9e-4 if chain else 3.2e-4}  # integer kernels again: 2.2e-4 and 8e-5


# ------------------------------------------------------------------------------- inputs


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _weights(fmt, rows, cols, g):
    """Random blocks of a format, [rows, row bytes]: uniform codes, scales spread threefold."""
    _, block, size, at, std = FORMATS[fmt]
    nb = cols // block
    w = torch.randint(0, 256, (rows * nb, size), dtype=torch.uint8, device="cuda", generator=g)
    d = (torch.rand(rows * nb, device="cuda", generator=g) + 0.5) / (std * math.sqrt(cols))
    w[:, at:at + 2] = d.half().view(torch.uint8).view(-1, 2)
    if fmt == "q4_k":  # minimums that centre the weights, as quantizing a trained matrix gives
        w[:, 2:4] = (7.5 * d).half().view(torch.uint8).view(-1, 2)
    return w.view(rows, nb * size)


def _inputs(case, seed):
    """The case's weights and activations as torch tensors on the GPU."""
    g = _generator(seed)
    kind = case["kind"]

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=g)

    if kind == "moe":
        dm, df, e = case["d_model"], case["d_ff"], case["experts"]
        return {"experts": [_weights("q4_k", e * df, dm, g), _weights("q4_k", e * df, dm, g),
                            _weights("q4_k", e * dm, df, g)],
                "logits": normal(case["tokens"], e), "x": normal(case["tokens"], dm)}
    if kind == "head":
        return {"w": _weights(case["fmt"], case["m"], case["n"], g), "x": normal(case["tokens"], case["n"])}
    dm, df = case["d_model"], case["d_ff"]
    fg, fu, fd = LAYERS[case["fmt"]]
    layers = []
    for _ in range(case.get("layers", 1)):
        layers.append((_weights(fg, df, dm, g), _weights(fu, df, dm, g), _weights(fd, dm, df, g),
                       torch.rand(dm, device="cuda", generator=g) + 0.5))
    return {"layers": layers, "x": normal(case.get("tokens", 1), dm)}


_engine = None


def _the_engine():
    global _engine
    if _engine is None:
        _engine = HipEngine(0)
    return _engine


class _Memory:
    """A device buffer's memory for torch (an hh_buf holds its engine, then its address)."""

    def __init__(self, buf, shape, typestr):
        address = ctypes.cast(buf.handle, ctypes.POINTER(ctypes.c_void_p))[1]
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (address, False),
                                         "version": 2, "strides": None}


def _tensor(buf, shape, typestr):
    return torch.as_tensor(_Memory(buf, shape, typestr), device="cuda")


def _buffer(engine, values):
    b = engine.alloc(values.numel() * values.element_size())
    _tensor(b, (b.nbytes,), "|u1").copy_(values.contiguous().view(-1).view(torch.uint8))
    return b


def _pack(engine, case, layer):
    """One layer's gate, up and down as a resident pack."""
    dm, df = case["d_model"], case["d_ff"]
    fg, fu, fd = LAYERS[case["fmt"]]
    lay = LayerPackLayout.ffn_only(QuantMatrix("ffn_gate", dm, df, FORMATS[fg][0]),
                                   QuantMatrix("ffn_up", dm, df, FORMATS[fu][0]),
                                   QuantMatrix("ffn_down", df, dm, FORMATS[fd][0]))
    pack = engine.alloc(lay.total)
    view = _tensor(pack, (pack.nbytes,), "|u1")
    for w, at in zip(layer[:3], (lay.gate_off, lay.up_off, lay.down_off)):
        view[at:at + w.numel()].copy_(w.view(-1))
    return pack, lay


def prepare(case, seed):
    engine, given, kind = _the_engine(), _inputs(case, seed), case["kind"]
    state = {"case": case, "engine": engine, "x": _buffer(engine, given["x"])}
    t = given["x"].shape[0]
    if kind == "moe":
        dm, df, e = case["d_model"], case["d_ff"], case["experts"]
        sizes = [w.numel() // e for w in given["experts"]]
        offs = [0, sizes[0], sizes[0] + sizes[1]]
        stride = (sum(sizes) + 255) // 256 * 256
        buf = engine.alloc(e * stride)
        view = _tensor(buf, (e, stride), "|u1")
        for w, at, n in zip(given["experts"], offs, sizes):
            view[:, at:at + n].copy_(w.view(e, n))
        state["experts"], state["logits"] = buf, _buffer(engine, given["logits"])
        state["desc"] = engine.moe_desc(dm, df, e, min(case["top_k"], e), stride, offs, norm_topk_prob=True)
        shape = (t, dm)
    elif kind == "head":
        state["w"] = _buffer(engine, given["w"])
        shape = (t, case["m"])
    else:
        dm, df = case["d_model"], case["d_ff"]
        packs = [_pack(engine, case, layer) for layer in given["layers"]]
        state["packs"] = [p for p, _ in packs]
        state["norms"] = [_buffer(engine, layer[3]) for layer in given["layers"]]
        types = [FORMATS[f][0] for f in LAYERS[case["fmt"]]]
        state["desc"] = engine.ffn_desc(types, dm, df, packs[0][1])
        shape = (t, dm)
    state["y"] = engine.alloc(4 * shape[0] * shape[1])
    if kind == "ffn":
        state["between"] = engine.alloc(state["y"].nbytes)  # odd layers' outputs in a chain
    state["out"] = _tensor(state["y"], shape, "<f4")
    state["out"].zero_()
    del given
    torch.cuda.synchronize()
    return state


def run(state):
    case, engine, x, y = state["case"], state["engine"], state["x"], state["y"]
    kind = case["kind"]
    if kind == "ffn":
        for i, pack in enumerate(state["packs"]):
            to = y if (len(state["packs"]) - i) % 2 else state["between"]
            engine.ffn_dev(state["desc"], pack, 0, x, 0, to, 0)
            x = to
    elif kind == "block":
        for pack, norm in zip(state["packs"], state["norms"]):
            engine.ffn_block_dev(state["desc"], pack, 0, norm, 0, EPS, x, 0, y, 0)
            x = y
    elif kind == "prompt":
        engine.ffn_batched_dev(state["desc"], state["packs"][0], 0, x, 0, case["tokens"], y, 0)
    elif kind == "moe":
        engine.moe_dev(state["desc"], state["experts"], 0, state["logits"], 0, None, 0, x, 0, case["tokens"], y, 0)
    elif case["tokens"] == 1:
        engine.gemv_dev(FORMATS[case["fmt"]][0], case["m"], case["n"], state["w"], 0, x, 0, y, 0)
    else:
        engine.gemv_batched_dev(FORMATS[case["fmt"]][0], case["m"], case["n"], state["w"], 0, x, 0, case["tokens"],
                                y, 0)
    return state["out"]


# ------------------------------------------------------------------- the same in 64 bits


def _codebooks():
    """The IQ formats' codebooks (data of the GGUF format) as the repository's header lists them."""
    here = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    with open(os.path.join(here, "hayai_amd", "csrc", "iq_grids.h")) as f:
        text = f.read()
    two = [int(v, 16) for v in re.findall(r"0x([0-9a-f]{16})ull", text)]
    three = [int(v, 16) for v in re.findall(r"0x([0-9a-f]{8})u\b", text)]
    grid2 = np.array(two, dtype="<u8").view(np.uint8).reshape(256, 8)
    grid3 = np.array(three, dtype="<u4").view(np.uint8).reshape(256, 4)
    return (torch.from_numpy(grid2.astype(np.float64)).cuda(), torch.from_numpy(grid3.astype(np.float64)).cuda())


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _signs(s):
    """[..., 8] of +-1: seven stored sign bits, the eighth makes their number even."""
    bits = torch.stack([(s >> i) & 1 for i in range(7)], -1)
    bits = torch.cat([bits, bits.sum(-1, keepdim=True) & 1], -1)
    return 1.0 - 2.0 * bits.double()


def _dequantized(fmt, w, cols):
    """[rows, row bytes] of a format -> [rows, cols] in 64 bits."""
    _, block, size, at, _ = FORMATS[fmt]
    rows = w.shape[0]
    b = w.reshape(-1, size)
    d = _f16(b[:, at:at + 2])
    if fmt == "q4_0":
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8
        v = d * q
    elif fmt == "q8_0":
        v = d * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "q4_k":
        s, qs = b[:, 4:16].int(), b[:, 16:].reshape(-1, 4, 32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        v = (d * sc).unsqueeze(2) * q - (_f16(b[:, 2:4]) * mn).unsqueeze(2)
    elif fmt == "q6_k":
        ql, qh = b[:, :128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        low = torch.stack([ql[:, :, :32] & 15, ql[:, :, 32:] & 15, ql[:, :, :32] >> 4, ql[:, :, 32:] >> 4], 2)
        high = torch.stack([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (low | (high << 4)).double() - 32
        v = (d * sc).unsqueeze(2) * q.reshape(-1, 16, 16)
    else:
        grids = _codebooks()
        if fmt == "iq2_xxs":
            groups = b[:, 2:].reshape(-1, 8, 8)
            index, aux = groups[:, :, :4].long(), groups[:, :, 4:].contiguous().view(torch.int32).squeeze(2).long()
            mags, step = grids[0][index], 0.25
        else:
            index = b[:, 2:66].reshape(-1, 8, 8).long()
            aux = b[:, 66:].reshape(-1, 8, 4).contiguous().view(torch.int32).squeeze(2).long()
            mags, step = grids[1][index].reshape(-1, 8, 4, 8), 0.5
        aux = aux & 0xFFFFFFFF
        sign = _signs(torch.stack([(aux >> (7 * i)) & 127 for i in range(4)], -1))
        scale = d.unsqueeze(1) * (0.5 + (aux >> 28).double().unsqueeze(2).unsqueeze(3)).squeeze(3) * step
        v = scale.unsqueeze(3) * mags * sign
    return v.reshape(rows, cols)


def _product(fmt, w, x):
    """x [tokens, cols] times the rows of w, in 64 bits, over slices of rows."""
    cols = x.shape[1]
    step = max(1, (1 << 26) // cols)
    return torch.cat([x @ _dequantized(fmt, w[r:r + step], cols).t().contiguous() for r in range(0, w.shape[0], step)], 1)


def _ffn(fmts, ws, x):
    gate, up = _product(fmts[0], ws[0], x), _product(fmts[1], ws[1], x)
    return _product(fmts[2], ws[2], gate / (1.0 + torch.exp(-gate)) * up)


def exact(case, seed):
    given, kind = _inputs(case, seed), case["kind"]
    x = given["x"].double()
    if kind == "head":
        return _product(case["fmt"], given["w"], x)
    if kind == "moe":
        e, k = case["experts"], min(case["top_k"], case["experts"])
        top, ids = torch.topk(torch.softmax(given["logits"].double(), 1), k, 1)
        share = top / top.sum(1, keepdim=True)
        parts = [w.reshape(e, -1, w.shape[1]) for w in given["experts"]]
        y = torch.zeros_like(x)
        for i in range(e):
            t, s = torch.nonzero(ids == i, as_tuple=True)
            if len(t):
                y.index_add_(0, t, share[t, s].unsqueeze(1) * _ffn(("q4_k",) * 3, [p[i] for p in parts], x[t]))
        return y
    for layer in given["layers"]:
        if kind == "block":
            n = x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * layer[3].double()
            x = x + _ffn(LAYERS[case["fmt"]], layer, n)
        else:
            x = _ffn(LAYERS[case["fmt"]], layer, x)
    return x

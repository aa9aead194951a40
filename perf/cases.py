"""What the engine is measured on: quantized products through `hk_amd.Engine`, and network passes
through `hk_amd.net.Net`, over the formats, sizes and token counts that they meet in use.

A case of kind "linear" is one product of a decoder's layer (or up to three that read one input):
`parts` matrices of `rows` x `cols` in format `fmt` on `n` tokens. Up to 8 tokens it is
`matvec_parts` on the f32 input (`matvec_parts_rmsnorm` with `norm`), as a decode step issues it;
longer inputs are quantized once (`prepare`) and multiplied (`mm`). With `silu` the matrix holds
interleaved gate and up rows and the output is silu(gate) * up. With `bias` each part has one.

A case of kind "net" is one pass of a decoder and its logits: `seqs` sequences with `new` tokens
each, after up to `ctx` tokens that are in the cache already (the i-th sequence holds
ctx * (i + 1) // seqs). `mixed` takes wv and w_down of every layer in Q6_K, the usual mix of a
4-bit file; the output matrix is Q6_K unless the network is Q8_0.

Weights are uniform quants under scales that vary by block, centred, with rows of about unit gain
(as trained weights after their norms); inputs are N(0, 1) with a few larger channels.
"""
import math

import numpy as np
import torch

from hk_amd import Engine, formats as F
from hk_amd.net import Config, Net, Options

INTEGER_DOT = ("q4_0", "q8_0", "q4_k", "q5_k", "q6_k", "iq4_nl", "iq4_xs")
FLOAT_DECODE = ("q2_k", "q3_k", "mxfp4")


def listed():
    small = dict(kind="net", dim=1024, heads=16, kv_heads=8, head_dim=128, ffn=3072, qk_norm=True)
    large = dict(kind="net", dim=4096, heads=32, kv_heads=8, head_dim=128, ffn=14336, qk_norm=False)

    def linear(name, fmt, rows, cols, n, parts=1, norm=False, silu=False, bias=False):
        return dict(name=name, kind="linear", fmt=fmt, rows=rows, cols=cols, n=n, parts=parts, norm=norm, silu=silu,
                    bias=bias)

    return [
        # The smallest call: a 0.6B model's q/k/v (equal parts here) on one token, norm included.
        linear("qkv_q8_0_1tok", "q8_0", 1024, 1024, 1, parts=3, norm=True, bias=True),
        # The largest single matrix of a decode step: an 8B model's output head.
        linear("head_q6_k_1tok", "q6_k", 128256, 4096, 1),
        # An FFN's first half of a file in a format that is decoded to floats, one token.
        linear("gate_up_q2_k_1tok", "q2_k", 14336, 4096, 1, parts=2),
        # The same place with sixteen sessions decoding together, in the most common 4-bit format.
        linear("gate_up_q4_k_16tok", "q4_k", 28672, 4096, 16, silu=True),
        # A short prompt of odd length through the long-K half of the FFN.
        linear("down_q6_k_100tok", "q6_k", 4096, 14336, 100),
        # A small model whose width is no multiple of a super-block, a prompt of odd length.
        linear("odd_q8_0_333tok", "q8_0", 4864, 896, 333, bias=True),
        # Prompt processing at its usual batch: the largest product of an 8B layer.
        linear("gate_up_q4_k_512tok", "q4_k", 28672, 4096, 512, silu=True),
        # The same size of prompt through a 3-bit file's FFN (decoded to floats).
        linear("up_q3_k_512tok", "q3_k", 14336, 4096, 512),
        # A whole 0.6B model, one token of a chat.
        dict(small, name="net_0p6b_q8_0_decode", layers=28, vocab=151936, fmt="q8_0", mixed=False, seqs=1, new=1, ctx=600),
        # An eighth of an 8B model (four layers and the head's share), one token of a long session ...
        dict(large, name="net_8b_q4_k_decode", layers=4, vocab=16384, fmt="q4_k", mixed=True, seqs=1, new=1, ctx=3000),
        # ... eight sessions of different lengths, one token each ...
        dict(large, name="net_8b_q4_k_sessions8", layers=4, vocab=16384, fmt="q4_k", mixed=True, seqs=8, new=1, ctx=2000),
        # ... and a prompt.
        dict(large, name="net_8b_q4_k_prompt", layers=4, vocab=16384, fmt="q4_k", mixed=True, seqs=1, new=1000, ctx=0),
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    if rng.random() < 0.65:
        fmt = rng.choice(INTEGER_DOT + FLOAT_DECODE)
        floats = fmt in FLOAT_DECODE
        rows = _log_int(rng, 256, 28672)
        n = _log_int(rng, 1, 640)
        cols = 256 * _log_int(rng, 2, 56)
        if fmt in ("q4_0", "q8_0", "iq4_nl") and rng.random() < 0.4:
            cols = 32 * rng.randrange(16, 160)
        # No more work than the largest listed products: 28672 x 4096 (14336 for the float-decode formats).
        rows = max(256, min(rows, (14336 if floats else 28672) * 4096 // cols))
        silu = rng.random() < 0.25
        if silu:
            rows += rows % 2
        norm = n <= 8 and not floats and cols % 256 == 0 and cols <= 4096 and rng.random() < 0.5
        return dict(kind="linear", fmt=fmt, rows=rows, cols=cols, n=n, parts=rng.choice((1, 2, 3)) if rows < 5000 else 1,
                    norm=norm, silu=silu, bias=not silu and rng.random() < 0.3)
    if rng.random() < 0.5:
        c = dict(kind="net", dim=1024, heads=16, kv_heads=8, head_dim=128, ffn=3072, qk_norm=True)
    else:
        c = dict(kind="net", dim=4096, heads=32, kv_heads=8, head_dim=128, ffn=14336, qk_norm=False)
    c.update(layers=rng.randrange(2, 5), vocab=16384, fmt=rng.choice(("q4_k", "q8_0", "q5_k")))
    c["mixed"] = c["fmt"] != "q8_0" and rng.random() < 0.5
    if rng.random() < 0.4:
        c.update(seqs=1, new=_log_int(rng, 9, 900), ctx=rng.choice((0, 0, 300)))
    else:
        c.update(seqs=_log_int(rng, 1, 12), new=1, ctx=_log_int(rng, 16, 4000))
    return c


# ---- weights: blocks in the file layout, and what they decode to in float64 --------------------

_IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
_FP4 = (0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12)
# Root mean square of a weight of the blocks below under a scale of one.
_UNIT = {"q8_0": 73.3, "q4_0": 4.64, "q4_k": 200.0, "q5_k": 402.0, "q6_k": 1540.0, "iq4_nl": 70.0, "iq4_xs": 1295.0,
         "q3_k": 42.5, "q2_k": 11.2, "mxfp4": 5.85}


def _blocks(fmt, rows, cols, std, g):
    """Random blocks [rows * blocks][bytes] (uint8, on the GPU) whose weights have about `std`."""
    elems, size = F.INFO[F.BY_NAME[fmt]]
    nb = rows * (cols // elems)

    def ints(lo, hi, *shape):  # lo..hi, both included
        return torch.randint(lo, hi + 1, shape, generator=g, device="cuda", dtype=torch.int32)

    def half(v):
        return v.half().view(torch.uint8).view(nb, 2)

    raw = torch.randint(0, 256, (nb, size), generator=g, device="cuda", dtype=torch.uint8)
    d = (0.5 + torch.rand(nb, generator=g, device="cuda")) * (std / _UNIT[fmt])
    if fmt == "q8_0":
        raw[:, 2:] = ints(-127, 127, nb, 32).to(torch.int8).view(torch.uint8)
        raw[:, 0:2] = half(d)
    elif fmt in ("q4_0", "iq4_nl", "iq4_xs"):
        raw[:, 0:2] = half(d)
    elif fmt in ("q4_k", "q5_k"):  # w = d sc q - dmin m, centred: m = sc, dmin = 7.5 d (15.5 d)
        sc = ints(20, 63, nb, 8)
        a, b = sc[:, :4], sc[:, 4:]
        raw[:, 0:2] = half(d)
        raw[:, 2:4] = half(d * (7.5 if fmt == "q4_k" else 15.5))
        raw[:, 4:8] = (a | (b >> 4 << 6)).to(torch.uint8)
        raw[:, 8:12] = (a | (b >> 4 << 6)).to(torch.uint8)
        raw[:, 12:16] = ((b & 15) | ((b & 15) << 4)).to(torch.uint8)
    elif fmt == "q6_k":
        sc = ints(30, 127, nb, 16) * (1 - 2 * ints(0, 1, nb, 16))
        raw[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
        raw[:, 208:210] = half(d)
    elif fmt == "q3_k":
        raw[:, 108:110] = half(d)
    elif fmt == "q2_k":
        sc = ints(4, 15, nb, 16)
        raw[:, 0:16] = (sc | (sc << 4)).to(torch.uint8)
        raw[:, 80:82] = half(d)
        raw[:, 82:84] = half(d * 1.5)
    elif fmt == "mxfp4":
        raw[:, 0] = (128 + round(math.log2(std / _UNIT[fmt])) + ints(-1, 0, nb)).to(torch.uint8)
    return raw


def _decode(fmt, raw, rows, cols):
    """float64 [rows][cols] of such blocks."""
    nb = raw.shape[0]
    b = raw.to(torch.int32)

    def half(at):
        return raw[:, at:at + 2].contiguous().view(torch.float16).double()  # [nb][1]

    def table(values, idx):
        return torch.tensor(values, dtype=torch.float64, device=raw.device)[idx]

    def scales_k():  # 8 scales and 8 mins of 6 bits
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1)
        return sc.double().unsqueeze(2), mn.double().unsqueeze(2)

    if fmt == "q8_0":
        w = raw[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif fmt == "q4_0":
        w = (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1) - 8).double() * half(0)
    elif fmt == "iq4_nl":
        w = table(_IQ4, torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1)) * half(0)
    elif fmt == "mxfp4":
        w = table(_FP4, torch.cat([b[:, 1:] & 15, b[:, 1:] >> 4], 1)) * torch.exp2(b[:, 0:1].double() - 128)
    elif fmt in ("q4_k", "q5_k"):
        sc, mn = scales_k()
        qs = b[:, 16 if fmt == "q4_k" else 48:].view(nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).view(nb, 8, 32)
        if fmt == "q5_k":
            q = q + 16 * (b[:, 16:48].unsqueeze(1) >> torch.arange(8, device=raw.device).view(1, 8, 1) & 1)
        w = half(0).unsqueeze(2) * sc * q - half(2).unsqueeze(2) * mn
    elif fmt == "q6_k":
        ql, qh = b[:, 0:128].view(nb, 2, 64), b[:, 128:192].view(nb, 2, 32)
        lo = torch.stack([ql[..., :32] & 15, ql[..., 32:] & 15, ql[..., :32] >> 4, ql[..., 32:] >> 4], 2)
        hi = torch.stack([qh >> s & 3 for s in (0, 2, 4, 6)], 2)
        q = ((lo | hi << 4) - 32).double().view(nb, 16, 16)
        sc = raw[:, 192:208].contiguous().view(torch.int8).double().unsqueeze(2)
        w = half(208).unsqueeze(2) * sc * q
    elif fmt == "iq4_xs":
        qs = b[:, 8:].view(nb, 8, 16)
        j = torch.arange(8, device=raw.device)
        low = (b[:, 4:8].unsqueeze(2) >> torch.tensor([0, 4], device=raw.device)).view(nb, 8) & 15
        high = (b[:, 2:3] | b[:, 3:4] << 8) >> (2 * j) & 3
        sc = ((low | high << 4) - 32).double().unsqueeze(2)
        w = half(0).unsqueeze(2) * sc * table(_IQ4, torch.cat([qs & 15, qs >> 4], 2))
    elif fmt == "q3_k":
        s = b[:, 96:108]
        low = torch.cat([s[:, 0:8] & 15, s[:, 0:8] >> 4], 1)
        high = torch.cat([s[:, 8:12] >> k & 3 for k in (0, 2, 4, 6)], 1)
        sc = ((low | high << 4) - 32).double().unsqueeze(2)
        qs, mask = b[:, 32:96].view(nb, 2, 1, 32), b[:, 0:32].view(nb, 1, 1, 32)
        it = torch.arange(4, device=raw.device).view(1, 1, 4, 1)
        bit = 4 * torch.arange(2, device=raw.device).view(1, 2, 1, 1) + it
        q = ((qs >> (2 * it) & 3) - 4 * (1 - (mask >> bit & 1))).double().view(nb, 16, 16)
        w = half(108).unsqueeze(2) * sc * q
    elif fmt == "q2_k":
        s = b[:, 0:16].unsqueeze(2)
        it = torch.arange(4, device=raw.device).view(1, 1, 4, 1)
        q = (b[:, 16:80].view(nb, 2, 1, 32) >> (2 * it) & 3).double().view(nb, 16, 16)
        w = half(80).unsqueeze(2) * (s & 15) * q - half(82).unsqueeze(2) * (s >> 4)
    return w.reshape(rows, cols)


def _quantized(fmt, x):
    """The 8-bit activations that a product with `fmt` is defined on, as float64 (d * q): per 32 values
    d = amax / 127, or per 256 the scale of the first value of the largest magnitude."""
    x = x.float()
    n, k = x.shape

    def away(v):  # round half away from zero
        return torch.sign(v) * torch.floor(v.abs() + 0.5)

    if F.ACT_KIND[F.BY_NAME[fmt]] == F.ACT_A8:
        v = x.view(n, k // 32, 32)
        d = (v.abs().amax(2, keepdim=True).double() / 127).float()
        inv = torch.where(d != 0, 1.0 / d.double(), 0.0).float()
        q = away((v * inv).double())
    else:
        v = x.view(n, k // 256, 256)
        at = v.abs().argmax(2, keepdim=True)
        top = v.gather(2, at).double()
        scale = torch.where(top != 0, -127.0 / top, 0.0).float()
        d = torch.where(scale != 0, 1.0 / scale.double(), 0.0).float()
        q = away((v * scale).double()).clamp(max=127)
    return (q * d.double()).view(n, k)


# ---- inputs -------------------------------------------------------------------------------------

_ENGINE = []


def _engine():
    if not _ENGINE:
        _ENGINE.append(Engine(0))
    return _ENGINE[0]


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFF)
    return g


def _linear_inputs(case, seed):
    g = _generator(seed)
    rows, cols, n = case["rows"], case["cols"], case["n"]
    raws = [_blocks(case["fmt"], rows, cols, cols ** -0.5, g) for _ in range(case["parts"])]
    x = torch.randn(n, cols, generator=g, device="cuda")
    x[:, torch.randint(0, cols, (max(1, cols // 500),), generator=g, device="cuda")] *= 8.0
    norm = 1.0 + 0.1 * torch.randn(cols, generator=g, device="cuda")
    biases = [0.3 * torch.randn(rows, generator=g, device="cuda") if case["bias"] else None for _ in raws]
    return raws, x, norm, biases


# In a trained network each half of a layer adds a fraction of the residual stream to it.
_GAIN = {"wo": 0.3, "w_down": 0.2}


def _formats(case):
    """The formats of a network's matrices."""
    fmt = case["fmt"]
    wide = "q6_k" if case["mixed"] else fmt
    t = {k: fmt for k in ("wq", "wk", "wo", "w_gate", "w_up")}
    t.update(wv=wide, w_down=wide, tok_embd=fmt, output="q8_0" if fmt == "q8_0" else "q6_k")
    return t


def _shapes(case):
    d, q, kv, f, v = case["dim"], case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["ffn"], case["vocab"]
    layer = {"wq": (q, d), "wk": (kv, d), "wv": (kv, d), "wo": (d, q), "w_gate": (f, d), "w_up": (f, d), "w_down": (d, f)}
    return layer, {"tok_embd": (v, d), "output": (v, d)}


def _net_inputs(case, seed):
    """(layers, io) as dicts of (format, blocks) and float32 vectors, and the sequences' tokens."""
    g = _generator(seed)
    fmts, (layer_shapes, io_shapes) = _formats(case), _shapes(case)
    d, hd = case["dim"], case["head_dim"]

    def vec(n):
        return 1.0 + 0.1 * torch.randn(n, generator=g, device="cuda")

    def mats(shapes):
        return {k: (fmts[k], _blocks(fmts[k], r, c, 1.0 if k == "tok_embd" else _GAIN.get(k, 1.0) * c ** -0.5, g), r, c)
                for k, (r, c) in shapes.items()}

    layers = []
    for _ in range(case["layers"]):
        m = mats(layer_shapes)
        m.update(attn_norm=vec(d), ffn_norm=vec(d))
        if case["qk_norm"]:
            m.update(q_norm=vec(hd), k_norm=vec(hd))
        layers.append(m)
    io = mats(io_shapes)
    io["out_norm"] = vec(d)
    lens = [case["ctx"] * (i + 1) // case["seqs"] for i in range(case["seqs"])]
    tokens = [torch.randint(0, case["vocab"], (n + case["new"],), generator=g, device="cuda").cpu().numpy().astype(np.uint32)
              for n in lens]
    return layers, io, lens, tokens


def _config(case):
    return Config(dim=case["dim"], n_layers=case["layers"], n_heads=case["heads"], n_kv_heads=case["kv_heads"],
                  head_dim=case["head_dim"], ffn_dim=case["ffn"], vocab=case["vocab"], max_ctx=case["ctx"] + case["new"] + 8,
                  rope_neox=case["qk_norm"], rope_base=1e6 if case["qk_norm"] else 5e5,
                  rms_eps=1e-6 if case["qk_norm"] else 1e-5)


class _Linear:
    """The matrices a program has uploaded, its input and its output buffers."""

    def __init__(self, case, seed):
        eng = _engine()
        raws, self.x, norm, self.biases = _linear_inputs(case, seed)
        torch.cuda.synchronize()
        t, n = F.BY_NAME[case["fmt"]], case["n"]
        self.mats = [eng.upload(r, t, case["rows"], case["cols"]) for r in raws]
        self.mode = 2 if case["silu"] else 0
        self.n, self.cols = n, case["cols"]
        self.norm = norm if case["norm"] else None
        if not case["bias"]:
            self.biases = None
        width = case["rows"] // 2 if case["silu"] else case["rows"]
        self.ys = [torch.zeros(n, width, device="cuda") for _ in raws]
        self.xq = torch.zeros(eng.act_bytes(n, case["cols"]), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()

    def run(self):
        eng, n = _engine(), self.n
        if self.norm is not None:
            eng.matvec_parts_rmsnorm(self.mats, self.ys, n, self.x, self.norm, 1e-6, biases=self.biases, mode=self.mode)
        elif n <= 8:
            eng.matvec_parts(self.mats, self.ys, n, x=self.x, biases=self.biases, mode=self.mode)
        else:
            eng.prepare(self.x, n, self.cols, self.mats, self.xq)
            for i, (m, y) in enumerate(zip(self.mats, self.ys)):
                eng.mm(m, self.xq, y, n, bias=None if self.biases is None else self.biases[i], mode=self.mode)
        return self.ys

    def __del__(self):
        torch.cuda.synchronize()
        for m in self.mats:
            _engine().free(m)


class _Network:
    """A loaded network whose sequences' earlier tokens are in its cache."""

    def __init__(self, case, seed):
        layers, io, lens, tokens = _net_inputs(case, seed)
        cfg = _config(case)

        def host(v):
            if isinstance(v, tuple):
                return v[1].view(v[2], -1).cpu().numpy(), F.BY_NAME[v[0]]
            return v.cpu().numpy()

        self.net = Net(_engine(), cfg, Options(slots=case["seqs"]))
        for i, layer in enumerate(layers):
            self.net.load_layer(i, {k: host(v) for k, v in layer.items()})
        self.net.load_io(host(io["tok_embd"]), host(io["out_norm"]), host(io["output"]))
        for s, (n, toks) in enumerate(zip(lens, tokens)):
            for at in range(0, n, 512):
                self.net.forward_items([(s, int(toks[p]), p) for p in range(at, min(n, at + 512))])
        self.new = [t[n:] for n, t in zip(lens, tokens)]
        self.lens, self.single = lens, case["seqs"] == 1
        self.items = [(s, int(t), n + j) for s, (n, toks) in enumerate(zip(lens, self.new)) for j, t in enumerate(toks)]
        self.last = [(s + 1) * case["new"] - 1 for s in range(case["seqs"])]

    def run(self):
        if self.single:
            self.net.forward(self.new[0], self.lens[0])
            return self.net.logits()
        self.net.forward_items(self.items)
        return self.net.logits_rows(self.last)

    def __del__(self):
        if hasattr(self, "net"):
            self.net.close()


def prepare(case, seed):
    return (_Linear if case["kind"] == "linear" else _Network)(case, seed)


def run(state):
    return state.run()


# ---- what a pass cannot do without ---------------------------------------------------------------

def work(case):
    if case["kind"] == "linear":
        rows, cols, n, parts = case["rows"], case["cols"], case["n"], case["parts"]
        out = rows // 2 if case["silu"] else rows
        return {"bytes": parts * F.matrix_bytes(F.BY_NAME[case["fmt"]], rows, cols) + 4 * n * cols + 4 * n * parts * out,
                "flops": 2 * parts * rows * cols * n}
    fmts, (layer, io) = _formats(case), _shapes(case)
    L, seqs, new = case["layers"], case["seqs"], case["new"]
    n = seqs * new
    size = {k: F.matrix_bytes(F.BY_NAME[fmts[k]], r, c) for k, (r, c) in {**layer, **io}.items()}
    lens = [case["ctx"] * (i + 1) // seqs for i in range(seqs)]
    kv = 2 * 2 * case["kv_heads"] * case["head_dim"]  # bytes of one position's key and value
    seen = sum((m + 1 + m + new) * new // 2 for m in lens)  # (token, position) pairs
    return {"bytes": L * (sum(size[k] for k in layer) + kv * sum(m + new for m in lens)) + size["output"] +
            n * size["tok_embd"] // case["vocab"] + 4 * seqs * case["vocab"],
            "flops": L * (2 * n * sum(r * c for r, c in layer.values()) + 4 * case["heads"] * case["head_dim"] * seen) +
            2 * seqs * case["vocab"] * case["dim"]}


def tolerance(case):
    if case["kind"] == "linear":
        # 32-bit sums of exact integer (or 32-bit) products. With the norm inside, its own rounding moves
        # a few activations across an 8-bit step.
        return {"rel": 2e-3, "max": 2e-2} if case["norm"] else {"rel": 1e-5, "max": 1e-4}
    # Keys, values and probabilities in 16 bits, and 8-bit activations that a rounding before them moves
    # by a step, through every layer (about 1 % of the logits).
    return {"rel": 3e-2, "max": 0.3}


# ---- the same in float64 -------------------------------------------------------------------------

def _silu(v):
    return v / (1.0 + torch.exp(-v))


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + eps) * w.double()


def _exact_linear(case, seed):
    raws, x, norm, biases = _linear_inputs(case, seed)
    x = x.double()
    if case["norm"]:
        x = _rms(x, norm, 1e-6)
    x = _quantized(case["fmt"], x)
    out = []
    for raw, b in zip(raws, biases):
        y = x @ _decode(case["fmt"], raw, case["rows"], case["cols"]).T
        if case["silu"]:
            y = _silu(y[:, 0::2]) * y[:, 1::2]
        out.append(y if b is None else y + b.double())
    return out


def _exact_net(case, seed):
    layers, io, lens, tokens = _net_inputs(case, seed)
    cfg = _config(case)
    H, KV, hd = case["heads"], case["kv_heads"], case["head_dim"]
    sizes = [len(t) for t in tokens]
    pos = torch.cat([torch.arange(n, device="cuda") for n in sizes])
    inv = torch.tensor(cfg.rope_base, dtype=torch.float64) ** (-torch.arange(0, hd, 2, dtype=torch.float64) / hd)
    angle = (pos.float().unsqueeze(1) * inv.float().cuda()).double().unsqueeze(1)  # angles are defined in float32
    cos, sin = torch.cos(angle), torch.sin(angle)

    def decode(m):
        return _decode(m[0], m[1], m[2], m[3])

    def product(m, x):
        return _quantized(m[0], x) @ decode(m).T

    def heads(v, count, norm):
        v = v.view(-1, count, hd)
        if norm is not None:
            v = v / torch.sqrt((v * v).mean(2, keepdim=True) + cfg.rms_eps) * norm.double()
        out = torch.empty_like(v)
        a, b = (v[..., :hd // 2], v[..., hd // 2:]) if cfg.rope_neox else (v[..., 0::2], v[..., 1::2])
        r, i = a * cos - b * sin, a * sin + b * cos
        if cfg.rope_neox:
            out[..., :hd // 2], out[..., hd // 2:] = r, i
        else:
            out[..., 0::2], out[..., 1::2] = r, i
        return out

    def attend(q, k, v):  # one sequence: [n][heads][hd]
        n, out = q.shape[0], torch.empty_like(q)
        at = torch.arange(n, device="cuda")
        for h in range(H):
            kh, vh = k[:, h * KV // H], v[:, h * KV // H]
            s = q[:, h] @ kh.T / math.sqrt(hd)
            s.masked_fill_(at.unsqueeze(0) > at.unsqueeze(1), -math.inf)
            out[:, h] = torch.softmax(s, 1) @ vh
        return out

    ids = torch.from_numpy(np.concatenate(tokens).astype(np.int64)).cuda()
    fmt, raw, rows, cols = io["tok_embd"]
    x = _decode(fmt, raw.view(rows, -1)[ids].reshape(-1, raw.shape[1]), len(ids), cols)
    for layer in layers:
        xb = _rms(x, layer["attn_norm"], cfg.rms_eps)
        q = heads(product(layer["wq"], xb), H, layer.get("q_norm"))
        k = heads(product(layer["wk"], xb), KV, layer.get("k_norm")).half().double()  # the cache holds 16 bits
        v = product(layer["wv"], xb).view(-1, KV, hd).half().double()
        att = torch.cat([attend(a, b, c) for a, b, c in zip(q.split(sizes), k.split(sizes), v.split(sizes))])
        x = x + product(layer["wo"], att.reshape(-1, H * hd))
        xb = _rms(x, layer["ffn_norm"], cfg.rms_eps)
        x = x + product(layer["w_down"], _silu(product(layer["w_gate"], xb)) * product(layer["w_up"], xb))
    ends = torch.tensor(sizes, device="cuda").cumsum(0) - 1
    y = product(io["output"], _rms(x[ends], io["out_norm"], cfg.rms_eps))
    return y[0] if case["seqs"] == 1 else y


def exact(case, seed):
    return (_exact_linear if case["kind"] == "linear" else _exact_net)(case, seed)

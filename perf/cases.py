"""The work that programs built on qste_amd have it do, as cases to time.

Each case is a dict of plain values; ``prepare`` makes what a program holds
before the call, ``run`` is one pass through the public entry points.  Kinds:

``decode``   token generation from exported weights: the SwiGLU MLPs of
             ``blocks`` decoder layers (``PackedLinear`` gate and up, the
             fused gate, ``PackedLinear`` down) for ``m`` sequences, replayed
             from a captured graph, each layer on the input that attention
             and norm would hand it
``linear``   one exported layer (``PackedLinear``) called eagerly
``train``    one ``QSTELinear``: forward, and backward with the evidence
             taken by the surface's sink
``gelu_mlp`` a GPT-2 MLP as ``convert`` leaves it (two binary layers with
             biases, packed tanh-GELU between them), forward and backward
``swiglu``   the SwiGLU MLP as one node (``nn.swiglu_mlp``), both directions
``table``    one vocabulary table used as the embedding and as the output
             head (tied, so its evidence is the sum of both uses)
``step``     the coordinate optimizer: evidence of every surface delivered,
             then ``QSTEOptimizer.step``
"""

from __future__ import annotations

import math

import torch
import torch.nn as nn
import torch.nn.functional as F

import qste_amd as qste

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # one sequence at a time through the MLPs of a Llama-3-8B-shaped decoder
        {"name": "decode_1", "kind": "decode", "m": 1, "d": 4096, "ffn": 14336, "blocks": 8, "dtype": "bf16"},
        # a small batch over the 28672 x 8192 matrices of a 70B-shaped MLP
        {"name": "decode_16", "kind": "decode", "m": 16, "d": 8192, "ffn": 28672, "blocks": 2, "dtype": "fp16"},
        # continuous batching: some forty sequences decode together
        {"name": "decode_40", "kind": "decode", "m": 40, "d": 4096, "ffn": 14336, "blocks": 8, "dtype": "bf16"},
        # the smallest call: one row through an exported fp32 layer
        {"name": "linear_fp32_1", "kind": "linear", "m": 1, "rows": 2048, "cols": 2048, "dtype": "fp32",
         "bias": True},
        # prefill of a prompt of no particular length
        {"name": "linear_prefill", "kind": "linear", "m": 1531, "rows": 4096, "cols": 4096, "dtype": "bf16",
         "bias": False},
        # a small fp32 layer with a bias (the 2048 -> 2048, 256-token workload)
        {"name": "train_fp32", "kind": "train", "tokens": 256, "rows": 2048, "cols": 2048, "dtype": "fp32",
         "bias": True},
        # a layer of the d=1024 ReLU MLP at 8192 tokens
        {"name": "train_bf16", "kind": "train", "tokens": 8192, "rows": 4096, "cols": 1024, "dtype": "bf16",
         "bias": True},
        # GPT-2 small's MLP, 8 sequences of 1023 predicted tokens
        {"name": "gelu_mlp", "kind": "gelu_mlp", "tokens": 8184, "d": 768, "ffn": 3072, "dtype": "bf16"},
        # the Llama-3-8B-shaped SwiGLU MLP at 16384 tokens, the largest case
        {"name": "swiglu", "kind": "swiglu", "tokens": 16384, "d": 4096, "ffn": 14336},
        # GPT-2's tied vocabulary table (an odd number of rows), 2 sequences of 1023
        {"name": "table", "kind": "table", "vocab": 50257, "d": 768, "tokens": 2046},
        # the optimizer over the first MLP matrices of eight GPT-2 layers
        {"name": "step_small", "kind": "step", "surfaces": 8, "rows": 3072, "cols": 768, "block": 256},
        # the optimizer over one Llama-3-8B MLP matrix
        {"name": "step_large", "kind": "step", "surfaces": 1, "rows": 14336, "cols": 4096, "block": 256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, grains=(256, 64, 64, 8, 1)):
    """A size between lo and hi, even over its logarithm, a multiple of one of the grains."""
    g = rng.choice(grains)
    return max(g, min(hi // g, max(-(-lo // g), round(_log(rng, lo, hi) / g))) * g)


def draw(rng):
    kind = rng.choice(["decode", "decode", "linear", "linear", "train", "train", "gelu_mlp", "swiglu", "table", "step"])
    if kind == "decode":
        m = _log(rng, 1, 96)
        d = _size(rng, 1024, 8192, (256, 128))
        ffn = _size(rng, 2 * d, 4 * d, (256, 128))
        blocks = max(1, min(8, (8 * 4096 * 14336) // (d * ffn)))
        return {"kind": kind, "m": m, "d": d, "ffn": ffn, "blocks": blocks, "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if kind == "linear":
        return {"kind": kind, "m": _log(rng, 1, 4096), "rows": _size(rng, 256, 8192), "cols": _size(rng, 256, 8192),
                "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"]), "bias": rng.random() < 0.5}
    if kind == "train":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        rows, cols = _size(rng, 256, 4096), _size(rng, 256, 4096)
        most = min(8192, (1 << 36 if dtype != "fp32" else 1 << 34) // (rows * cols))
        return {"kind": kind, "tokens": _log(rng, 64, max(65, most)), "rows": rows, "cols": cols, "dtype": dtype,
                "bias": rng.random() < 0.5}
    if kind == "gelu_mlp":
        d = _size(rng, 384, 1600, (64,))
        return {"kind": kind, "tokens": _log(rng, 256, 8192), "d": d, "ffn": 4 * d, "dtype": rng.choice(["bf16", "fp16"])}
    if kind == "swiglu":
        d = _size(rng, 1024, 4096, (256, 64))
        ffn = _size(rng, 2 * d, min(14336, 4 * d), (256, 64))
        return {"kind": kind, "tokens": _log(rng, 512, 16384), "d": d, "ffn": ffn}
    if kind == "table":
        return {"kind": kind, "vocab": _log(rng, 8192, 50304), "d": _size(rng, 384, 1024, (128, 64)),
                "tokens": _log(rng, 256, 2048)}
    rows, cols = _size(rng, 256, 14336), _size(rng, 256, 8192)
    return {"kind": "step", "surfaces": max(1, min(8, (4096 * 14336) // (rows * cols))), "rows": rows, "cols": cols,
            "block": rng.choice([256, 256, 128])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


class _Seeded:
    """Tensors of one seeded stream on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, std=1.0):
        return torch.randn(*shape, generator=self.g, device=DEV).mul_(std).to(dtype)

    def bits(self, rows, cols):
        """Packed random signs; the bits past the last column are zero."""
        packed = torch.randint(0, 256, (rows, (cols + 7) // 8), generator=self.g, device=DEV, dtype=torch.uint8)
        if cols % 8:
            packed[:, -1] &= (1 << (cols % 8)) - 1
        return packed

    def coordinate(self, rows, cols):
        return torch.randint(-127, 128, (rows, cols), generator=self.g, device=DEV, dtype=torch.int8)

    def scale(self, rows, around):
        """Positive row scales spread by about a third around one value."""
        return around * (1.0 + 0.3 * torch.rand(rows, generator=self.g, device=DEV))


def _packed_layer(s, rows, cols, bias=False):
    b = s.normal(rows, std=0.1) if bias else None
    return qste.PackedLinear(s.bits(rows, cols), s.scale(rows, cols ** -0.5), cols, b)


def _layer(s, rows, cols, bias=False):
    surface = qste.Surface.from_state(s.coordinate(rows, cols), s.scale(rows, cols ** -0.5).log())
    return qste.QSTELinear(surface, s.normal(rows, std=0.1) if bias else None)


def _collect(surfaces):
    """The surfaces' evidence goes into a dict, as a program that applies it itself takes it."""
    got = {}
    for i, surface in enumerate(surfaces):
        surface.route_evidence(lambda _, evidence, i=i: got.__setitem__(i, evidence))
    return got


class _DecodeMLP(nn.Module):
    def __init__(self, s, d, ffn):
        super().__init__()
        self.gate, self.up = _packed_layer(s, ffn, d), _packed_layer(s, ffn, d)
        self.down = _packed_layer(s, d, ffn)

    def forward(self, x):
        return self.down(qste.nn.swiglu(self.gate(x), self.up(x)))


def prepare(case, seed):
    s = _Seeded(seed)
    kind = case["kind"]
    st = {"kind": kind}
    if kind == "decode":
        dtype = DTYPES[case["dtype"]]
        mlps = [_DecodeMLP(s, case["d"], case["ffn"]) for _ in range(case["blocks"])]
        xs = [s.normal(case["m"], case["d"], dtype=dtype) for _ in mlps]
        with torch.no_grad():
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):  # once off the capture
                mlps[0](xs[0])
            torch.cuda.current_stream().wait_stream(side)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                ys = [mlp(x) for mlp, x in zip(mlps, xs)]
        st.update(mlps=mlps, xs=xs, ys=ys, graph=graph)
    elif kind == "linear":
        st.update(layer=_packed_layer(s, case["rows"], case["cols"], case["bias"]),
                  x=s.normal(case["m"], case["cols"], dtype=DTYPES[case["dtype"]]))
    elif kind == "train":
        dtype = DTYPES[case["dtype"]]
        layer = _layer(s, case["rows"], case["cols"], case["bias"])
        st.update(layer=layer, evidence=_collect([layer.surface]),
                  x=s.normal(case["tokens"], case["cols"], dtype=dtype).requires_grad_(True),
                  dy=s.normal(case["tokens"], case["rows"], dtype=dtype))
    elif kind == "gelu_mlp":
        dtype = DTYPES[case["dtype"]]
        d, ffn = case["d"], case["ffn"]
        mlp = nn.Sequential(_layer(s, ffn, d, True), qste.nn.GELU(approximate="tanh"), _layer(s, d, ffn, True))
        st.update(mlp=mlp, evidence=_collect([mlp[0].surface, mlp[2].surface]),
                  x=s.normal(case["tokens"], d, dtype=dtype).requires_grad_(True),
                  dy=s.normal(case["tokens"], d, dtype=dtype))
    elif kind == "swiglu":
        d, ffn = case["d"], case["ffn"]
        layers = [_layer(s, ffn, d), _layer(s, ffn, d), _layer(s, d, ffn)]
        st.update(layers=layers, evidence=_collect([m.surface for m in layers]),
                  x=s.normal(case["tokens"], d, dtype=torch.bfloat16).requires_grad_(True),
                  dy=s.normal(case["tokens"], d, dtype=torch.bfloat16))
    elif kind == "table":
        vocab, d, tokens = case["vocab"], case["d"], case["tokens"]
        surface = qste.Surface.from_state(s.coordinate(vocab, d), s.scale(vocab, 0.02).log())
        surface = surface.to(torch.bfloat16)  # a bf16 model: the integer state stays as it is
        st.update(embedding=qste.QSTEEmbedding(surface), head=qste.QSTELinear(surface), surface=surface,
                  evidence=_collect([surface]),
                  ids=torch.randint(0, vocab, (tokens,), generator=s.g, device=DEV),
                  hidden=s.normal(tokens, d, dtype=torch.bfloat16),  # what the decoder adds to its input
                  dlogits=s.normal(tokens, vocab, dtype=torch.bfloat16, std=0.01))
    else:
        rows, cols = case["rows"], case["cols"]
        surfaces = [_layer(s, rows, cols).surface for _ in range(case["surfaces"])]
        optimizer = qste.QSTEOptimizer(surfaces, qste.QSTEConfig(momentum_block_size=case["block"]))
        st.update(surfaces=surfaces, optimizer=optimizer, evidence=[s.normal(rows, cols) for _ in surfaces])
        for _ in range(32):  # past the first steps, where the update clip always engages
            run(st)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(st):
    kind = st["kind"]
    if kind == "decode":
        st["graph"].replay()
        return st["ys"]
    if kind == "linear":
        return st["layer"](st["x"])
    if kind == "step":
        opt = st["optimizer"]
        for surface, evidence in zip(st["surfaces"], st["evidence"]):
            surface.consume_evidence(evidence)
        flips = opt.step()
        return [flips] + [[s.coordinate, s.packed_sign, *(opt.state[id(s)][k] for k in ("moment_q", "moment_scale", "row_v", "col_v"))]
                          for s in st["surfaces"]]
    st["evidence"].clear()
    if kind == "train":
        layer = st["layer"]
        y = layer(st["x"])
        leaves = [st["x"], layer.surface.log_scale] + ([] if layer.bias is None else [layer.bias])
        grads = torch.autograd.grad(y, leaves, st["dy"])
    elif kind == "gelu_mlp":
        first, second = st["mlp"][0], st["mlp"][2]
        y = st["mlp"](st["x"])
        grads = torch.autograd.grad(
            y, [st["x"], first.surface.log_scale, first.bias, second.surface.log_scale, second.bias], st["dy"])
    elif kind == "swiglu":
        y = qste.nn.swiglu_mlp(st["x"], *st["layers"])
        grads = torch.autograd.grad(y, [st["x"], *(m.surface.log_scale for m in st["layers"])], st["dy"])
    else:
        hidden = st["embedding"](st["ids"]) + st["hidden"]
        y = st["head"](hidden)
        grads = torch.autograd.grad(y, [st["surface"].log_scale], st["dlogits"])
    return [y, list(grads), [st["evidence"][i] for i in sorted(st["evidence"])]]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    size = DTYPES[case["dtype"]].itemsize if "dtype" in case else 2
    if kind == "decode":
        m, d, ffn, b = case["m"], case["d"], case["ffn"], case["blocks"]
        return {"bytes": b * (3 * d * ffn / 8 + 4 * (2 * ffn + d) + 2 * m * d * size), "flops": b * 6 * m * d * ffn}
    if kind == "linear":
        m, r, c = case["m"], case["rows"], case["cols"]
        return {"bytes": r * c / 8 + 4 * r + m * (r + c) * size, "flops": 2 * m * r * c}
    if kind == "train":
        t, r, c = case["tokens"], case["rows"], case["cols"]
        # x, dy read; y, dx, evidence written; signs read
        return {"bytes": 2 * t * (r + c) * size + 4 * r * c + r * c / 8, "flops": 6 * t * r * c}
    if kind == "gelu_mlp":
        t, d, f = case["tokens"], case["d"], case["ffn"]
        return {"bytes": 4 * t * d * size + 2 * (4 * d * f + d * f / 8), "flops": 12 * t * d * f}
    if kind == "swiglu":
        t, d, f = case["tokens"], case["d"], case["ffn"]
        return {"bytes": 4 * t * d * 2 + 3 * (4 * d * f + d * f / 8), "flops": 18 * t * d * f}
    if kind == "table":
        t, v, d = case["tokens"], case["vocab"], case["d"]
        return {"bytes": 2 * t * v * 2 + t * d * 2 + 4 * v * d + v * d / 8, "flops": 6 * t * v * d}
    n, r, c = case["surfaces"], case["rows"], case["cols"]
    # evidence read; coordinate and momentum read and written; signs written
    return {"bytes": n * (8 * r * c + r * c / 8 + 4 * r * c / case["block"] + 4 * (r + c)), "flops": n * 20 * r * c}


def tolerance(case):
    if case["kind"] == "step":
        return "exact"  # whole numbers, and fp16 statistics of sums formed in 64 bits
    if case.get("dtype") == "fp32":
        # 32-bit sums of up to 8192 terms; an element that sits on its row's
        # mean may be encoded on either side, which moves one evidence column
        return {"rel": 1e-5, "max": 2e-4}
    if case["kind"] in ("linear", "train"):
        return {"rel": 4e-3, "max": 4e-2}
    return {"rel": 1e-2, "max": 2e-1}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------


def _signs(packed, cols):
    shifts = torch.arange(8, device=packed.device, dtype=torch.uint8)
    bits = (packed.unsqueeze(-1) >> shifts) & 1
    return bits.reshape(packed.shape[0], -1)[:, :cols].double().mul_(2).sub_(1)


def _affine(x):
    """What a layer keeps of its input: offset + scale * sign(x - offset) per row."""
    offset = x.mean(1, keepdim=True)
    centered = x - offset
    sign = (centered >= 0).double().mul_(2).sub_(1)
    return sign.mul_(centered.abs().mean(1, keepdim=True)).add_(offset)


class _Exact:
    """One binary layer in 64 bits: signs, row scale and bias."""

    def __init__(self, signs, scale, bias=None):
        self.s, self.scale = signs, scale.double()
        self.bias = None if bias is None else bias.detach().double()

    @classmethod
    def of(cls, layer):
        surface = layer.surface
        scale = surface.log_scale.detach().double().exp().clamp(surface.cfg.scale_min, surface.cfg.scale_max)
        return cls(_signs(surface.packed_sign.data, surface.columns), scale, layer.bias)

    def forward(self, x):
        y = (x @ self.s.t()).mul_(self.scale)
        return y if self.bias is None else y.add_(self.bias)

    def backward(self, x, dy):
        """(dx, evidence, gradient of the log scale, gradient of the bias)."""
        dx = (dy * self.scale) @ self.s
        e = dy.t() @ _affine(x)
        ds = (e * self.s).sum(1) * self.scale
        return dx, e.mul_(self.scale.unsqueeze(1)), ds, None if self.bias is None else dy.sum(0)


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return None  # whole numbers that the specification fixes
    st = prepare(case, seed)
    if kind == "decode":
        ys = []
        for mlp, x in zip(st["mlps"], st["xs"]):
            def lin(m, v):
                return (v @ _signs(m.packed_sign, m.in_features).t()).mul_(m.scale.double())
            g, u = lin(mlp.gate, x.double()), lin(mlp.up, x.double())
            ys.append(lin(mlp.down, F.silu(g) * u))
        return ys
    if kind == "linear":
        m = st["layer"]
        return _Exact(_signs(m.packed_sign, m.in_features), m.scale, m.bias).forward(st["x"].double())
    if kind == "train":
        layer = _Exact.of(st["layer"])
        x = st["x"].detach().double()
        dx, e, ds, db = layer.backward(x, st["dy"].double())
        return [layer.forward(x), [dx, ds] + ([] if db is None else [db]), [e]]
    if kind == "gelu_mlp":
        first, second = _Exact.of(st["mlp"][0]), _Exact.of(st["mlp"][2])
        x, dy = st["x"].detach().double(), st["dy"].double()
        a = first.forward(x).requires_grad_(True)
        h = F.gelu(a, approximate="tanh")
        (slope,) = torch.autograd.grad(h.sum(), a)
        h = h.detach()
        step = slope.abs().amax(1, keepdim=True) / 127  # the slope is kept in 8 bits
        dh, e2, ds2, db2 = second.backward(h, dy)
        da = dh * (slope / step).round_().mul_(step)
        dx, e1, ds1, db1 = first.backward(x, da)
        return [second.forward(h), [dx, ds1, db1, ds2, db2], [e1, e2]]
    if kind == "swiglu":
        gate, up, down = (_Exact.of(m) for m in st["layers"])
        x, dy = st["x"].detach().double(), st["dy"].double()
        g, u = gate.forward(x), up.forward(x)
        silu, sig = F.silu(g), torch.sigmoid(g)
        h = silu * u
        y = down.forward(h)
        dh, ed, dsd, _ = down.backward(h, dy)
        slope = sig.mul_(1 + g - silu)
        dxg, eg, dsg, _ = gate.backward(x, dh * u * slope)
        dxu, eu, dsu, _ = up.backward(x, dh * silu)
        return [y, [dxg + dxu, dsg, dsu, dsd], [eg, eu, ed]]
    head = _Exact.of(st["head"])
    ids, dl = st["ids"], st["dlogits"].double()
    hidden = head.s[ids] * head.scale[ids].unsqueeze(1) + st["hidden"].double()
    dx, e, ds, _ = head.backward(hidden, dl)
    g = torch.zeros_like(head.s).index_add_(0, ids, dx)
    ds += (g * head.s).sum(1) * head.scale
    e += g * head.scale.unsqueeze(1)
    return [head.forward(hidden), [ds], [e]]

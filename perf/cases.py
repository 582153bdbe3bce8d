"""Performance cases: the work this framework is asked to do, through its public entry points.

Two kinds of calls are covered.  A worker translates packed batches with an
engine (HipEngine); a host that drives the layers itself calls the op-level
functions of marian-edge_amd/device.py on device buffers.  Sizes are the
repository's own: the 64-sentence and the 256-item batches of bench.py, the
GEMM shapes and rows and the packed attention workload of bench_ops.py, the
512-wide transformer (8 heads of 64, FFN 2048) and the 384-wide SSRU graph
(8 heads of 48, FFN 1536), both over 32000 ids.

listed() names the cases, draw() gives more of the same ranges, prepare()
builds what a caller holds before the call, run() is one call, exact() the
same result in 64-bit arithmetic from plain torch, work() the bytes and
operations no implementation can do without.
"""

from __future__ import annotations

import importlib
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

_ROOT = Path(__file__).resolve().parents[1]
_NAME = "marian_edge_amd"
_VOCAB = 32000
_DEV = "cuda"


def _package():
    """The package directory marian-edge_amd/ (not an identifier), as marian_edge_amd."""
    if _NAME not in sys.modules:
        where = _ROOT / "marian-edge_amd"
        spec = importlib.util.spec_from_file_location(_NAME, where / "__init__.py",
                                                      submodule_search_locations=[str(where)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[_NAME] = mod
        spec.loader.exec_module(mod)
    return sys.modules[_NAME]


def _device():
    return importlib.import_module(_package().__name__ + ".device")


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # One decode row through the FFN's first layer: the smallest call a host makes, all latency.
        _linear("linear-decode-1", 1, 512, 2048, relu=True),
        # One decode step of a 61-sentence batch through the SSRU graph's FFN down-projection
        # (static activation multiplier, 1536 -> 384).
        _linear("linear-static-61", 61, 1536, 384, act="static"),
        # The encoder of the 64-sentence batch: 1459 packed rows through the FFN's first layer.
        _linear("linear-encoder-1459", 1459, 512, 2048, relu=True),
        # Scoring many rows against the whole vocabulary (the largest shape of the GEMM sweep).
        _linear("linear-vocab-4096", 4096, 512, _VOCAB),
        # Encoder self-attention of 256 packed sentences, lengths lognormal(3.2, 0.6) in [4, 256].
        _attention("attention-self-256", 256, "sentences", 2),
        # The same layer over long segments (texts split at 256 tokens), bfloat16 inputs.
        _attention("attention-long-bf16", 48, "segments", 7, bf16=True),
        # Cross-attention of one decode step: one query per sentence over its encoder rows.
        _attention("attention-cross-256", 256, "sentences", 2, cross=True),
        # The encoder's post-norm on the rows of the 256-sentence workload, quantized for the next layer.
        _norm("norm-7405", 7405, 512),
        # Token choice of one 64-row decode step over the whole vocabulary, logits kept.
        _vocab("vocab-argmax-64", 64, 512),
        # Token choice over lexical-shortlist candidates, 64 rows of the SSRU graph.
        _candidates("candidates-64", 64, 384, 1000),
        # The headline batch: 64 ragged sentences, greedy decoding to their forced stops.
        _translate("translate-ragged-64", "transformer", "ragged", 64, 3),
        # The largest batch: 256 items, long ones split at 256 tokens, stops up to 512.
        _translate("translate-stress-256", "transformer", "stress", 256, 4),
    ]


def _case(name, **fields):
    return dict(fields, name=name) if name else dict(fields)


def _linear(name, m, k, n, relu=False, act="dynamic", i32=False):
    return _case(name, kind="linear", m=m, k=k, n=n, relu=relu, act=act, i32=i32)


def _attention(name, n, lengths, shape_seed, heads=8, head_dim=64, bf16=False, cross=False):
    return _case(name, kind="attention", n=n, lengths=lengths, shape_seed=shape_seed, heads=heads,
                 head_dim=head_dim, bf16=bf16, cross=cross)


def _norm(name, rows, dim, op="residual"):
    return _case(name, kind="norm", rows=rows, dim=dim, op=op)


def _vocab(name, m, k, v=_VOCAB, logits=True):
    return _case(name, kind="vocab", m=m, k=k, v=v, logits=logits)


def _candidates(name, m, k, longest, v=_VOCAB):
    return _case(name, kind="candidates", m=m, k=k, longest=longest, v=v)


def _translate(name, graph, style, n, shape_seed):
    return _case(name, kind="translate", graph=graph, style=style, n=n, shape_seed=shape_seed)


def _log(rng, lo, hi):
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "attention", "attention", "attention", "norm", "vocab",
                       "candidates", "translate"])
    if kind == "linear":
        k, n = rng.choice([(512, 1536), (512, 512), (512, 2048), (2048, 512), (512, _VOCAB),
                           (384, 1152), (384, 384), (384, 1536), (1536, 384), (384, _VOCAB),
                           (64 * rng.randint(1, 32), rng.randint(100, 2500))])
        m = _log(rng, 1, 16384 if n < 4096 else 4096)
        return _linear(None, m, k, n, relu=rng.random() < 0.3,
                       act=rng.choice(["dynamic", "dynamic", "quantized", "static"]), i32=rng.random() < 0.2)
    if kind == "attention":
        lengths = rng.choice(["sentences", "sentences", "segments", "long"])
        n = _log(rng, 1, {"sentences": 512, "segments": 96, "long": 24}[lengths])
        return _attention(None, n, lengths, rng.randrange(1 << 16), heads=rng.choice([8, 8, 4]),
                          head_dim=rng.choice([64, 64, 48]), bf16=rng.random() < 0.35, cross=rng.random() < 0.3)
    if kind == "norm":
        return _norm(None, _log(rng, 1, 16384), rng.choice([512, 512, 384, 384, 256, 64 * rng.randint(1, 16)]),
                     op=rng.choice(["residual", "residual", "ssru"]))
    if kind == "vocab":
        return _vocab(None, _log(rng, 1, 512), rng.choice([512, 512, 384, 256]),
                      v=rng.choice([_VOCAB, _VOCAB, _log(rng, 2000, 40000)]), logits=rng.random() < 0.5)
    if kind == "candidates":
        return _candidates(None, _log(rng, 1, 512), rng.choice([384, 384, 512, 256]), _log(rng, 104, 4000))
    return _translate(None, rng.choice(["transformer", "transformer", "ssru"]), rng.choice(["ragged", "ragged", "stress"]),
                      _log(rng, 1, 256), rng.randrange(1 << 16))


def _lengths(case):
    """Sequence lengths of an attention case (its shape does not depend on the seed of the inputs)."""
    r = np.random.Generator(np.random.PCG64(case["shape_seed"]))
    n = case["n"]
    if case["lengths"] == "sentences":  # the packed workload of bench_ops.py
        return np.clip(np.rint(r.lognormal(3.2, 0.6, size=n)), 4, 256).astype(np.int64)
    if case["lengths"] == "segments":  # long texts split at 256 tokens
        return r.integers(96, 257, size=n)
    return r.integers(257, 513, size=n)  # unsplit long texts


def _batch(case):
    """The packed batch of a translate case: lengths and forced stops from its shape seed."""
    pkg = _package()
    make = pkg.ragged_batch if case["style"] == "ragged" else pkg.stress_batch
    return make(seed=case["shape_seed"], n=case["n"], vocab=_VOCAB)


def _probe_step(batch):
    return min(8, int(batch.max_output_tokens.max()) - 1)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
class _Buf:
    """A torch tensor on the GPU as the device buffer the op-level functions take."""

    __slots__ = ("t", "ptr", "shape", "dtype")

    def __init__(self, t):
        self.t, self.ptr, self.shape, self.dtype = t, t.data_ptr(), tuple(t.shape), t.dtype


def _gen(seed):
    g = torch.Generator(device=_DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=_DEV, dtype=torch.float32)


def _uniform(g, lo, hi, n):
    return torch.rand(n, generator=g, device=_DEV, dtype=torch.float32) * (hi - lo) + lo


def _weights(g, n, k):
    """int8 weights with per-column multipliers 1 / s, s ~ U(0.001, 0.02), and biases N(0, 0.02)."""
    w = torch.randint(-127, 128, (n, k), generator=g, device=_DEV, dtype=torch.int8)
    return w, 1.0 / _uniform(g, 0.001, 0.02, n), 0.02 * _normal(g, n)


def _row_multiplier(x):
    """127 / max|row| in 32 bits (1 for a zero row), on the host: IEEE division."""
    m = x.abs().amax(dim=1).cpu().numpy()
    return torch.from_numpy(np.where(m > 0, np.float32(127) / np.where(m > 0, m, np.float32(1)),
                                     np.float32(1)).astype(np.float32)).to(x.device)


def _quantize(x, a):
    """q = clamp(rne(x a), -127, 127) with the product in 32 bits."""
    return torch.clamp(torch.round(x * a[:, None]), -127, 127).to(torch.int8)


_STATIC_MULT = float(np.float32(127.0 / 4.5))  # LayerNorm outputs lie within about 4.5


def _inputs(case, seed):
    """The call's inputs as torch tensors, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "linear":
        x = _normal(g, case["m"], case["k"])
        w, mult, bias = _weights(g, case["n"], case["k"])
        got = dict(x=x, w=w, mult=mult, bias=bias)
        if case["act"] == "quantized":
            got["a"] = _row_multiplier(x)
            got["q"] = _quantize(x, got["a"])
        return got
    if kind == "attention":
        lens = _lengths(case)
        cu = np.zeros(len(lens) + 1, np.int64)
        cu[1:] = np.cumsum(lens)
        t, d = int(cu[-1]), case["heads"] * case["head_dim"]
        rows = len(lens) if case["cross"] else t
        dt = torch.bfloat16 if case["bf16"] else torch.float32
        seq = np.arange(len(lens)) if case["cross"] else np.repeat(np.arange(len(lens)), lens)
        return dict(q=_normal(g, rows, d).to(dt), k=_normal(g, t, d).to(dt), v=_normal(g, t, d).to(dt),
                    seq=torch.from_numpy(seq.astype(np.int32)).to(_DEV),
                    cu=torch.from_numpy(cu.astype(np.int32)).to(_DEV))
    if kind == "norm":
        r, d = case["rows"], case["dim"]
        got = dict(x=_normal(g, r, d), r=_normal(g, r, d), scale=1.0 + 0.02 * _normal(g, d), bias=0.02 * _normal(g, d))
        if case["op"] == "ssru":
            got["forget"], got["state"] = _normal(g, r, d), _normal(g, r, d)
        return got
    if kind in ("vocab", "candidates"):
        # Rows are LayerNorm outputs, embedding columns N(0, 0.02) quantized per id.
        x = _normal(g, case["m"], case["k"])
        e = 0.02 * _normal(g, case["v"], case["k"])
        mult = _row_multiplier(e)
        a = _row_multiplier(x)
        got = dict(q=_quantize(x, a), a=a, emb=_quantize(e, mult), mult=mult, bias=0.02 * _normal(g, case["v"]))
        if kind == "candidates":
            counts = _cand_counts(case)
            off = np.zeros(case["m"] + 1, np.int64)
            off[1:] = np.cumsum(counts)
            ids = np.random.Generator(np.random.PCG64(int(seed) & 0x7FFFFFFF))
            lists = [np.sort(ids.permutation(case["v"] - 1)[:c - 1] + 1) for c in counts]
            flat = np.concatenate([np.concatenate([[0], one]) for one in lists])
            got["cand"] = torch.from_numpy(flat.astype(np.int32)).to(_DEV)
            got["off"] = torch.from_numpy(off.astype(np.int32)).to(_DEV)
        return got
    batch = _batch(case)
    ids = np.random.Generator(np.random.PCG64(int(seed) & 0x7FFFFFFF))
    return dict(batch=batch, tokens=ids.integers(3, _VOCAB, size=batch.tokens.size).astype(np.int32))


def _cand_counts(case):
    """Candidates per row: multiples of 8 (the shortlist pads to them), at most case["longest"]."""
    r = np.random.Generator(np.random.PCG64(case["m"] * 8191 + case["longest"]))
    c = np.maximum(104, r.integers(case["longest"] // 3, case["longest"] + 1, size=case["m"]))
    return (c + 7) // 8 * 8


_engines = {}


def _engine(graph):
    """The engine of a graph: a program loads its model once and translates many batches."""
    if graph not in _engines:
        pkg = _package()
        model = pkg.seeded_ssru_model() if graph == "ssru" else pkg.seeded_model()
        _engines[graph] = (pkg.HipEngine(model, limits=pkg.LIFTED_LIMITS), model)
    return _engines[graph]


def prepare(case, seed):
    got = _inputs(case, seed)
    kind = case["kind"]
    if kind == "translate":
        got["engine"] = _engine(case["graph"])[0]
        got["probe_step"] = _probe_step(got["batch"])
        got["kind"] = kind
        return got
    s = {name: _Buf(t) for name, t in got.items()}
    new = lambda shape, dtype: _Buf(torch.zeros(shape, device=_DEV, dtype=dtype))  # noqa: E731
    if kind == "linear":
        s["out"] = new((case["m"], case["n"]), torch.float32)
        s["acc"] = new((case["m"], case["n"]), torch.int32) if case["i32"] else None
    elif kind == "attention":
        s["out"] = new(got["q"].shape, torch.float32)
        s["max_keys"] = int(_lengths(case).max())
    elif kind == "norm":
        s["out"] = new((case["rows"], case["dim"]), torch.float32)
        s["oq"], s["oa"] = new((case["rows"], case["dim"]), torch.int8), new((case["rows"],), torch.float32)
    elif kind == "vocab":
        s["token"] = new((case["m"],), torch.int32)
        s["logits"] = new((case["m"], case["v"]), torch.float32) if case["logits"] else None
    else:
        s["token"] = new((case["m"],), torch.int32)
        s["logits"] = new((got["cand"].numel(),), torch.float32)
        s["longest"] = int(_cand_counts(case).max())
    s["case"], s["kind"] = dict(case), kind
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind == "translate":
        b = s["batch"]
        out, enc, logits, active = s["engine"].translate_probe(
            s["tokens"], b.offsets, b.max_output_tokens, flags=_package().FLAG_IGNORE_EOS, probe_step=s["probe_step"])
        return dict(tokens=out.tokens, offsets=out.offsets, encoder=enc, logits=logits, active=active)
    dev, c = _device(), s["case"]
    if kind == "linear":
        if c["act"] == "static":
            dev.q8_linear_static(s["x"], _STATIC_MULT, s["w"], s["mult"], s["bias"], s["acc"], s["out"], relu=c["relu"])
        elif c["act"] == "quantized":
            dev.q8_linear(None, s["w"], s["mult"], s["bias"], s["acc"], s["out"], relu=c["relu"], xq=s["q"], xa=s["a"])
        else:
            dev.q8_linear(s["x"], s["w"], s["mult"], s["bias"], s["acc"], s["out"], relu=c["relu"])
        return dict(out=s["out"].t, acc=s["acc"].t) if c["i32"] else s["out"].t
    if kind == "attention":
        dev.attention(s["q"], s["k"], s["v"], s["seq"], s["cu"], s["out"], heads=c["heads"], max_keys=s["max_keys"],
                      bf16=c["bf16"], packed_self=not c["cross"], head_dim=c["head_dim"])
        return s["out"].t
    if kind == "norm":
        if c["op"] == "ssru":
            state = _Buf(s["state"].t.clone())  # the call updates it in place
            dev.ssru_layer_norm(s["x"], s["forget"], state, s["r"], s["scale"], s["bias"], s["out"], s["oq"], s["oa"])
            return dict(out=s["out"].t, q=s["oq"].t, a=s["oa"].t, state=state.t)
        dev.residual_layer_norm(s["x"], s["r"], s["scale"], s["bias"], s["out"], s["oq"], s["oa"])
        return dict(out=s["out"].t, q=s["oq"].t, a=s["oa"].t)
    if kind == "vocab":
        dev.vocab_argmax(s["q"], s["a"], s["emb"], s["mult"], s["bias"], s["token"], logits=s["logits"])
        return dict(token=s["token"].t, logits=s["logits"].t) if c["logits"] else s["token"].t
    dev.candidate_argmax(s["q"], s["a"], s["emb"], s["mult"], s["bias"], s["cand"], s["off"], s["longest"], s["token"],
                         logits=s["logits"])
    return dict(token=s["token"].t, logits=s["logits"].t)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        a = k + 4 if case["act"] == "quantized" else 4 * k
        return {"bytes": m * a + k * n + 8 * n + (8 if case["i32"] else 4) * m * n, "flops": 2 * m * n * k}
    if kind == "attention":
        lens = _lengths(case)
        t, d, b = int(lens.sum()), case["heads"] * case["head_dim"], 2 if case["bf16"] else 4
        rows = len(lens) if case["cross"] else t
        pairs = t if case["cross"] else int((lens ** 2).sum())
        return {"bytes": 2 * t * d * b + rows * d * (b + 4), "flops": 4 * d * pairs}
    if kind == "norm":
        r, d = case["rows"], case["dim"]
        return {"bytes": r * d * (13 if case["op"] == "residual" else 25) + 4 * r + 8 * d, "flops": 10 * r * d}
    if kind == "vocab":
        m, k, v = case["m"], case["k"], case["v"]
        return {"bytes": v * (k + 8) + m * (k + 8) + (4 * m * v if case["logits"] else 0), "flops": 2 * m * k * v}
    if kind == "candidates":
        m, k, c = case["m"], case["k"], int(_cand_counts(case).sum())
        return {"bytes": min(c, case["v"]) * (k + 8) + 8 * c + m * (k + 8), "flops": 2 * c * k}
    # Every weight and every output once; every token's products, attention over its own keys.
    ssru = case["graph"] == "ssru"
    d, f, enc, dec = (384, 1536, 6, 4) if ssru else (512, 2048, 6, 2)
    b = _batch(case)
    src, gen = b.lengths, b.max_output_tokens.astype(np.int64)
    layer = 4 * d * d + 2 * d * f
    cross = 2 * d * d
    step = ((2 * d * d if ssru else 4 * d * d) + 2 * d * d + 2 * d * f) * dec + d * _VOCAB
    flops = 2 * int(src.sum()) * (layer * enc + cross * dec) + 2 * int(gen.sum()) * step
    flops += 4 * d * (int((src ** 2).sum()) * enc + int((src * gen).sum()) * dec)
    if not ssru:
        flops += 2 * d * int((gen * (gen + 1)).sum()) * dec
    weights = layer * enc + cross * dec + step + (d * _VOCAB if ssru else 0)
    return {"bytes": weights + 4 * int(src.sum()) * (d + 1) + 4 * len(src) * _VOCAB + 4 * int(gen.sum()), "flops": flops}


def tolerance(case):
    """About four times what exact() shows (relative 2-norm): dequantized products 5e-8, attention up to
    5e-7 (512 keys), norms 1.7e-7."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 2e-7}
    if kind == "attention":
        return {"rel": 2e-6}
    if kind == "norm":  # a last-bit difference can move a quantized value by one step
        return {"rel": 8e-7, "differ": 1e-4}
    if kind in ("vocab", "candidates"):
        return {"rel": 2e-7, "differ": 0.0}
    # A reordered sum that crosses an int8 rounding boundary moves an activation by a whole step: up to
    # 5.7e-3 on the logits with another summation order in the decoder.
    return {"rel": 2e-2, "differ": 0.01}


# ---------------------------------------------------------------------------
# The same results in 64 bits
# ---------------------------------------------------------------------------
def _linear64(q, a, w, mult, bias, relu=False):
    """y = acc / (a w) + b in 64 bits; the integers are the definition of the quantized layer."""
    acc = q.double() @ w.double().T
    y = acc / (a.double()[:, None] * mult.double()[None, :]) + bias.double()
    return acc, y.clamp_min(0.0) if relu else y


def _attend64(q, k, v, heads):
    n, d = q.shape
    dh = d // heads
    split = lambda t: t.double().reshape(t.shape[0], heads, dh).transpose(0, 1).contiguous()  # noqa: E731
    s = torch.matmul(split(q), split(k).transpose(1, 2).contiguous()) / math.sqrt(dh)
    return torch.matmul(torch.softmax(s, dim=-1), split(v)).transpose(0, 1).reshape(n, d)


def _norm64(z, scale, bias):
    z = z.double()
    mean = z.mean(dim=-1, keepdim=True)
    var = ((z - mean) ** 2).mean(dim=-1, keepdim=True)
    return (z - mean) / torch.sqrt(var + 1e-6) * scale.double() + bias.double()


def _encoder64(model, tokens, offsets):
    """Encoder states of the transformer graph, quantized as the layers define it, the rest in 64 bits."""
    g = model.geometry
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(_DEV)  # noqa: E731
    half = g.dim // 2
    f = torch.exp(-torch.arange(half, device=_DEV, dtype=torch.float64) * math.log(10000.0) / (half - 1))
    offs = [int(o) for o in offsets]
    p = torch.cat([torch.arange(b - a, device=_DEV) for a, b in zip(offs, offs[1:])]).double()[:, None] * f[None, :]
    tok = to(tokens.astype(np.int64))
    x = to(model.embedding)[tok].double() / to(model.embedding_mult)[tok].double()[:, None] * math.sqrt(g.dim)
    x = x + torch.cat([torch.sin(p), torch.cos(p)], dim=1)

    def dense(t, lin, relu=False):
        m = t.abs().amax(dim=1)
        a = torch.where(m > 0, 127.0 / torch.where(m > 0, m, torch.ones_like(m)), torch.ones_like(m))
        q = torch.clamp(torch.round(t * a[:, None]), -127, 127)
        return _linear64(q, a, to(lin["weight"]), to(lin["mult"]), to(lin["bias"]), relu)[1]

    for layer in model.encoder:
        qkv = dense(x, layer["qkv"])
        q, k, v = qkv[:, :g.dim], qkv[:, g.dim:2 * g.dim], qkv[:, 2 * g.dim:]
        att = torch.cat([_attend64(q[a:b], k[a:b], v[a:b], g.heads) for a, b in zip(offs, offs[1:])])
        x = _norm64(dense(att, layer["out"]) + x, to(layer["ln1"]["scale"]), to(layer["ln1"]["bias"]))
        y = dense(dense(x, layer["ffn1"], relu=True), layer["ffn2"])
        x = _norm64(y + x, to(layer["ln2"]["scale"]), to(layer["ln2"]["bias"]))
    return x


def exact(case, seed):
    got, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        if case["act"] == "static":
            a = torch.full((case["m"],), _STATIC_MULT, device=_DEV, dtype=torch.float32)
        else:
            a = got["a"] if case["act"] == "quantized" else _row_multiplier(got["x"])
        q = got["q"] if case["act"] == "quantized" else _quantize(got["x"], a)
        acc, y = _linear64(q, a, got["w"], got["mult"], got["bias"], case["relu"])
        return dict(out=y, acc=acc.to(torch.int32)) if case["i32"] else y
    if kind == "attention":
        cu = [int(c) for c in got["cu"].cpu()]
        rows = [slice(i, i + 1) if case["cross"] else slice(cu[i], cu[i + 1]) for i in range(len(cu) - 1)]
        return torch.cat([_attend64(got["q"][r], got["k"][a:b], got["v"][a:b], case["heads"])
                          for r, a, b in zip(rows, cu, cu[1:])])
    if kind == "norm":
        state = None
        if case["op"] == "ssru":
            gate = torch.sigmoid(got["forget"].double())
            state = gate * got["state"].double() + (1.0 - gate) * got["x"].double()
            out = _norm64(state.clamp_min(0.0) + got["r"].double(), got["scale"], got["bias"])
        else:
            out = _norm64(got["x"].double() + got["r"].double(), got["scale"], got["bias"])
        got = dict(out=out, q=None, a=127.0 / out.abs().amax(dim=1))
        return dict(got, state=state) if case["op"] == "ssru" else got
    if kind == "vocab":
        if not case["logits"]:
            return None
        _, y = _linear64(got["q"], got["a"], got["emb"], got["mult"], got["bias"])
        y[:, 1] = -math.inf
        y[:, 7:39] = -math.inf
        return dict(token=None, logits=y)
    if kind == "candidates":
        _, y = _linear64(got["q"], got["a"], got["emb"], got["mult"], got["bias"])
        off = [int(o) for o in got["off"].cpu()]
        cand = got["cand"].long()
        return dict(token=None, logits=torch.cat([y[i, cand[a:b]] for i, (a, b) in enumerate(zip(off, off[1:]))]))
    if case["graph"] != "transformer":
        return None
    # The decoder's logits follow from the tokens chosen before them, which 64 bits may choose otherwise.
    enc = _encoder64(_engine("transformer")[1], got["tokens"], got["batch"].offsets)
    return dict(tokens=None, offsets=None, encoder=enc, logits=None, active=None)

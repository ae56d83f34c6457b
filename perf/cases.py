"""The work a program has this library do, as cases that can be timed and checked.

One pass is one MoE feed-forward (or a few, one per transformer block) through the
public Python entry points: MoELayer.forward / forward_norm (with the RMSNorm partial
sums carried or not) and GeGLUMoELayer.forward_gemma4, over the layer shapes of this
repository's workloads, one to 4096 tokens, Q4_0 and Q8_0 experts, with and without the
chunk-major weight copies.

A case:
  model   one of MODELS
  tokens  rows of the call
  blocks  layers run by one pass, each on rows of its own (attention sits between them in
          a model); the decode cases run several so that a pass reads weights that are
          not in a cache, as a whole model does
  entry   "forward" (y = MoE(x)), "residual" (y = x + MoE(x)), "norm" (y = x +
          MoE(RMSNorm(x) w)), "chain" (the same with x's partial sums handed over and y's
          returned), "gemma4" (the Gemma 4 branch from the residual rows)
  copies  the layers keep chunk-major copies of their experts (the constructors' opt-in;
          off by default)
  graph   the pass is a replay of a HIP graph captured once, as a serving loop runs its
          decode step; otherwise the calls are made one by one
"""
import math

import numpy as np
import torch

from qwenium_amd import TYPE_Q4_0, TYPE_Q8_0, Workspace, synthetic
from qwenium_amd.moe import rms_partials

EPS = synthetic.NORM_EPS

MODELS = {
    "35b-q4": synthetic.QWEN35B,            # hidden 2048, 256 experts, top-8 + shared, ffn 512
    "35b-q8": synthetic.QWEN35B_Q8,
    "35b-skew": synthetic.QWEN35B_SKEW,     # Q8_0, half of the assignments on 8 experts, 40 without any
    "gemma4-q4": synthetic.GEMMA4,          # hidden 2816, 128 experts, top-8, ffn 704, GeGLU
    "gemma4-q8": synthetic.GEMMA4_Q8,
    "small-q8": synthetic.CONFIG1,          # hidden 1024, 16 experts, top-2, ffn 512
    # generic shapes beside the named ones
    "wide-q4": synthetic.LayerSpec(4096, 32, 4, 1024, False, TYPE_Q4_0),
    "mid-q4": synthetic.LayerSpec(1536, 64, 6, 768, True, TYPE_Q4_0),
    "many-q8": synthetic.LayerSpec(1024, 512, 10, 256, True, TYPE_Q8_0),
}


def _case(name, model, tokens, entry, blocks=1, copies=False, graph=False):
    return {"name": name, "model": model, "tokens": tokens, "blocks": blocks, "entry": entry, "copies": copies,
            "graph": graph}


def listed():
    return [
        # one user's decode step: every launch waits for the one before it
        _case("decode 1", "35b-q4", 1, "norm", blocks=8, graph=True),
        # ten users' decode step (the benchmark's headline batch)
        _case("decode 10", "35b-q4", 10, "forward", blocks=4, graph=True),
        # a full decode batch in the larger weight type, partial sums carried from block to block
        _case("decode 16 q8", "35b-q8", 16, "chain", blocks=2, graph=True),
        # decode of the GeGLU model
        _case("gemma4 decode 5", "gemma4-q4", 5, "gemma4", blocks=4, graph=True),
        # a small model's short prompt, called directly: launches and host time count
        _case("small 32", "small-q8", 32, "forward"),
        # a large decode batch, or speculative decoding
        _case("batch 64", "35b-q4", 64, "norm"),
        # a short prompt over weights as a GGUF file has them
        _case("prompt 211", "35b-q4", 211, "norm"),
        # a chunk of a prompt in a chunked prefill, Q8_0
        _case("chunk 512 q8", "35b-q8", 512, "residual", copies=True),
        # a prompt of ordinary length over the GGUF weights
        _case("prompt 1000", "35b-q4", 1000, "norm"),
        # a prompt on the GeGLU model
        _case("gemma4 prompt 1500", "gemma4-q4", 1500, "gemma4", copies=True),
        # routing as unbalanced as trained models show it
        _case("skewed 2048 q8", "35b-skew", 2048, "forward", copies=True),
        # a long prompt (the benchmark's prefill)
        _case("prefill 4096", "35b-q4", 4096, "forward", copies=True),
    ]


# the most tokens of a drawn case: its work stays below the largest listed case's
MOST_TOKENS = {"35b-q4": 3800, "35b-q8": 3200, "35b-skew": 3000, "gemma4-q4": 2300, "gemma4-q8": 2000, "small-q8": 4096,
               "wide-q4": 2500, "mid-q4": 3600, "many-q8": 3000}


def draw(rng):
    model = rng.choice(["35b-q4", "35b-q4", "35b-q8", "35b-skew", "gemma4-q4", "gemma4-q8", "small-q8", "wide-q4",
                        "mid-q4", "many-q8"])
    tokens = int(round(math.exp(rng.uniform(0.0, math.log(MOST_TOKENS[model])))))
    graph = tokens <= 16
    blocks = rng.choice([2, 3, 4]) if graph else 1
    if MODELS[model].geglu:
        entry = "gemma4"
    elif model == "35b-skew":
        entry = "forward"
    else:
        entry = rng.choice(["forward", "residual", "norm", "chain"])
    c = _case("", model, tokens, entry, blocks, rng.random() < 0.5, graph)
    del c["name"]
    return c


def _weights(case, seed, block):
    return synthetic.make_layer_tensors(MODELS[case["model"]], seed, layer=block)


def _inputs(case, seed, block):
    """The rows of one block and its norm weights."""
    spec = MODELS[case["model"]]
    x = synthetic.make_x(spec, case["tokens"], seed, batch=block)
    if case["entry"] == "gemma4":
        return x, synthetic.make_gemma4_norms(spec, seed, block)
    if case["entry"] in ("norm", "chain"):
        return x, (synthetic.make_norm_weight(spec, seed, block),)
    return x, ()


def _block(case, layer, ws, x, norms, x_ssq, out, y_ssq):
    entry = case["entry"]
    if entry == "gemma4":
        return layer.forward_gemma4(x, norms[0], norms[1], EPS, out=out, workspace=ws)
    if entry == "norm":
        return layer.forward_norm(x, norms[0], EPS, out=out, workspace=ws)
    if entry == "chain":
        return layer.forward_norm(x, norms[0], EPS, out=out, workspace=ws, x_ssq=x_ssq, y_ssq=y_ssq)
    return layer.forward(x, residual=x if entry == "residual" else None, out=out, workspace=ws)


def prepare(case, seed):
    """Layers over seeded weights, one workspace, the rows; for a graph case the captured step."""
    spec = MODELS[case["model"]]
    st = {"case": case, "blocks": [], "graph": None}
    for b in range(case["blocks"]):
        layer = synthetic.make_layer(spec, seed, layer=b, tensors=_weights(case, seed, b),
                                     prefill_copies=case["copies"])
        x, norms = _inputs(case, seed, b)
        x_ssq = rms_partials(x) if case["entry"] == "chain" else None
        y_ssq = torch.empty_like(x_ssq) if x_ssq is not None else None
        st["blocks"].append((layer, x, norms, x_ssq, y_ssq))
    st["ws"] = Workspace(st["blocks"][0][0], case["tokens"])
    if case["graph"]:
        st["out"] = [torch.empty_like(x) for _, x, _, _, _ in st["blocks"]]
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _step(st, st["out"])
        torch.cuda.current_stream().wait_stream(stream)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            _step(st, st["out"])
    return st


def _step(st, out):
    return [_block(st["case"], layer, st["ws"], x, norms, x_ssq, out[i] if out else None, y_ssq)
            for i, (layer, x, norms, x_ssq, y_ssq) in enumerate(st["blocks"])]


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        ys = state["out"]
    else:
        ys = _step(state, None)
    if state["case"]["entry"] == "chain":
        return {"y": ys, "y_ssq": [b[4] for b in state["blocks"]]}
    return {"y": ys}


def _row_bytes(spec, n):
    return n // 32 * (18 if spec.wtype == TYPE_Q4_0 else 34)


def work(case):
    """Every expert that tokens reach read once, the router, the rows in and out; the
    products of the router and of the chosen experts."""
    spec, T = MODELS[case["model"]], case["tokens"]
    H, E, K, F, S = spec.n_embd, spec.n_experts, spec.top_k, spec.ffn_dim, int(spec.shared)
    live = E - spec.skew.n_empty if spec.skew is not None else E
    distinct = live * (1.0 - (1.0 - K / live) ** T)
    expert = 2 * F * _row_bytes(spec, H) + H * _row_bytes(spec, F)
    nbytes = (distinct + S) * expert + (E + S) * H * 4 + 2 * T * H * 4
    flops = 2.0 * T * (K + S) * 3 * H * F + 2.0 * T * (E + S) * H
    return {"bytes": case["blocks"] * nbytes, "flops": case["blocks"] * flops}


def tolerance(case):
    """Rows of 32-bit values whose products are summed exactly or in 32 bits, between
    quantizations (of x and of h) that every correct implementation rounds alike."""
    return {"rel": 2e-6, "max": 4e-5}


# ---------------------------------------------------------------------------
# The same pass in 64 bits
# ---------------------------------------------------------------------------
def _dequant(data, wtype, rows, cols):
    """GGUF block rows as float64 [rows, cols]."""
    nb = cols // 32
    if wtype == TYPE_Q8_0:
        b = data.view(rows, nb, 34)
        d = b[..., :2].contiguous().view(torch.float16).double()
        return (b[..., 2:].contiguous().view(torch.int8).double() * d).view(rows, cols)
    b = data.view(rows, nb, 18)
    d = b[..., :2].contiguous().view(torch.float16).double()
    q = b[..., 2:]
    q = torch.cat([q & 15, q >> 4], dim=-1).double() - 8.0
    return (q * d).view(rows, cols)


def _q8_0(v):
    """The values that Q8_0 activations stand for (the format's own rounding, of float32
    rows: scale fp16(amax / 127), quants rint(v * (127 / amax)) in float32), in float64."""
    t = v.float().view(v.shape[0], -1, 32)
    amax = t.abs().amax(dim=-1, keepdim=True)
    d = (amax.double() / 127.0).float().half().double()
    inv = torch.where(amax > 0, 127.0 / amax.double(), torch.zeros_like(amax, dtype=torch.float64)).float()
    return (torch.round(t * inv).double() * d).view(v.shape)


def _gelu(g):
    """gelu through the table that defines it: fp16 values of a float32 formula over fp16 arguments."""
    one = np.float32(1.0)
    a = np.arange(65536, dtype=np.uint16).view(np.float16).astype(np.float32)
    with np.errstate(all="ignore"):
        z = np.float32(math.sqrt(2.0 / math.pi)) * a * (one + np.float32(0.044715) * a * a)
        table = (np.float32(0.5) * a * (one + np.tanh(z.astype(np.float64)).astype(np.float32))).astype(np.float16)
    t = torch.from_numpy(table).to(g.device)[g.half().view(torch.int16).long() & 0xffff].double()
    g = g.double()
    return torch.where(g <= -10.0, torch.zeros_like(g), torch.where(g >= 10.0, g, t))


def _expert(spec, xq, wg, wu, wd):
    g, u = (xq @ wg.T).float(), (xq @ wu.T).float()  # the activation's float32 arguments
    if spec.geglu:
        h = (_gelu(g).float() * u).double()
    else:
        g = g.double()
        h = (g / (1.0 + torch.exp(-g)) * u.double()).float().double()
    return _q8_0(h) @ wd.T


def _exact_block(case, seed, block):
    spec = MODELS[case["model"]]
    H, E, K, F, wt = spec.n_embd, spec.n_experts, spec.top_k, spec.ffn_dim, spec.wtype
    t = _weights(case, seed, block)
    x, norms = _inputs(case, seed, block)
    xin = xr = x
    if norms:
        mean = (x * x).double().mean(dim=1, keepdim=True).float()
        scale = (1.0 / torch.sqrt((mean + EPS).double()).float().double()).float()
        xin = xr = (x * scale) * norms[0]
        if case["entry"] == "gemma4":
            s = (1.0 / torch.tensor(float(H), device=x.device).double().sqrt().float().double()).float()
            xr = ((x * scale) * s) * norms[1]
    logits = (xr.double() @ t["router"].data.view(E, H).double().T).float()
    val, idx = torch.sort(logits, dim=1, descending=True, stable=True)
    val, idx = val[:, :K].double(), idx[:, :K]
    w = torch.softmax(val, dim=1)
    xq = _q8_0(xin)
    if spec.geglu:
        gu = t["gate_up"].data.view(E, -1)
        gate, up = gu[:, :gu.shape[1] // 2], gu[:, gu.shape[1] // 2:]
    else:
        gate, up = t["gate"].data.view(E, -1), t["up"].data.view(E, -1)
    down = t["down"].data.view(E, -1)
    y = torch.zeros((x.shape[0], H), dtype=torch.float64, device=x.device)
    order = torch.argsort(idx.reshape(-1), stable=True)
    counts = torch.bincount(idx.reshape(-1), minlength=E).tolist()
    at = 0
    for e in range(E):
        if not counts[e]:
            continue
        a = order[at:at + counts[e]]
        at += counts[e]
        tok = a // K
        ye = _expert(spec, xq[tok], _dequant(gate[e].contiguous(), wt, F, H), _dequant(up[e].contiguous(), wt, F, H),
                     _dequant(down[e].contiguous(), wt, H, F))
        y.index_add_(0, tok, ye * w.reshape(-1)[a][:, None])
    if spec.shared:
        ys = _expert(spec, xq, _dequant(t["sh_gate"].data, wt, F, H), _dequant(t["sh_up"].data, wt, F, H),
                     _dequant(t["sh_down"].data, wt, H, F))
        sg = (xr.double() @ t["sh_norm"].data.double()).float().double()
        y += ys * torch.sigmoid(sg)[:, None]
    if case["entry"] in ("residual", "norm", "chain"):
        y += x.double()
    return y


def exact(case, seed):
    """The same rows from float64 products and sums.  Where the layer is defined by a
    rounding (Q8_0 of x and of h from float32 values, the logits that select, the fp16
    gelu table), that rounding is part of the value."""
    ys = [_exact_block(case, seed, b) for b in range(case["blocks"])]
    if case["entry"] != "chain":
        return {"y": ys}
    return {"y": ys, "y_ssq": [(y * y).view(y.shape[0], -1, 32).sum(-1) for y in ys]}

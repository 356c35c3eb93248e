"""What is timed to say whether the library got faster: passes through its public entry points as programs call them.

listed() names the cases; draw() gives more of the same ranges; prepare() builds what a program holds before the call
(compressed matrices, inputs, a captured graph where it decodes under one); run() makes one pass; work() says what a
pass cannot do without; exact() is the same pass in float64 without this library.

Kinds of case:
  linear  one NWCLinear on `tokens` vectors
  layers  the four projections (fused qkv, output, fused gate and up, down) of `layers` decoder layers, each layer with
          its own weights in memory, on `tokens` vectors; with `graph` captured once and replayed, as a decoding
          program does with its token step
  mlp     a gate / up / down block put through fuse() and convert(), called as a module
  embed   NWCEmbedding on `ids` token ids
  encode  a BF16 matrix in host memory compressed and placed on the GPU, down to the tensors a checkpoint keeps

Weights are N(0, 0.02^2) in BF16, activations N(0, 1).
"""
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

import nwc_amd as nwc

DEVICE = "cuda"
WEIGHT_STD = 0.02


def listed():
    return [
        # the smallest call: one token through a 0.6B model's output projection, called eagerly; launch latency and
        # the host's way to the kernel are all of it
        dict(name="token_small", kind="linear", elem="bf16", layout=0, rows=1024, cols=2048, tokens=1, bias=False),
        # batch-1 decoding of a 4B model, the library's headline use: one token through three layers' projections
        dict(name="token_layers_bf16", kind="layers", elem="bf16", layout=0, hidden=2560, qkv=6144, attn=4096, ffn=9728,
             layers=3, tokens=1, graph=True),
        # the same with weight-only fp8
        dict(name="token_layers_fp8", kind="layers", elem="fp8", layout=0, hidden=2560, qkv=6144, attn=4096, ffn=9728,
             layers=4, tokens=1, graph=True),
        # batch-1 decoding of a 7B model in the fixed-width layout
        dict(name="token_layers_fixed", kind="layers", elem="bf16", layout=2, hidden=3584, qkv=4608, attn=3584,
             ffn=18944, layers=2, tokens=1, graph=True),
        # the vocabulary projection of a decoding step: the logits of one token, the largest matrix of a model
        dict(name="head_logits", kind="linear", elem="bf16", layout=0, rows=151936, cols=2560, tokens=1, bias=False),
        # a projection of no round size, with a bias, in the fragment-order layout
        dict(name="token_ragged", kind="linear", elem="bf16", layout=1, rows=9001, cols=3333, tokens=1, bias=True),
        # a few tokens at once, a draft being checked or a few users: one layer's projections for four vectors
        dict(name="few_tokens", kind="layers", elem="bf16", layout=1, hidden=2560, qkv=6144, attn=4096, ffn=9728,
             layers=1, tokens=4, graph=False),
        # a small serving batch through an MLP block that fuse() and convert() built
        dict(name="batch_mlp", kind="mlp", elem="bf16", hidden=2560, ffn=9728, tokens=32),
        # a small batch on a ragged fixed-width fp8 matrix with a bias
        dict(name="batch_fixed_fp8", kind="linear", elem="fp8", layout=2, rows=4999, cols=3590, tokens=11, bias=True),
        # a prompt of 512 tokens through one layer's projections
        dict(name="prefill", kind="layers", elem="bf16", layout=0, hidden=2560, qkv=6144, attn=4096, ffn=9728, layers=1,
             tokens=512, graph=False),
        # the embedding lookup of a prompt
        dict(name="embed_prompt", kind="embed", elem="bf16", layout=0, rows=151936, cols=2560, ids=512),
        # converting one projection of a model that was loaded into host memory
        dict(name="encode", kind="encode", elem="bf16", layout=0, rows=2560, cols=9728),
    ]


MAX_WEIGHTS = 50_000_000            # of a drawn matrix: about the largest projection listed; the head is larger


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choices(["token", "few", "batch", "prompt", "embed", "encode"], [6, 3, 4, 2, 2, 2])[0]
    rows, cols = _log_int(rng, 256, 38000), _log_int(rng, 256, 19000)
    rows = max(256, min(rows, MAX_WEIGHTS // cols))
    if rng.random() < 0.5:                       # half of the matrices have round sizes, as most models' do
        rows, cols = max(256, rows // 128 * 128), max(256, cols // 128 * 128)
    case = dict(kind="linear", elem=rng.choice(["bf16", "bf16", "fp8"]), layout=rng.choice([0, 0, 1, 2]), rows=rows,
                cols=cols)
    if kind == "embed":
        return dict(case, kind="embed", ids=_log_int(rng, 1, 2048))
    if kind == "encode":
        return dict(case, kind="encode")
    low, high = {"token": (1, 1), "few": (2, 8), "batch": (9, 64), "prompt": (65, 1024)}[kind]
    return dict(case, tokens=_log_int(rng, low, high), bias=rng.random() < 0.3)


# ---- inputs ----

def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _matrix(g, rows, cols):
    return (torch.randn(rows, cols, generator=g, device=DEVICE) * WEIGHT_STD).bfloat16()


def _vectors(g, tokens, cols):
    return torch.randn(tokens, cols, generator=g, device=DEVICE).bfloat16()


def _projections(case):
    """(rows, columns) of the matrices of one pass, in order."""
    if case["kind"] == "layers":
        one = [(case["qkv"], case["hidden"]), (case["hidden"], case["attn"]), (2 * case["ffn"], case["hidden"]),
               (case["hidden"], case["ffn"])]
        return one * case["layers"]
    if case["kind"] == "mlp":
        return [(2 * case["ffn"], case["hidden"]), (case["hidden"], case["ffn"])]
    return [(case["rows"], case["cols"])]


def _linear_inputs(case, seed):
    """Yields (weight, bias or None, x) of each product, from the seed alone."""
    g = _gen(seed)
    for rows, cols in _projections(case):
        w = _matrix(g, rows, cols)
        bias = _vectors(g, 1, rows).view(-1) if case.get("bias") else None
        yield w, bias, _vectors(g, case["tokens"], cols)


class Mlp(nn.Module):
    def __init__(self, hidden, ffn, g):
        super().__init__()
        for name, rows, cols in (("gate_proj", ffn, hidden), ("up_proj", ffn, hidden), ("down_proj", hidden, ffn)):
            lin = nn.Linear(cols, rows, bias=False, device="meta", dtype=torch.bfloat16)
            lin.weight = nn.Parameter(_matrix(g, rows, cols), requires_grad=False)
            setattr(self, name, lin)

    def forward(self, x):
        return self.down_proj(F.silu(self.gate_proj(x)) * self.up_proj(x))


def _encode_source(case, seed):
    return _matrix(_gen(seed), case["rows"], case["cols"]).cpu()


def _stream_capacity(case):
    """Four bits per weight of the matrix padded to whole 16 x 512 blocks, which these weights' streams stay under."""
    return -(-case["rows"] // 16) * 16 * (-(-case["cols"] // 512) * 512) // 2 + 4096


def _ids(case, g):
    return torch.randint(0, case["rows"], (case["ids"],), generator=g, device=DEVICE)


# ---- what a program holds before the call ----

def prepare(case, seed):
    kind = case["kind"]
    if kind == "encode":
        return {"case": case, "source": _encode_source(case, seed)}
    if kind == "embed":
        g = _gen(seed)
        table = nwc.NWCWeight(_matrix(g, case["rows"], case["cols"]), DEVICE, elem=case["elem"], layout=case["layout"])
        return {"case": case, "module": nwc.NWCEmbedding(w=table), "ids": _ids(case, g)}
    if kind == "mlp":
        g = _gen(seed)
        model = Mlp(case["hidden"], case["ffn"], g)
        x = _vectors(g, case["tokens"], case["hidden"])
        nwc.fuse(model, device=DEVICE, elem=case["elem"])
        nwc.convert(model, device=DEVICE, verbose=False, elem=case["elem"])
        return {"case": case, "module": model, "x": x}
    steps = []
    for w, bias, x in _linear_inputs(case, seed):
        held = nwc.NWCWeight(w, DEVICE, elem=case["elem"], layout=case["layout"])
        steps.append((nwc.NWCLinear(w=held, bias=bias, device=DEVICE), x))
    state = {"case": case, "steps": steps}
    if case.get("graph"):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                for lin, x in steps:
                    lin(x)
        torch.cuda.current_stream().wait_stream(side)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = [lin(x) for lin, x in steps]
    return state


# ---- one pass ----

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "encode":
        stored = nwc.NWCWeight(state["source"], DEVICE, elem=case["elem"], layout=case["layout"]).tensors()
        # the streams' length depends on the weights; a reader of several such matrices keeps them in equal buffers
        stored["data"] = F.pad(stored["data"], (0, _stream_capacity(case) - stored["data"].numel()))
        return stored
    if kind == "embed":
        return state["module"](state["ids"])
    if kind == "mlp":
        return state["module"](state["x"])
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return [lin(x) for lin, x in state["steps"]]


# ---- what a pass cannot do without ----

def _bytes_per_weight(case):
    """Compressed bytes per weight for N(0, 0.02^2): raw byte + code bits (about 2.72), or nibble codes (layout 2)."""
    if case.get("layout") == 2:
        return 1.5 if case["elem"] == "bf16" else 0.875
    return 1.37 if case["elem"] == "bf16" else 0.875


def work(case):
    kind = case["kind"]
    per = _bytes_per_weight(case)
    if kind == "encode":
        n = case["rows"] * case["cols"]
        return {"bytes": (2 + per) * n, "flops": 0}
    if kind == "embed":
        return {"bytes": (2 + per) * case["ids"] * case["cols"] + 8 * case["ids"], "flops": 0}
    tokens, total, flops = case["tokens"], 0.0, 0.0
    for rows, cols in _projections(case):
        total += per * rows * cols + 2 * tokens * (rows + cols)
        flops += 2.0 * tokens * rows * cols
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Lookups and encoded tensors are exact (a scaled fp8 row is one product in fp32, rounded once).  Products have
    fp32 sums rounded to BF16: about 1.7e-3 off float64 by the rounding alone, 2.1e-3 where fp8 rounds twice (the
    unscaled product, then the scaled one), 3.9e-3 after a block's second rounding; four times that.  The largest single
    difference is two BF16 steps of the value."""
    if case["kind"] in ("encode", "embed"):
        return "exact"
    rel = 0.0156 if case["kind"] == "mlp" else 0.0084 if case["elem"] == "fp8" else 0.0068
    return {"rel": rel, "max": 0.03}


# ---- the same pass in float64 ----

def _weights64(w, elem):
    if elem == "bf16":
        return w.double()
    wf = w.float()
    amax = wf.abs().amax(dim=1).clamp_min(1e-12)
    scale = amax / torch.full_like(amax, 448.0)
    codes = torch.clamp(wf / scale.unsqueeze(1), min=-448.0, max=448.0).to(torch.float8_e4m3fn)
    return codes.float().double() * scale.double().unsqueeze(1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "encode":
        return None
    if kind == "embed":
        g = _gen(seed)
        w = _matrix(g, case["rows"], case["cols"])
        ids = _ids(case, g)
        if case["elem"] == "bf16":
            return w[ids].double()
        return _weights64(w, "fp8")[ids]
    if kind == "mlp":
        g = _gen(seed)
        gate, up, down = (_matrix(g, r, c).double() for r, c in ((case["ffn"], case["hidden"]), (case["ffn"], case["hidden"]),
                                                                (case["hidden"], case["ffn"])))
        x = _vectors(g, case["tokens"], case["hidden"]).double()
        return (F.silu(x @ gate.T) * (x @ up.T)) @ down.T
    out = []
    for w, bias, x in _linear_inputs(case, seed):
        y = x.double() @ _weights64(w, case["elem"]).T
        out.append(y if bias is None else y + bias.double())
    return out

"""The work a user of this engine has it do: EXL3 linear modules of a decoder, driven through the
plugin's linear method (create_weights, weight loaders, process_weights_after_loading, apply,
apply_silu_mul) or the torch ops, from one decode token to a 2048-token prefill chunk.

A case names modules and a row count:
  part    "linear" (one checkpoint tensor), "qkv" (a fused module of three tensors), "mlp" (gate/up
          module, then the down module on its SiLU-and-mul), or "layer" (qkv, o, then the MLP)
  m       rows of the batch: decode tokens or prefill tokens
  k, n    the hidden width and, for a linear, the output width; q and kv: the widths of a qkv
          module's tensors; inter: an MLP's intermediate width
  bits, kv_bits, book   bits per weight (kv_bits: of a qkv module's k and v) and codebook
  graph   the pass is one replay of a HIP graph captured from the eager calls, as a server replays
          its decode step; otherwise the calls themselves
Modules of a layer take inputs of their own (the attention and the norms between them are not this
engine's); the down module takes the gate/up module's output, as in the model.
"""
import math
import os
import sys

import numpy as np
import torch

_REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_REPO, "qwen38-27b-exl3-rdna4_amd"))

H, I, KV = 5120, 17408, 1024          # hidden, intermediate and k / v widths of the 27B decoder
HEAD = 248320                         # its vocabulary


def listed():
    return [
        # the smallest call: one k projection for one token, called eagerly (no graph: a server run
        # with eager execution, a debugger, a draft head): latency of the call and of one launch
        dict(name="k_proj_m1_eager", part="linear", m=1, k=H, n=KV, bits=5, book="mul1", graph=False),
        # single-stream decode: all seven linears of a decoder layer on one token
        dict(name="layer_m1", part="layer", m=1, k=H, q=H, kv=KV, inter=I, bits=4, kv_bits=4, book="mul1", graph=True),
        # the logits of one token
        dict(name="lm_head_m1", part="linear", m=1, k=H, n=HEAD, bits=4, book="mul1", graph=True),
        # a small server batch (or the draft tokens of speculative decoding) through an MLP
        dict(name="mlp_m8", part="mlp", m=8, k=H, inter=I, bits=3, book="mul1", graph=True),
        # a generic square layer of another model, mcg codebook, a few rows
        dict(name="square_m13", part="linear", m=13, k=4096, n=4096, bits=6, book="mcg", graph=True),
        # continuous batching: 32, 48 and 96 sequences decoded together
        dict(name="layer_m32", part="layer", m=32, k=H, q=H, kv=KV, inter=I, bits=4, kv_bits=4, book="mul1", graph=True),
        # the checkpoint's mixed-bitrate attention module (2-bit q and gate, 5-bit k and v)
        dict(name="qkv_mixed_m48", part="qkv", m=48, k=H, q=12288, kv=KV, bits=2, kv_bits=5, book="mul1", graph=True),
        dict(name="mlp_m96", part="mlp", m=96, k=H, inter=I, bits=4, book="mul1", graph=True),
        # short prompts and the last chunk of longer ones: ragged prefills
        dict(name="gdn_out_m200", part="linear", m=200, k=6144, n=H, bits=4, book="3inst", graph=False),
        dict(name="mlp_m515", part="mlp", m=515, k=H, inter=I, bits=3, book="mul1", graph=False),
        # prefill chunks: the linear-attention input projection alone, and a whole layer
        dict(name="gdn_qkv_m1024", part="linear", m=1024, k=H, n=10240, bits=2, book="mul1", graph=False),
        dict(name="layer_m2048", part="layer", m=2048, k=H, q=H, kv=KV, inter=I, bits=4, kv_bits=4, book="mul1", graph=False),
    ]


def draw(rng):
    part = rng.choice(["linear", "linear", "qkv", "mlp", "mlp", "layer"])
    m = int(round(math.exp(rng.uniform(0.0, math.log(2048.0)))))
    c = dict(part=part, m=m)
    if part == "linear":
        if rng.random() < 0.6:        # the checkpoint's modules
            c["k"], c["n"] = rng.choice([(H, H), (H, KV), (H, 6144), (H, 10240), (H, 12288), (H, I), (6144, H), (I, H)])
        else:                         # any model's: multiples of 128
            c["k"], c["n"] = (128 * int(round(math.exp(rng.uniform(math.log(4.0), math.log(136.0))))) for _ in range(2))
    else:
        c["k"] = rng.choice([H, H, H, 4096, 2048, 128 * rng.randint(6, 40)])
        if part in ("qkv", "layer"):
            c["q"], c["kv"] = (rng.choice([H, 12288]), KV) if c["k"] == H else (c["k"], 128 * rng.randint(1, 8))
        if part in ("mlp", "layer"):
            c["inter"] = I if c["k"] == H else 128 * rng.randint(c["k"] // 128, 3 * c["k"] // 128)
    c["bits"] = rng.choice([1, 2, 2, 3, 3, 4, 4, 4, 4, 5, 6, 7, 8])
    if part in ("qkv", "layer"):
        c["kv_bits"] = rng.choice([c["bits"], c["bits"], 5, 6])
    c["book"] = rng.choice(["mul1", "mul1", "mul1", "mcg", "3inst"])
    c["graph"] = m <= 128 and rng.random() < 0.85
    return c


# ---------------------------------------------------------------------------------------------
# modules, inputs
# ---------------------------------------------------------------------------------------------
def _modules(c):
    """[(name, k, [(n, bits), ...])] in call order."""
    b = c["bits"]
    if c["part"] == "linear":
        return [("lin", c["k"], [(c["n"], b)])]
    out = []
    if c["part"] in ("qkv", "layer"):
        out.append(("qkv", c["k"], [(c["q"], b), (c["kv"], c["kv_bits"]), (c["kv"], c["kv_bits"])]))
    if c["part"] == "layer":
        out.append(("o", c["q"], [(c["k"], b)]))
    if c["part"] in ("mlp", "layer"):
        out.append(("gate_up", c["k"], [(c["inter"], b), (c["inter"], b)]))
        out.append(("down", c["inter"], [(c["k"], b)]))
    return out


def _tensors(c, seed):
    """Per module: its input rows (None for down) and each tensor's trellis, suh, svh.  Any bit
    string is a valid trellis; suh and svh are signs times exp(N(0, 1/16)), svh times k ** -0.5 so that
    outputs are of the order of the inputs; activations N(0, 1) with one channel in a hundred 20
    times larger, as a decoder's hidden states have them."""
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 17)

    def randn(*s):
        return torch.randn(*s, device="cuda", generator=g)

    def scale(n):
        return (randn(n).sign() * torch.exp(0.25 * randn(n))).half()

    out = []
    for name, k, parts in _modules(c):
        x = None
        if name != "down":
            x = randn(c["m"], k)
            x *= torch.where(torch.rand(k, device="cuda", generator=g) < 0.01, 20.0, 1.0)
            x = x.half()
        ts = []
        for n, b in parts:
            words = torch.randint(-2 ** 31, 2 ** 31, (k // 16, n // 16, 8 * b), device="cuda", dtype=torch.int32, generator=g)
            ts.append((words.view(torch.int16), scale(k), (scale(n).float() * k ** -0.5).half()))
        out.append((name, k, parts, x, ts))
    return out


_MULT = {"mul1": 0x83DCD12D, "mcg": 0xCBAC1FED}
_capture = None                       # one capture stream per process, as a server has


def _load(k, parts, ts, book):
    """(method, layer) of one module, its checkpoint tensors through the plugin's loaders."""
    from exl3rocm import plugin
    method = plugin.Exl3LinearMethod(plugin.Exl3Config(book), [(f"t{i}", b, k, n) for i, (n, b) in enumerate(parts)])
    layer = torch.nn.Module()
    widths = [n for n, _ in parts]
    method.create_weights(layer, k, widths, k, sum(widths), torch.float16)
    layer.to("cuda")
    for i, t in enumerate(ts):
        shard = None if len(ts) == 1 else i
        for kind, w in zip(plugin.TENSOR_KINDS, t):
            target = getattr(layer, kind)
            target.weight_loader(target, w, shard)
        if book in _MULT:
            target = getattr(layer, book)
            target.weight_loader(target, torch.tensor(_MULT[book] - 2 ** 32), shard)
    method.process_weights_after_loading(layer)
    return method, layer


def _forward(st):
    out, gu = [], None
    for name, method, layer, x in st["mods"]:
        if name == "down":
            out.append(method.apply_silu_mul(layer, gu))
        else:
            y = method.apply(layer, x)
            if name == "gate_up":
                gu = y
            out.append(y)
    return out


def prepare(case, seed):
    global _capture
    st = {"mods": [(name, *_load(k, parts, ts, case["book"]), x) for name, k, parts, x, ts in _tensors(case, seed)]}
    if case["graph"]:
        if _capture is None:
            _capture = torch.cuda.Stream()
        _capture.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(_capture):          # an eager pass first, as a server warms up
            _forward(st)
        torch.cuda.current_stream().wait_stream(_capture)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"], stream=_capture):
            st["out"] = _forward(st)
    return st


def run(st):
    if "graph" in st:
        st["graph"].replay()
        return st["out"]
    return _forward(st)


def work(case):
    m, nbytes, flops = case["m"], 0, 0
    for name, k, parts in _modules(case):
        nbytes += 2 * m * (2 * k if name == "down" else k)
        for n, b in parts:
            nbytes += k * n * b // 8 + 2 * k + 2 * n + 2 * m * n
            flops += 2 * m * k * n
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # against 64-bit arithmetic the outputs are 4.5e-4 off, a down module's 8.7e-4 (the rounding of its input,
    # the rotated input, the sums and the outputs to fp16): two to four times that
    return {"rel": 2e-3}


# ---------------------------------------------------------------------------------------------
# the same in 64 bits: the format restated in plain torch
# ---------------------------------------------------------------------------------------------
def _codebook(book):
    """All 65536 states' weights (the format's own fp16 values), as float64 on the GPU."""
    w = np.arange(65536, dtype=np.uint64)
    if book == "mul1":
        x = (w * np.uint64(0x83DCD12D)) & np.uint64(0xFFFFFFFF)
        s = sum((x >> np.uint64(8 * i)) & np.uint64(255) for i in range(4)).astype(np.float64)
        inv, bias = (float(np.array(b, dtype=np.uint16).view(np.float16)) for b in (0x1EEE, 0xC931))
        v = ((1024.0 + s) * inv + bias).astype(np.float16)
    else:
        x = w * np.uint64(0xCBAC1FED) if book == "mcg" else w * np.uint64(89226354) + np.uint64(64248484)
        x = ((x & np.uint64(0x8FFF8FFF)) ^ np.uint64(0x3B603B60)).astype(np.uint32)
        lo, hi = (h.astype(np.uint16).view(np.float16).astype(np.float64) for h in (x & 0xFFFF, x >> 16))
        v = (lo + hi).astype(np.float16)
    return torch.from_numpy(v.astype(np.float64)).cuda()


def _weights(trellis, bits, table):
    """float64 W[k, n] of trellis tiles (k / 16, n / 16, 16 bits): state t is the 16 bits ending at
    ring bit (t + 1) bits, the ring's bits numbered from the top of each 32-bit word."""
    kt, nt, _ = trellis.shape
    t = torch.arange(256, device="cuda")
    first = ((t + 1) * bits - 16) % (256 * bits)
    h, r = first // 16, first % 16
    at = lambda i: trellis[..., (i % (16 * bits)) ^ 1].to(torch.int32) & 0xFFFF  # noqa: E731
    st = (((at(h).to(torch.int64) << 16) | at(h + 1)) >> (16 - r)) & 0xFFFF
    L, i = t >> 3, t & 7
    row = 2 * (L & 3) + (i & 1) + 8 * ((i >> 1) & 1)
    col = 2 * (L >> 3) + ((L >> 2) & 1) + 8 * (i >> 2)
    W = torch.empty(kt, nt, 16, 16, device="cuda", dtype=torch.float64)
    W[:, :, row, col] = table[st]
    return W.permute(0, 2, 1, 3).reshape(kt * 16, nt * 16)


def _had(x):
    h = torch.ones(1, 1, device="cuda", dtype=torch.float64)
    while h.shape[0] < 128:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.reshape(-1, 128) @ h / math.sqrt(128.0)).reshape(x.shape)


def exact(case, seed):
    out, gu, table = [], None, _codebook(case["book"])
    for name, k, parts, x, ts in _tensors(case, seed):
        if name == "down":
            x = torch.nn.functional.silu(gu[:, :k]) * gu[:, k:]
        x = x.double()
        cols = []
        for (n, b), (tr, su, sv) in zip(parts, ts):
            xh = _had(x * su.double())
            for c0 in range(0, n, 4096):
                c1 = min(n, c0 + 4096)
                y = xh @ _weights(tr[:, c0 // 16:c1 // 16], b, table)
                cols.append(_had(y) * sv[c0:c1].double())
        y = torch.cat(cols, 1)
        if name == "gate_up":
            gu = y
        out.append(y)
    return out

"""The work a program has this library do, as timed cases.

The shapes are those of the models behind the repository's benchmark and tests (hidden 1536 or
2048, FFN 8192 or 10752, q / k / v rows, a 65536-row Q8_0 head) and sizes around them, odd ones
among them.  What is timed is one call of one layer, a stack of layers or a whole decode step,
through ``llmhost_amd.q4``.

A decode step (up to 64 tokens: one per sequence that is being decoded) is captured once in a HIP
graph and replayed, as a serving loop and the benchmark do; prefill and single calls are made
directly.  A stack of layers holds distinct weights, so that they come from HBM as in a model.
"""

import numpy as np
import torch

from llmhost_amd import q4
from llmhost_amd.formats import BLOCK_Q8_0

EPS = 1e-5


# ---- the cases -------------------------------------------------------------------------------
def listed():
    return [
        # One projection of one token, called directly: the smallest call there is.
        {"name": "gemv_call", "kind": "linear", "tokens": 1, "k": 1536, "n": 1536, "layers": 1, "graph": False,
         "add": False, "row": False},
        # The same seam with host slices, as an engine that keeps its activations on the host calls it.
        {"name": "host_gemv", "kind": "host", "tokens": 1, "k": 2048, "n": 8192, "add": False},
        # One decode step of a 16-layer model, one sequence: every launch waits for the one before it.
        {"name": "decode_t1", "kind": "decode", "tokens": 1, "dim": 1536, "inter": 8192, "kv": 256, "layers": 16,
         "vocab": 65536},
        # The same for four sequences decoded together.
        {"name": "decode_t4", "kind": "decode", "tokens": 4, "dim": 2048, "inter": 8192, "kv": 512, "layers": 8,
         "vocab": 65536},
        # FFN blocks of a ragged batch of sequences (13 rows), a layer's own rows each.
        {"name": "ffn_t13", "kind": "ffn", "tokens": 13, "dim": 1536, "inter": 8192, "layers": 8, "graph": True},
        # Attention blocks' input projections of a larger batch: norm, then q / k / v.
        {"name": "qkv_t40", "kind": "qkv", "tokens": 40, "dim": 2048, "kv": 512, "layers": 16, "graph": True},
        # Ragged projections at the widest batch that is decoded.
        {"name": "ragged_t64", "kind": "linear", "tokens": 64, "k": 2048, "n": 8192, "layers": 8, "graph": True,
         "add": False, "row": False},
        # The final norm and output head of a batch of sequences.
        {"name": "head_t16", "kind": "head", "tokens": 16, "dim": 1536, "vocab": 65536},
        # A short prompt (97 tokens) through a layer's FFN block.
        {"name": "prefill_ffn_t97", "kind": "ffn", "tokens": 97, "dim": 1536, "inter": 8192, "layers": 2,
         "graph": False},
        # An ordinary prompt through the wider model's FFN block.
        {"name": "prefill_ffn_t512", "kind": "ffn", "tokens": 512, "dim": 2048, "inter": 10752, "layers": 1,
         "graph": False},
        # A prompt of odd length with one activation scale per row (ActQuant.PerRow), odd row count.
        {"name": "prefill_row_t777", "kind": "linear", "tokens": 777, "k": 2048, "n": 10749, "layers": 1,
         "graph": False, "add": False, "row": True},
        # The largest: a long prompt's down projection, added onto the residual rows.
        {"name": "prefill_down_t2048", "kind": "linear", "tokens": 2048, "k": 10752, "n": 2048, "layers": 1,
         "graph": False, "add": True, "row": False},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _width(rng, lo, hi):
    return max(lo, _log(rng, lo, hi) // 32 * 32)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "host", "decode", "ffn", "ffn", "qkv", "head"])
    if kind == "decode":
        return {"kind": kind, "tokens": rng.randint(1, 8), "dim": _width(rng, 1024, 2048),
                "inter": _width(rng, 4608, 10752), "kv": _width(rng, 256, 512), "layers": rng.randint(2, 8),
                "vocab": _log(rng, 32000, 65536)}
    if kind == "head":
        return {"kind": kind, "tokens": _log(rng, 1, 64), "dim": _width(rng, 1024, 2048),
                "vocab": _log(rng, 32000, 65536)}
    if kind == "host":
        return {"kind": kind, "tokens": _log(rng, 1, 32), "k": _width(rng, 512, 10752), "n": _log(rng, 512, 10752),
                "add": rng.random() < 0.5}
    tokens = _log(rng, 1, 1024)
    graph = tokens <= 64
    if kind == "ffn":
        return {"kind": kind, "tokens": tokens, "dim": _width(rng, 1024, 2048), "inter": _width(rng, 4608, 10752),
                "layers": rng.randint(4, 8) if graph else 1, "graph": graph}
    if kind == "qkv":
        return {"kind": kind, "tokens": tokens, "dim": _width(rng, 1024, 2048), "kv": _log(rng, 250, 1024),
                "layers": rng.randint(8, 16) if graph else 1, "graph": graph}
    return {"kind": kind, "tokens": tokens, "k": _width(rng, 512, 10752), "n": _log(rng, 500, 10752),
            "layers": rng.randint(4, 8) if graph else 1, "graph": graph, "add": rng.random() < 0.5,
            "row": rng.random() < 0.3}


# ---- inputs ------------------------------------------------------------------------------------
class _Source:
    """Weights and activations of one seed.  The same calls in the same order give the same values."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(1 + int(seed))

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.gen, device="cuda")

    def q4(self, n, k):
        """BlockQ4 bytes [n * k / 32, 18]: the codes and scales that quantizing Gaussian weights of
        variance 1 / k gives (32 values reach about 2.5 sigma, code -8)."""
        nb = n * (k // 32)
        code = torch.clamp(torch.round(self.normal(nb, 32) * 3.2), -8, 7).to(torch.int32) & 15
        scale = (0.9 + 0.2 * torch.rand(nb, 1, generator=self.gen, device="cuda")) / (3.2 * k ** 0.5)
        return torch.cat([scale.to(torch.float16).view(torch.uint8),
                          (code[:, 0::2] | (code[:, 1::2] << 4)).to(torch.uint8)], 1)

    def q8(self, n, k):
        """BlockQ8_0 bytes [n * k / 32, 34] of such weights."""
        nb = n * (k // 32)
        code = torch.clamp(torch.round(self.normal(nb, 32) * 45.0), -127, 127).to(torch.int8)
        scale = (0.9 + 0.2 * torch.rand(nb, 1, generator=self.gen, device="cuda")) / (45.0 * k ** 0.5)
        return torch.cat([scale.to(torch.float16).view(torch.uint8), code.view(torch.uint8)], 1)

    def rows(self, tokens, k):
        """Residual rows: unit variance, a few channels much larger, as in a trained model."""
        x = self.normal(tokens, k)
        x[:, :: max(1, k // 12)] *= 8.0
        return x

    def norm(self, k):
        return 1.0 + 0.1 * self.normal(k)


def _shapes(case):
    """The Q4 matrices (n, k) of one layer."""
    if case["kind"] in ("linear", "host"):
        return [(case["n"], case["k"])]
    d = case["dim"]
    qkv = [(d, d), (case["kv"], d), (case["kv"], d)] if "kv" in case else []
    ffn = [(case["inter"], d), (case["inter"], d), (d, case["inter"])] if "inter" in case else []
    return qkv + ([(d, d)] if case["kind"] == "decode" else []) + ffn


def _operands(case, seed):
    """The case's weights (as block bytes) and activations, in the order they are drawn."""
    s, t = _Source(seed), case["tokens"]
    layers = []
    for _ in range(case.get("layers", 0 if case["kind"] == "head" else 1)):
        L = {"w": [s.q4(n, k) for n, k in _shapes(case)]}
        if case["kind"] in ("linear", "host"):
            L["x"] = s.rows(t, case["k"])
            L["y0"] = s.normal(t, case["n"])
        else:
            L["nw"] = [s.norm(case["dim"]) for _ in range(2 if case["kind"] == "decode" else 1)]
            if case["kind"] != "decode":
                L["x"] = s.rows(t, case["dim"])
        layers.append(L)
    head = None
    if case["kind"] in ("decode", "head"):
        head = {"w": s.q8(case["vocab"], case["dim"]), "nw": s.norm(case["dim"]), "x": s.rows(t, case["dim"])}
    return layers, head


class _State:
    pass


def prepare(case, seed):
    """What the program holds: a context on its stream, uploaded weights (with the GEMM image where a
    prompt's length needs it), activations and output buffers, and the captured decode step."""
    layers, head = _operands(case, seed)
    st = _State()
    st.case, st.kind, st.tokens = case, case["kind"], case["tokens"]
    st.ctx = q4.Context(0)
    st.graph = None
    if st.kind == "host":
        L = layers[0]
        st.w = q4.Q4Matrix.from_blocks(case["n"], case["k"], L["w"][0], st.ctx)
        st.x = L["x"].cpu().numpy()
        st.y0 = L["y0"].cpu().numpy()
        st.out = np.zeros_like(st.y0)
        st.call = q4.gemm_q4_add if case["add"] else q4.gemm_q4
        return st
    st.stream = torch.cuda.Stream()
    st.ctx.set_stream(st.stream.cuda_stream)
    if case.get("row"):
        q4.set_act_quant(q4.ActQuant.PerRow, st.ctx)
    torch.cuda.synchronize()
    with torch.cuda.stream(st.stream):
        st.layers = []
        for L in layers:
            mats = [q4.Q4Matrix.from_blocks(n, k, b, st.ctx) for (n, k), b in zip(_shapes(case), L["w"])]
            if st.tokens > 48:
                for w in mats:
                    w.prepare_gemm()
            rows = [torch.zeros(st.tokens, w.n, device="cuda") for w in mats]
            st.layers.append({**L, "w": mats, "out": rows, "hidden": torch.empty_like(L["x"]) if "x" in L else None})
        if head is not None:
            blocks = head["w"].cpu().numpy().reshape(-1).view(BLOCK_Q8_0)
            st.head = q4.Q8Matrix.from_blocks(case["vocab"], case["dim"], blocks, st.ctx)
            st.head_nw, st.x = head["nw"], head["x"]
            st.hidden = torch.empty_like(st.x)
            st.logits = torch.zeros(st.tokens, case["vocab"], device="cuda")
        if case.get("graph") or st.kind == "decode":
            _step(st)  # sizes the workspaces: nothing may grow under capture
            torch.cuda.synchronize()
            st.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(st.graph, stream=st.stream):
                _step(st)
            st.graph.replay()  # the first replay uploads the graph
    torch.cuda.synchronize()
    return st


# ---- one pass ------------------------------------------------------------------------------------
def _step(st):
    t, kind = st.tokens, st.kind
    if kind == "linear":
        for L in st.layers:
            if st.case["add"]:
                L["out"][0].copy_(L["y0"])
                q4.gemm_q4_add(L["w"][0], L["x"], L["out"][0], t)
            else:
                q4.gemm_q4(L["w"][0], L["x"], L["out"][0], t)
        return [L["out"][0] for L in st.layers]
    if kind == "ffn":
        for L in st.layers:
            L["hidden"].copy_(L["x"])
            q4.ffn_residual(L["w"][0], L["w"][1], L["w"][2], L["nw"][0], EPS, L["hidden"], t)
        return [L["hidden"] for L in st.layers]
    if kind == "qkv":
        for L in st.layers:
            q4.norm_gemv(L["w"], L["nw"][0], EPS, L["x"], L["out"], t)
        return [o for L in st.layers for o in L["out"]]
    if kind == "head":
        q4.q8_norm_apply(st.head, st.head_nw, EPS, st.x, t, st.logits)
        return [st.logits]
    # decode: per layer the block's input side (q stands in for the attention output), the output
    # projection onto the residual rows, the FFN block; then the final norm and the head.
    st.hidden.copy_(st.x)
    for L in st.layers:
        q, k, v, o, w1, w3, w2 = L["w"]
        q4.norm_gemv([q, k, v], L["nw"][0], EPS, st.hidden, L["out"][:3], t)
        q4.apply_add_inplace(o, L["out"][0], st.hidden, t)
        q4.ffn_residual(w1, w3, w2, L["nw"][1], EPS, st.hidden, t)
    q4.q8_norm_apply(st.head, st.head_nw, EPS, st.hidden, t, st.logits)
    return [st.hidden, st.logits]


def _outputs(st):
    if st.kind == "linear":
        return [L["out"][0] for L in st.layers]
    if st.kind == "ffn":
        return [L["hidden"] for L in st.layers]
    if st.kind == "qkv":
        return [o for L in st.layers for o in L["out"]]
    return [st.hidden, st.logits]


def run(st):
    if st.kind == "host":
        if st.case["add"]:
            np.copyto(st.out, st.y0)
        st.call(st.w, st.x, st.out, st.tokens)
        return [st.out]
    with torch.cuda.stream(st.stream):
        if st.graph is None:
            return _step(st)
        st.graph.replay()
        return _outputs(st)


# ---- what a pass cannot do without -----------------------------------------------------------------
def work(case):
    t = case["tokens"]
    b = f = 0.0
    for n, k in _shapes(case) if case["kind"] != "head" else []:
        b += n * (k // 32) * 18
        f += 2.0 * t * n * k
    if case["kind"] in ("linear", "host"):
        b += 4.0 * t * (case["k"] + case["n"] * (2 if case["add"] else 1))
    elif case["kind"] == "ffn":
        b += 4.0 * (2 * t + 1) * case["dim"]
    elif case["kind"] == "qkv":
        b += 4.0 * ((t + 1) * case["dim"] + t * sum(n for n, _ in _shapes(case)))
    elif case["kind"] == "decode":  # q, k and v leave each layer; the residual rows stay on the chip
        b += 4.0 * (2 * case["dim"] + t * (case["dim"] + 2 * case["kv"]))
    b, f = b * case.get("layers", 1), f * case.get("layers", 1)
    if case["kind"] in ("decode", "head"):
        b += case["vocab"] * (case["dim"] // 32) * 34 + 4.0 * ((2 * t + 1) * case["dim"] + t * case["vocab"])
        f += 2.0 * t * case["vocab"] * case["dim"]
    return {"bytes": b, "flops": f}


def tolerance(case):
    """One projection is a sum of 32-bit terms over integer dots that are exact.  An FFN block
    quantizes its intermediate rows, where the last bit of a sum can move a value across a rounding
    tie: a few 8-bit codes of a million differ.  In a chain of layers such a code changes what
    follows it."""
    return {"ffn": {"rel": 5e-4, "max": 0.02}, "decode": {"rel": 2e-2, "max": 0.2}}.get(
        case["kind"], {"rel": 1e-6, "max": 2e-5})


# ---- the values in 64 bits -------------------------------------------------------------------------
def _act(x, per_row=False):
    """int8 codes times scale per 32 values (or per row), in f64: scale = amax / 127 and its inverse
    rounded to f32 as the format defines them, halves away from zero."""
    t, k = x.shape
    xb = x.reshape(t, k // 32, 32)
    amax = xb.abs().amax(2, keepdim=True)
    if per_row:
        amax = amax.amax(1, keepdim=True).expand(t, k // 32, 1)
    scale = (amax.double() / 127.0).float()
    inv = torch.where(scale > 0, (1.0 / scale.double()).float(), torch.zeros_like(scale))
    y = (xb * inv).double()
    q = torch.clamp(torch.sign(y) * torch.floor(y.abs() + 0.5), -127, 127)
    return (q * scale.double()).reshape(t, k)


def _w4(b, n, k):
    scale = b[:, :2].contiguous().view(torch.float16).double()
    qs = b[:, 2:].to(torch.int32)
    code = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 32)
    return ((((code ^ 8) - 8).double()) * scale).reshape(n, k)


def _w8(b, n, k):
    scale = b[:, :2].contiguous().view(torch.float16).double()
    return (b[:, 2:].contiguous().view(torch.int8).double() * scale).reshape(n, k)


def _normed(x, nw):
    """rms_norm with its f32 roundings: what is quantized is an f32 row."""
    scale = (1.0 / torch.sqrt(x.double().square().mean(1, keepdim=True) + float(np.float32(EPS)))).float()
    return nw * (x * scale)


def exact(case, seed):
    if case["kind"] == "decode":
        return None  # a code at a rounding tie decides what every later layer computes
    if case["kind"] == "ffn" and case["tokens"] <= 64:
        return None  # so few intermediate values that one code at a tie, or none, is the whole difference
    layers, head = _operands(case, seed)
    if case["kind"] == "head":
        a = _act(_normed(head["x"], head["nw"]))
        return [a @ _w8(head["w"], case["vocab"], case["dim"]).T]
    out = []
    for L in layers:
        w = [_w4(b, n, k) for (n, k), b in zip(_shapes(case), L["w"])]
        if case["kind"] in ("linear", "host"):
            y = _act(L["x"], bool(case.get("row"))) @ w[0].T
            y = y + L["y0"].double() if case["add"] else y
            out.append(y.cpu().numpy() if case["kind"] == "host" else y)
            continue
        a = _act(_normed(L["x"], L["nw"][0]))
        if case["kind"] == "qkv":
            out += [a @ m.T for m in w]
            continue
        g, u = a @ w[0].T, a @ w[1].T
        h = (g / (1.0 + torch.exp(-g)) * u).float()
        out.append(L["x"].double() + _act(h) @ w[2].T)
    return out

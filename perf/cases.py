"""Measured cases: the MUL_MATs of transformer layers, as this framework's users run them.

Four kinds, all through public entry points:

- "decode": token steps on resident K-quant weights (hip.gemv_decode), 1..16 rows, captured in a HIP graph as a
  serving loop keeps it. A step runs every layer's four launches (q/k/v, o, gate+up, down) on weights of their own,
  so they stream from HBM as they do between two tokens.
- "w8a8": prompt and batched-decode steps on resident W8 (hip.quantize_a8 + hip.gemm_w8a8), the same four products a
  layer; short ones in a graph, long prompts eagerly.
- "repack": a layer's (or a head's) K-quant tensors turned into W8 when a model is loaded (hip.repack_w8).
- "host": a layer through the routing over the C ABI on host buffers (route.run), as a ggml backend calls it: one
  call per group of nodes, weights resident after the first call, f16 weights sent along.

Weights hold uniform quants with scales as the benchmark's synthetic tensors have them; activations are N(0, 1).
"""
from __future__ import annotations

import numpy as np
import torch

from rocknpu_amd import hip, route
from rocknpu_amd.capi import Context

QK = 256
BLOCK = {4: 144, 5: 176, 6: 210}
ROUTE_TYPE = {4: route.Q4_K, 5: route.Q5_K, 6: route.Q6_K, 16: route.F16}
MAX_LAYERS = 32


def listed():
    tiny = {"hidden": 2048, "kv": 256, "ffn": 5632}   # TinyLlama-1.1B
    small = {"hidden": 2048, "kv": 512, "ffn": 8192}  # Llama-3.2-1B
    large = {"hidden": 4096, "kv": 1024, "ffn": 14336}  # Llama-3-8B
    return [
        # one user's token step on a small model: 88 short launches, each a few microseconds
        {"name": "decode-tiny-1", "kind": "decode", **tiny, "layers": 22, "rows": 1},
        # one user's token step on a larger model: streaming launches, 61 % of them gate+up
        {"name": "decode-large-1", "kind": "decode", **large, "layers": 8, "rows": 1},
        # eight sequences decoded together
        {"name": "decode-small-8", "kind": "decode", **small, "layers": 16, "rows": 8},
        # thirty-two sequences decoded together: past the GEMV's range, W8A8
        {"name": "batch-large-32", "kind": "w8a8", **large, "layers": 4, "rows": 32, "graph": True},
        # a short prompt on a small model (the reference's pp128)
        {"name": "prompt-tiny-128", "kind": "w8a8", **tiny, "layers": 22, "rows": 128, "graph": True},
        # a middling prompt of a length that no tile divides
        {"name": "prompt-small-509", "kind": "w8a8", **small, "layers": 8, "rows": 509, "graph": True},
        # a long prompt on a larger model
        {"name": "prompt-large-4096", "kind": "w8a8", **large, "layers": 1, "rows": 4096, "graph": False},
        # loading one layer of a larger Q4_K_M model (Q6_K down projection)
        {"name": "repack-large", "kind": "repack", **large, "quant": 4, "down": 6},
        # loading a vocabulary head, the largest single tensor
        {"name": "repack-head", "kind": "repack", "n": 128256, "k": 2048, "quant": 6},
        # a plugin's decode step of one layer on host buffers
        {"name": "host-tiny-1", "kind": "host", **tiny, "rows": 1, "quant": 4, "down": 6},
        # a plugin's short prompt, one layer on host buffers
        {"name": "host-tiny-128", "kind": "host", **tiny, "rows": 128, "quant": 4, "down": 6},
        # the same on an f16 model: the weights travel with every call
        {"name": "host-f16-64", "kind": "host", **tiny, "rows": 64, "quant": 16, "down": 16},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _model(rng, most):
    hidden = QK * _log(rng, 2, most)
    return {"hidden": hidden, "kv": rng.randrange(max(16, hidden // 16), hidden // 2 + 1),
            "ffn": QK * max(1, round(hidden / QK * (1.5 + 2.5 * rng.random())))}


def draw(rng):
    kind = rng.choice(["decode", "decode", "w8a8", "w8a8", "repack", "host"])
    if kind == "repack":
        quant = rng.choice([4, 5, 6])
        if rng.random() < 0.5:  # one tensor with any number of rows
            k = QK * _log(rng, 2, 56)
            return {"kind": kind, "n": _log(rng, 64, min(128256, (128256 * 2048) // k)), "k": k, "quant": quant}
        return {"kind": kind, **_model(rng, 16), "quant": quant, "down": rng.choice([quant, 6])}
    if kind == "host":
        quant = rng.choice([4, 4, 5, 6, 16])
        rows = _log(rng, 2, 64 if quant == 16 else 128) if quant in (5, 16) or rng.random() < 0.6 else 1
        return {"kind": kind, **_model(rng, 8 if quant == 16 else 12), "rows": rows, "quant": quant,
                "down": quant if quant in (5, 16) else 6}
    model = _model(rng, 16)
    per_layer = 2 * model["hidden"] ** 2 + 2 * model["kv"] * model["hidden"] + 3 * model["ffn"] * model["hidden"]
    layers = max(1, min(MAX_LAYERS, int(6e8 // per_layer)))
    if kind == "decode":
        return {"kind": kind, **model, "layers": layers, "rows": rng.randrange(1, 17)}
    rows = _log(rng, 1, 4096)
    return {"kind": kind, **model, "layers": max(1, min(layers, int(4e11 // (per_layer * rows)))), "rows": rows,
            "graph": rows <= 1024}


# (name, output rows, row length, which input it reads, is it the down projection) of a layer's projections
def _projections(c):
    h, kv, f = c["hidden"], c["kv"], c["ffn"]
    return [("q", h, h, 0), ("k", kv, h, 0), ("v", kv, h, 0), ("o", h, h, 1), ("gate", f, h, 2), ("up", f, h, 2),
            ("down", h, f, 3)]


def _calls(c):
    p = _projections(c)
    return [p[0:3], p[3:4], p[4:6], p[6:7]]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _blocks(g, quant, n, k):
    """Flat uint8 of n rows of k values as K-quant blocks."""
    nb = n * (k // QK)
    b = torch.randint(0, 256, (nb, BLOCK[quant]), dtype=torch.uint8, device="cuda", generator=g)

    def scale():
        return torch.randn(nb, device="cuda", generator=g).mul_(0.01).abs_().half().view(torch.uint8).view(nb, 2)

    if quant == 6:
        b[:, 192:208] = torch.randint(-63, 64, (nb, 16), device="cuda", generator=g).to(torch.int8).view(torch.uint8)
        b[:, 208:210] = scale()
    else:
        b[:, 0:2], b[:, 2:4] = scale(), scale()
    return b.view(-1)


def _inputs(g, c, layers):
    m = c["rows"]
    return [torch.randn(layers, m, k, device="cuda", generator=g) for k in
            (c["hidden"], c["hidden"], c["hidden"], c["ffn"])]


def _w8(g, n, k):
    w = torch.randn(n, hip.k_pad_of(k), device="cuda", generator=g).mul_(32).round_().clamp_(-127, 127).to(torch.int8)
    w[:, k:] = 0
    return w, torch.rand(n, device="cuda", generator=g).mul_(1e-3).add_(1e-4)


def _decode_data(c, seed):
    g = _generator(seed)
    x = _inputs(g, c, c["layers"])
    w = [[[_blocks(g, 6 if k == c["ffn"] and name == "down" else 4, n, k) for name, n, k, _ in call]
          for call in _calls(c)] for _ in range(c["layers"])]
    return x, w


def _w8a8_data(c, seed):
    g = _generator(seed)
    x = _inputs(g, c, c["layers"])
    w = [[_w8(g, sum(p[1] for p in call), call[0][2]) for call in _calls(c)] for _ in range(c["layers"])]
    return x, w


def _tensors(c):
    if "n" in c:
        return [(c["quant"], c["n"], c["k"])]
    return [(c["down"] if name == "down" else c["quant"], n, k) for name, n, k, _ in _projections(c)]


def _repack_data(c, seed):
    g = _generator(seed)
    return [_blocks(g, q, n, k) for q, n, k in _tensors(c)]


def _host_data(c, seed):
    g = _generator(seed)
    x = [t[0] for t in _inputs(g, c, 1)]
    w = [torch.randn(n, k, device="cuda", generator=g).mul_(0.02).half() if q == 16 else _blocks(g, q, n, k)
         for q, n, k in _tensors(c)]
    return x, w


_side = None


def _captured(step):
    """`step` as a HIP graph: run once on the capture stream (which brings that stream's workspaces), then captured."""
    global _side
    if _side is None:
        _side = torch.cuda.Stream()
    _side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(_side):
        step()
    _side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=_side):
        step()
    return graph


def prepare(case, seed):
    return {"decode": _prepare_decode, "w8a8": _prepare_w8a8, "repack": _prepare_repack,
            "host": _prepare_host}[case["kind"]](case, seed)


def _prepare_decode(c, seed):
    x, raw = _decode_data(c, seed)
    m, layers = c["rows"], c["layers"]
    outs = [[torch.empty(layers, m, n, device="cuda") for _, n, _, _ in call] for call in _calls(c)]
    kinds = (4, 4, 4, 6)
    tiled = [[None] * 4 for _ in range(layers)]
    for i, call in enumerate(_calls(c)):
        k = call[0][2]
        if hip.gemv_tiled_preferred(kinds[i], m, k):  # the one copy that this step reads
            for layer in range(layers):
                tiled[layer][i] = [hip.gemv_tile_weights(kinds[i], w, k, p[1]) for p, w in zip(call, raw[layer][i])]
                raw[layer][i] = None

    def step():
        for layer in range(layers):
            for i, call in enumerate(_calls(c)):
                hip.gemv_decode(kinds[i], raw[layer][i], tiled[layer][i], call[0][2], [p[1] for p in call],
                                x[i][layer], outs=[o[layer] for o in outs[i]])

    graph = _captured(step)
    return {"run": graph.replay, "outs": outs, "keep": (x, raw, tiled)}


def _prepare_w8a8(c, seed):
    x, w = _w8a8_data(c, seed)
    m, layers = c["rows"], c["layers"]
    outs = [torch.empty(layers, m, sum(p[1] for p in call), device="cuda") for call in _calls(c)]
    a8 = [torch.empty(m, hip.k_pad_of(call[0][2]), dtype=torch.int8, device="cuda") for call in _calls(c)]
    scales = torch.empty(m, device="cuda")

    def step():
        for layer in range(layers):
            for i in range(4):
                hip.quantize_a8(x[i][layer], a8=a8[i], scales=scales)
                hip.gemm_w8a8(a8[i], scales, *w[layer][i], out=outs[i][layer])

    run = _captured(step).replay if c["graph"] else step
    return {"run": run, "outs": outs, "keep": (x, w, a8, scales)}


def _prepare_repack(c, seed):
    blocks, tensors = _repack_data(c, seed), _tensors(c)
    outs = [(torch.empty(n, hip.k_pad_of(k), dtype=torch.int8, device="cuda"), torch.empty(n, device="cuda"))
            for _, n, k in tensors]

    def step():
        for (q, n, k), b, o in zip(tensors, blocks, outs):
            hip.repack_w8(q, b, k, n, *o)

    return {"run": step, "outs": outs}


def _prepare_host(c, seed):
    x, w = _host_data(c, seed)
    x = [t.cpu().numpy() for t in x]
    w = [(t.view(torch.int16) if t.dtype == torch.float16 else t).cpu().numpy() for t in w]
    outs, groups = [], []
    for call in _calls(c):
        nodes = []
        for _, n, k, i in call:
            outs.append(np.zeros((c["rows"], n), np.float32))
            j = len(outs) - 1
            nodes.append(route.node(ROUTE_TYPE[_tensors(c)[j][0]], w[j], k, n, x[i], outs[j]))
        groups.append(nodes)
    ctx = Context()

    def step():
        for nodes in groups:
            status = route.run(ctx, nodes, decode=route.DECODE_GGML)
            if status != 0:
                raise RuntimeError(f"route.run returned {status}")

    step()  # the weights become resident
    return {"run": step, "outs": outs, "keep": (ctx, x, w)}


def run(state):
    state["run"]()
    return state["outs"]


def work(case):
    if case["kind"] == "repack":
        return {"bytes": sum(n * (k // QK * BLOCK[q] + hip.k_pad_of(k) + 4) for q, n, k in _tensors(case)), "flops": 0}
    m, total, flops = case["rows"], 0, 0
    for call in _calls(case):
        total += 4 * m * call[0][2]  # activations, once a call
        for name, n, k, _ in call:
            if case["kind"] == "w8a8":
                weight = n * (hip.k_pad_of(k) + 4)
            elif case["kind"] == "decode":
                weight = n * (k // QK) * (210 if name == "down" else 144)
            else:
                q = case["down"] if name == "down" else case["quant"]
                weight = n * k * 2 if q == 16 else n * k // QK * BLOCK[q] if m == 1 else n * (hip.k_pad_of(k) + 4)
            total += weight + 4 * m * n
            flops += 2 * m * n * k
    layers = case.get("layers", 1)
    return {"bytes": total * layers, "flops": flops * layers}


def tolerance(case):
    # W8A8 sums are whole numbers below 2^31, rescaled by two f32 products in a stated order, and the repack is
    # bytes: both exact. The decode GEMV adds one f32 term per block (8e-8 off the 64-bit sums), the f16 product one
    # per value (1.3e-6 off).
    if case["kind"] == "repack" or case["kind"] == "w8a8":
        return "exact"
    if case["kind"] == "host" and case["quant"] == 16:
        return {"rel": 5e-6, "max": 5e-5}
    if case["kind"] == "host" and case["rows"] > 1:
        return "exact"
    return {"rel": 4e-7, "max": 5e-6}


# --- the same values in 64 bits ------------------------------------------------------------------------------------
# The quantisers are part of what the entry points compute, so their f32 scale and rounding are followed; everything
# after them is 64-bit.

def _half(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(quant, blocks, n, k):
    """[n, k] f64 values of K-quant blocks (sums of products that f64 holds exactly)."""
    b = blocks.view(-1, BLOCK[quant])
    nb = b.shape[0]
    if quant == 6:
        ql, qh = b[:, 0:128].view(nb, 2, 64).int(), b[:, 128:192].view(nb, 2, 32).int()
        lo, hi = ql[:, :, :32], ql[:, :, 32:]
        q = torch.stack([(lo & 15) | ((qh & 3) << 4), (hi & 15) | ((qh >> 2 & 3) << 4),
                         (lo >> 4) | ((qh >> 4 & 3) << 4), (hi >> 4) | ((qh >> 6 & 3) << 4)], 2).view(nb, 16, 16)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return ((q - 32).double() * (sc * _half(b[:, 208:210]))[:, :, None]).view(n, k)
    s = b[:, 4:16].int()
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1).double() * _half(b[:, 0:2])
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double() * _half(b[:, 2:4])
    qs = b[:, -128:].view(nb, 4, 32).int()
    q = torch.stack([qs & 15, qs >> 4], 2).view(nb, 8, 32)
    if quant == 5:
        bits = torch.arange(8, device=b.device).view(1, 8, 1)
        q = q + ((b[:, 16:48].int()[:, None, :] >> bits & 1) << 4)
    return (q.double() * sc[:, :, None] - mn[:, :, None]).view(n, k)


def _quotient(a, b):
    """The correctly rounded f32 quotient (a device's own f32 division may be an ulp off)."""
    a, b = (t.double() if isinstance(t, torch.Tensor) else t for t in (a, b))
    return (a / b).float()


def _symmetric(v):
    """f32 rows -> (whole numbers in [-127, 127], f32 scales), halves away from zero."""
    top = v.abs().amax(1)
    scale = torch.where(top > 0, _quotient(top, 127.0), torch.ones_like(top))
    r = _quotient(v, scale[:, None])
    return torch.copysign((r.abs().double() + 0.5).floor(), r).clamp_(-127, 127), scale


def _w8_of(quant, blocks, n, k):
    return _symmetric(_dequant(quant, blocks, n, k).float())


def _q8_k(x):
    """f32 rows -> the f64 values of their Q8_K blocks."""
    v = x.view(-1, QK)
    at = v.abs().argmax(1, keepdim=True)
    top = v.gather(1, at)
    inverse = _quotient(-127.0, top)
    q = torch.round(inverse * v).clamp_(max=127).double() * _quotient(1.0, inverse).double()
    return torch.where(top == 0, torch.zeros_like(q), q).view(x.shape)


def exact(case, seed):
    kind = case["kind"]
    if kind == "repack":
        outs = []
        for (q, n, k), b in zip(_tensors(case), _repack_data(case, seed)):
            w, s = _w8_of(q, b, n, k)
            outs.append((w.to(torch.int8), s))
        return outs
    if kind == "host":
        x, w = _host_data(case, seed)
        outs = []
        for (q, n, k), (_, _, _, i), b in zip(_tensors(case), _projections(case), w):
            if q == 16:
                outs.append(x[i].half().double() @ b.double().T)
            elif case["rows"] == 1:
                outs.append(_q8_k(x[i]) @ _dequant(q, b, n, k).T)
            else:
                (a, sa), (v, sv) = _symmetric(x[i]), _w8_of(q, b, n, k)
                outs.append((a @ v.T) * sa.double()[:, None] * sv.double()[None, :])
        return [o.cpu().numpy() for o in outs]
    if kind == "decode":
        x, w = _decode_data(case, seed)
        return [[torch.stack([_q8_k(x[i][layer]) @ _dequant(6 if i == 3 else 4, w[layer][i][j], n, k).T
                              for layer in range(case["layers"])]) for j, (_, n, k, _) in enumerate(call)]
                for i, call in enumerate(_calls(case))]
    x, w = _w8a8_data(case, seed)
    outs = []
    for i, call in enumerate(_calls(case)):
        k, rows = call[0][2], []
        for layer in range(case["layers"]):
            (a, sa), (v, sv) = _symmetric(x[i][layer]), w[layer][i]
            rows.append((a @ v[:, :k].double().T) * sa.double()[:, None] * sv.double()[None, :])
        outs.append(torch.stack(rows))
    return outs

"""The work that a program using this package has it do, as cases that can be timed and checked: trellis-coded linear
layers and MoE layers over decode rows and over prompts, the LM head, and a few layers of the whole decoder.

Decode-sized calls (up to 32 rows) run as a captured graph over several layers or several steps, as a serving engine
runs them: the weights of one pass then come from memory and not from a cache that holds a single layer. Prompts run
eagerly, in the package's default prefill mode (32-row windows' bits) and in its prompt ("tile") mode.

Sizes are those of the package's own benchmark (hidden 2048; q/k/v 4096 + 512 + 512; 256 experts of 512, top 8, one gated
shared expert; a vocabulary of 151936), and spread around them by draw().
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "vllm-espalier_amd"))

from vllm_espalier import experts as G  # noqa: E402
from vllm_espalier import linear as LN  # noqa: E402
from vllm_espalier import moe as M  # noqa: E402
from vllm_espalier import step as ST  # noqa: E402
from vllm_espalier import workloads as WL  # noqa: E402

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    block = {"hidden": 2048, "q": 4096, "kv": 512, "inter": 512, "attn_grid": "int6", "mlp_grid": "int5", "bits": 4,
             "dtype": "bf16"}
    layer = {"hidden": 2048, "inter": 512, "experts": 256, "k": 8, "shared": True, "dtype": "bf16"}
    return [
        # one matrix, one fp16 row, called eagerly: the smallest call, bound by launch and host latency
        {"name": "matrix_1", "kind": "matrix", "rows": 1, "in": 2048, "out": 2048, "grid": "int6", "bits": 4},
        # the dense layers of a decode step at batch 1 and at the largest batch one launch takes
        {"name": "dense_1", "kind": "dense", "rows": 1, "layers": 12, **block},
        {"name": "dense_32", "kind": "dense", "rows": 32, "layers": 12, **block},
        # the LM head of a decode step: the largest single matrix
        {"name": "head_1", "kind": "head", "rows": 1, "hidden": 2048, "vocab": 151936, "bits": 6, "dtype": "bf16"},
        # routing and experts of one MoE layer over decode steps, at batch 1 and at an odd batch of many sequences
        {"name": "moe_1", "kind": "moe", "rows": 1, "steps": 16, **layer},
        {"name": "moe_29", "kind": "moe", "rows": 29, "steps": 4, **layer},
        # a prompt through the dense layers: the default mode over a ragged prompt, the prompt mode over a long one
        {"name": "dense_prompt_509", "kind": "dense_prompt", "mode": "default", "rows": 509, **block},
        {"name": "dense_prompt_tile_2048", "kind": "dense_prompt", "mode": "tile", "rows": 2048, **block},
        # a prompt through the MoE layer, in the same two modes
        {"name": "moe_prompt_391", "kind": "moe_prompt", "mode": "default", "rows": 391, **layer},
        {"name": "moe_prompt_tile_1531", "kind": "moe_prompt", "mode": "tile", "rows": 1531, **layer},
        # whole calls: a captured decode step, and the prefill of a 512-token prompt, with the LM head
        {"name": "decoder_step", "kind": "decoder", "rows": 1, "layers": 4, "vocab": 151936},
        {"name": "decoder_prefill_512", "kind": "prefill", "rows": 512, "layers": 4, "vocab": 151936},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matrix", "dense", "dense", "head", "moe", "moe", "dense_prompt", "dense_prompt", "moe_prompt",
                       "moe_prompt", "decoder", "prefill"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    hidden = 128 * rng.choice([8, 12, 16, 16, 20, 24])
    block = {"hidden": hidden, "q": 128 * rng.randint(8, 32), "kv": 128 * rng.randint(1, 6),
             "inter": 128 * rng.randint(2, 8), "attn_grid": rng.choice(["int6", "mcg"]),
             "mlp_grid": rng.choice(["int5", "mcg"]), "bits": rng.choice([3, 4]), "dtype": dtype}
    layer = {"hidden": 256 * rng.choice([4, 6, 8, 8]), "inter": 128 * rng.choice([2, 3, 4, 4, 6, 8]),
             "experts": rng.choice([64, 100, 128, 256]), "k": rng.choice([2, 4, 6, 8]), "shared": rng.random() < 0.7,
             "dtype": dtype}
    if kind == "matrix":
        grid, bits = rng.choice([("mcg", rng.randint(2, 8)), ("int6", 4), ("int6", 5), ("int5", 3), ("e2m1", 2)])
        return {"kind": kind, "rows": _log(rng, 1, 32), "in": 128 * rng.randint(4, 32), "out": 128 * rng.randint(2, 40),
                "grid": grid, "bits": bits}
    if kind == "dense":
        return {"kind": kind, "rows": _log(rng, 1, 32), "layers": rng.randint(4, 8), **block}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 1, 16), "hidden": hidden if hidden <= 2048 else 2048,
                "vocab": 128 * rng.randint(250, 1187), "bits": rng.choice([4, 5, 6]), "dtype": dtype}
    if kind == "moe":
        return {"kind": kind, "rows": _log(rng, 1, 32), "steps": rng.randint(2, 4), **layer}
    if kind == "dense_prompt":
        return {"kind": kind, "mode": rng.choice(["default", "tile"]), "rows": _log(rng, 33, 1400), **block}
    if kind == "moe_prompt":
        return {"kind": kind, "mode": rng.choice(["default", "tile"]), "rows": _log(rng, 33, 1500), **layer}
    if kind == "decoder":
        return {"kind": kind, "rows": _log(rng, 1, 8), "layers": rng.randint(1, 4), "vocab": 128 * rng.randint(250, 1187)}
    return {"kind": kind, "rows": _log(rng, 33, 500), "layers": rng.randint(1, 4), "vocab": 128 * rng.randint(250, 1187)}


# ---- what a program has in hand

def _block_shapes(c):
    """(input width, [output widths], grid) of a block's four linear layers: q/k/v, o, gate/up, down."""
    h, q, kv, i = c["hidden"], c["q"], c["kv"], c["inter"]
    return [(h, [q, kv, kv], c["attn_grid"]), (q, [h], c["attn_grid"]), (h, [i, i], c["mlp_grid"]), (i, [h], c["mlp_grid"])]


def _linear(K, outs, grid, bits, gen):
    mats = [WL.matrix(K, n, bits, grid, gen, DEV) for n in outs]
    return LN.TrellisLinear(mats, sum(outs), fused=True)


def _rows(T, K, gen, dtype):
    return torch.randn((T, K), generator=gen, device=DEV).to(dtype)


def _expert_mats(c, gen):
    """Routed experts of 1 to 3 bits (E2M1 at 1 and 2, int5 at 3), the shared expert of 4 bits."""
    D, I = c["hidden"], c["inter"]
    grid = {1: "e2m1", 2: "e2m1", 3: "int5"}
    widths = torch.randint(1, 4, (c["experts"],), generator=gen, device=DEV).tolist()
    experts = [tuple(WL.matrix(k, n, b, grid[b], gen, DEV) for k, n in ((D, I), (D, I), (I, D))) for b in widths]
    shared = tuple(WL.matrix(k, n, 4, "int5", gen, DEV) for k, n in ((D, I), (D, I), (I, D))) if c["shared"] else None
    return experts, shared


def _make(case, seed):
    """Weights and inputs of a layer case from the seed alone."""
    c = case
    gen = torch.Generator(device=DEV).manual_seed(seed)
    if c["kind"] == "matrix":
        return {"mats": [WL.matrix(c["in"], c["out"], c["bits"], c["grid"], gen, DEV)],
                "x": [_rows(c["rows"], c["in"], gen, torch.float16)]}
    dtype = DTYPES[c["dtype"]]
    if c["kind"] == "head":
        return {"layers": [_linear(c["hidden"], [c["vocab"]], "mcg", c["bits"], gen)],
                "x": [_rows(c["rows"], c["hidden"], gen, dtype)]}
    if c["kind"] in ("dense", "dense_prompt"):
        shapes = _block_shapes(c) * c.get("layers", 1)
        return {"layers": [_linear(K, outs, grid, c["bits"], gen) for K, outs, grid in shapes],
                "x": [_rows(c["rows"], K, gen, dtype) for K, _, _ in shapes]}
    experts, shared = _expert_mats(c, gen)
    D = c["hidden"]
    gate_w = (torch.randn((D,), generator=gen, device=DEV) * 0.05).to(dtype) if c["shared"] else None
    router = (torch.randn((c["experts"], D), generator=gen, device=DEV) * 0.02).to(dtype)
    return {"experts": experts, "shared": shared, "gate_w": gate_w, "router": router, "k": c["k"],
            "x": [_rows(c["rows"], D, gen, dtype) for _ in range(c.get("steps", 1))]}


def _captured(call):
    """(graph, outputs) of call(), after two warm-up passes on a side stream."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return graph, out


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decoder", "prefill"):
        dec = ST.SyntheticDecoder(case["layers"], seed, DEV, vocab=case["vocab"])
        gen = torch.Generator(device=DEV).manual_seed(seed + 1)
        T = case["rows"]
        ids = torch.randint(0, case["vocab"], (T,), generator=gen, device=DEV, dtype=torch.int32)
        if kind == "prefill":
            dec.prefill_buffers(T).ids_in.copy_(ids)
            dec.prefill_scratch(T)
            return {"call": lambda: dec.prefill(T).logits[T - 1:]}
        dec.buffers(T).ids_in.copy_(ids)
        graph, out = _captured(lambda: dec.forward(T).logits)
        return {"graph": graph, "out": out, "keep": dec}
    s = _make(case, seed)
    if kind == "matrix":
        m, x = s["mats"][0], s["x"][0]
        return {"call": lambda: m.forward(x)}
    if kind in ("dense", "head"):
        graph, out = _captured(lambda: [layer(x) for layer, x in zip(s["layers"], s["x"])])
        return {"graph": graph, "out": out, "keep": s}
    if kind == "dense_prompt":
        if case["mode"] == "default":
            return {"call": lambda: [layer(x) for layer, x in zip(s["layers"], s["x"])]}
        from vllm_espalier import ops
        dense = [ops.DENSE_LAYERS[layer.dense_key] for layer in s["layers"]]
        return {"call": lambda: [d.forward_tile(x) for d, x in zip(dense, s["x"])], "keep": s}
    L = G.prepare(s["experts"], s["shared"], s["gate_w"])
    k, router, slots = s["k"], s["router"], s["k"] + case["shared"]
    if kind == "moe":
        graph, out = _captured(lambda: [M.run_grouped(L, x, None, None, k, router) for x in s["x"]])
        return {"graph": graph, "out": out, "keep": (s, L)}
    x = s["x"][0]
    if case["mode"] == "default":
        return {"call": lambda: M.run_grouped(L, x, None, None, k, router), "keep": s}
    scratch = G.prefill_scratch(L, case["rows"], slots, x.device)
    return {"call": lambda: G.prefill(x, None, None, L, scratch, k, gate=router), "keep": s}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["call"]()


# ---- what a pass cannot do without

def _matrix_bytes(K, N, bits):
    return K * N * bits / 8 + 2 * K + 2 * N


def _moe_work(c, T, steps=1):
    """The distinct experts that T rows pick (their expected number), each read once, at the experts' mean of 2 bits."""
    D, I, E, k = c["hidden"], c["inter"], c["experts"], c["k"]
    distinct = E * (1 - (1 - k / E) ** T)
    per = 2 * _matrix_bytes(D, I, 2) + _matrix_bytes(I, D, 2)
    b = distinct * per + (2 * _matrix_bytes(D, I, 4) + _matrix_bytes(I, D, 4)) * c["shared"] + 2 * E * D
    b += 2 * T * D * (2 + c["shared"])
    flops = 2 * T * 3 * D * I * (k + c["shared"]) + 2 * T * E * D
    return steps * b, steps * flops


def _dense_work(c, T):
    b = f = 0
    for K, outs, _ in _block_shapes(c):
        b += sum(_matrix_bytes(K, n, c["bits"]) for n in outs) + 2 * T * (K + sum(outs))
        f += 2 * T * K * sum(outs)
    return b, f


def work(case):
    c, T = case, case["rows"]
    if c["kind"] == "matrix":
        b, f = _matrix_bytes(c["in"], c["out"], c["bits"]) + 2 * T * (c["in"] + c["out"]), 2 * T * c["in"] * c["out"]
    elif c["kind"] in ("dense", "dense_prompt"):
        b, f = (c.get("layers", 1) * v for v in _dense_work(c, T))
    elif c["kind"] == "head":
        b = _matrix_bytes(c["hidden"], c["vocab"], c["bits"]) + 2 * T * (c["hidden"] + c["vocab"])
        f = 2 * T * c["hidden"] * c["vocab"]
    elif c["kind"] in ("moe", "moe_prompt"):
        b, f = _moe_work(c, T, c.get("steps", 1))
    else:
        D = ST.D_MODEL
        layer = {"hidden": D, "inter": ST.EXPERT_I, "experts": 256, "k": ST.TOPK, "shared": 1}
        b, f = _moe_work(layer, T)
        for K, n in ((D, ST.Q_OUT), (D, 2 * ST.KV_OUT), (ST.Q_OUT, D)):
            b, f = b + _matrix_bytes(K, n, 4), f + 2 * T * K * n
        rows = T if c["kind"] == "decoder" else 1
        b = c["layers"] * b + _matrix_bytes(D, c["vocab"], 6) + 2 * T * D + 2 * rows * c["vocab"]
        f = c["layers"] * f + 2 * rows * D * c["vocab"]
    return {"bytes": b, "flops": f}


def tolerance(case):
    # Against 64 bits, 16-bit outputs of a layer are about 1.7e-3 off (bf16) or 4e-4 (fp16, with the fp16 rounding of
    # the rotated rows); an expert layer rounds its rows once more between its products. Four times that. A few layers
    # of the whole decoder carry each layer's roundings on.
    if case["kind"] == "matrix":
        return {"rel": 2e-3}
    if case["kind"] in ("decoder", "prefill"):
        return {"rel": 2e-2}
    return {"rel": 7e-3}


# ---- the same in 64 bits, from the format's definition

def _grid(grid, v):
    """The decoded weight of an mcg value (float64, exact fp16 values) on a grid."""
    if grid == 0:
        return v
    if grid == 1:                                  # E2M1: the nearest of 0.75 * {0, .5, 1, 1.5, 2, 3, 4, 6}, ties down
        points = 0.75 * torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=v.device)
        edges = (points[1:] + points[:-1]) / 2
        return torch.copysign(points[torch.bucketize(v.abs(), edges, right=False)], v)
    c = torch.tensor(3.94921875 / (15 if grid == 3 else 31), dtype=torch.float32, device=v.device)
    q = torch.round(v.float() / c)                 # the format's index: a quotient of 32-bit floats, ties to even
    return (q * c).to(torch.float16).to(torch.float64)


_VALUES = {}


def _table(grid):
    """The weight of each of the 65536 trellis states."""
    if grid not in _VALUES:
        s = torch.arange(65536, dtype=torch.int64, device=DEV)
        h = ((s * 0xCBAC1FED) & 0x8FFF8FFF) ^ 0x3B603B60
        halves = [((h >> sh) & 0xFFFF).to(torch.int32) for sh in (0, 16)]
        lo, hi = ((u - 65536 * (u >= 32768)).to(torch.int16).view(torch.float16) for u in halves)
        _VALUES[grid] = _grid(grid, (lo.float() + hi.float()).to(torch.float16).to(torch.float64))
    return _VALUES[grid]


def _weight(m):
    """W [in, out] of a matrix in float64: state p of a 16x16 tile is the 16 bits of its circular big-endian bit stream
    that end at bit (p + 1) * bits."""
    kt, nt, words = m.trellis.shape
    b, dev = words // 16, m.trellis.device
    w = m.trellis.reshape(kt, nt, words // 2, 2).to(torch.int64) & 0xFFFF
    w = w[..., 0] | (w[..., 1] << 16)                                  # 8 * bits 32-bit words a tile
    p = torch.arange(256, device=dev)
    start = ((p + 1) * b - 16) % (256 * b)
    word, off = start // 32, start % 32
    two = (w[..., word] << 16) | (w[..., (word + 1) % (8 * b)] >> 16)  # 48 bits
    s = (two >> (32 - off)) & 0xFFFF
    lane, j = p // 8, p % 8
    q, t, g = j // 2, lane % 4, lane // 4
    row, col = 2 * t + 8 * (q & 1) + (j & 1), g + 8 * (q >> 1)
    out = torch.empty((kt, nt, 16, 16), dtype=torch.float64, device=dev)
    out[:, :, row, col] = _table(m.cb)[s]
    return out.permute(0, 2, 1, 3).reshape(16 * kt, 16 * nt)


def _hadamard():
    h = torch.ones((1, 1), dtype=torch.float64, device=DEV)
    while h.shape[0] < 128:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(128)


def _times(x, m):
    """H(H(x * suh) @ W) * svh in float64."""
    H = _hadamard()
    x = ((x.double() * m.suh.double()).reshape(x.shape[0], -1, 128) @ H).reshape(x.shape[0], -1)
    y = x @ _weight(m)
    return (y.reshape(x.shape[0], -1, 128) @ H).reshape(x.shape[0], -1) * m.svh.double()


def _mlp(x, mats):
    g, u, d = mats
    a = _times(x, g)
    return _times(a * torch.sigmoid(a) * _times(x, u), d)


def _moe_exact(s, x):
    logits = (x.double() @ s["router"].double().t()).to(torch.bfloat16 if x.dtype == torch.bfloat16 else torch.float16)
    order = torch.sort(logits.double(), dim=1, descending=True, stable=True)      # ties: the lowest id first
    ids, top = order.indices[:, :s["k"]], order.values[:, :s["k"]]
    w = torch.softmax(top, dim=1)
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    for e in torch.unique(ids).tolist():
        r, slot = torch.nonzero(ids == e, as_tuple=True)
        out.index_add_(0, r, _mlp(x[r], s["experts"][e]) * w[r, slot, None])
    if s["shared"] is None:
        return out, None
    gate = torch.sigmoid(x.double() @ s["gate_w"].double())
    return out, _mlp(x, s["shared"]) * gate[:, None]


def exact(case, seed):
    if case["kind"] in ("decoder", "prefill"):
        return None
    s = _make(case, seed)
    if case["kind"] == "matrix":
        return _times(s["x"][0], s["mats"][0])
    if case["kind"] in ("dense", "head", "dense_prompt"):
        return [torch.cat([_times(x, m) for m in layer.mats], dim=1) for layer, x in zip(s["layers"], s["x"])]
    outs = [_moe_exact(s, x) for x in s["x"]]
    return outs if case["kind"] == "moe" else outs[0]

"""cases.py -- the routed-expert work whose speed is measured: what a program that runs EXL3 experts on this library asks
of it, through its public entry points (radiance-exl3_amd/exl3c4.py over include/exl3c4.h).

Four kinds of work:
  layer   one routed MoE layer on the device, as a serving step runs it: router_topk_scatter on the router's logits, then
          launch_gather (gate_up_down over the live experts and the weighted sum of each token's slots)
  expert  one gate_up_down launch of a single expert (top_k 1), another resident expert each state
  chain   the ops one by one, as an engine that schedules them apart runs them: prep_gu, gate_up on the rotated input with
          its output rotated for down, down
  load    a loader's host step: the canonical planes of one expert re-laid into the stored records

Experts are drawn as stored records of uniform random bits (every symbol sequence is a valid trellis) with sign scales of
varied magnitude; activations are N(0, 1); routing logits are N(0, 1), or with `zipf` a Zipf(1.1) popularity over a random
permutation of the experts plus Gumbel noise.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "radiance-exl3_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import exl3c4  # noqa: E402

ZIPF_S = 1.1


def _layer(name, tokens, **kw):
    c = {"name": name, "kind": "layer", "tokens": tokens, "hidden": 2048, "widths": "512", "n_expert": 512, "top_k": 10,
         "bits": 4, "dn_bits": 4, "codebook": "mul1", "bf16": False, "zipf": False}
    c.update(kw)
    return c


def listed():
    return [
        # one sequence's decode step: ten experts of one row, latency and launches
        _layer("decode-1", 1),
        # two sequences x four speculative positions: the decode layer's usual batch
        _layer("decode-8", 8),
        # the same step in a layer whose projections carry different bits a weight
        _layer("decode-8-mixed-k", 8, bits=3, dn_bits=6),
        # a batched decode or verify step, bf16 hidden states: most of the layer's experts live, about one row each
        _layer("decode-32-bf16", 32, bf16=True),
        # a short prompt: every expert live, two or three rows each
        _layer("prefill-128", 128),
        # a prompt of odd length, bf16 hidden states, 3 bits, another codebook
        _layer("prefill-613-mcg", 613, bits=3, dn_bits=3, codebook="mcg", bf16=True),
        # a long prompt with a skewed expert popularity
        _layer("prefill-2048-zipf", 2048, zipf=True),
        # the largest prompt chunk
        _layer("prefill-4096", 4096),
        # a tensor-parallel slice whose experts come in two widths, a ragged prompt
        _layer("two-class-77", 77, hidden=2560, widths="384,256"),
        # one SwiGLU expert on a small batch
        {"name": "expert-16", "kind": "expert", "tokens": 16, "hidden": 2048, "widths": "512", "n_expert": 64,
         "top_k": 1, "bits": 5, "dn_bits": 5, "codebook": "mul1", "bf16": False, "zipf": False},
        # the ops launched one by one on a speculative batch
        {"name": "chain-4-3inst", "kind": "chain", "tokens": 4, "hidden": 2560, "widths": "640", "n_expert": 512,
         "top_k": 10, "bits": 4, "dn_bits": 4, "codebook": "3inst", "bf16": False, "zipf": False},
        # loading one expert: gate_up's and down's planes
        {"name": "load-expert", "kind": "load", "hidden": 2048, "widths": "512", "bits": 4, "dn_bits": 4},
    ]


def draw(rng):
    kind = rng.choice(["layer"] * 7 + ["expert", "chain", "load"])
    hidden, widths = rng.choice([(2048, "512"), (2560, "640"), (1024, "256"), (2048, "768"), (2560, "384,256"),
                                 (1536, "384")])
    bits = rng.choice([2, 3, 4, 4, 4, 5, 6, 8])
    dn_bits = rng.choice([bits, bits, bits, rng.choice([2, 3, 4, 5, 6, 8])])
    if kind == "load":
        return {"kind": "load", "hidden": hidden, "widths": widths.split(",")[0], "bits": bits, "dn_bits": dn_bits}
    codebook = rng.choice(["mul1", "mul1", "mul1", "mcg", "3inst"])
    bf16 = rng.random() < 0.4
    if kind == "expert":
        return {"kind": "expert", "tokens": rng.choice([1, 2, 3, 4, 7, 8, 11, 16]), "hidden": hidden,
                "widths": widths.split(",")[0], "n_expert": 64, "top_k": 1, "bits": bits, "dn_bits": dn_bits,
                "codebook": codebook, "bf16": bf16, "zipf": False}
    n_expert, top_k = rng.choice([(512, 10), (512, 10), (512, 8), (256, 8), (128, 8), (128, 6)])
    if kind == "chain":
        return {"kind": "chain", "tokens": rng.randint(1, 16), "hidden": hidden, "widths": widths,
                "n_expert": n_expert, "top_k": top_k, "bits": bits, "dn_bits": bits, "codebook": codebook,
                "bf16": bf16, "zipf": False}
    # tokens over their logarithm; no draw costs more than the largest listed case
    tokens = int(round(math.exp(rng.uniform(0.0, math.log(1500.0)))))
    return {"kind": "layer", "tokens": max(1, tokens), "hidden": hidden, "widths": widths, "n_expert": n_expert,
            "top_k": top_k, "bits": bits, "dn_bits": dn_bits, "codebook": codebook, "bf16": bf16,
            "zipf": rng.random() < 0.3}


# ------------------------------------------------------------------------------------------ inputs
def _widths(case):
    return [int(w) for w in case["widths"].split(",")]


def _scales(g, shape, mag):
    """Signs times magnitudes in [0.5, 1.5) x mag, f16 (their bits)."""
    s = torch.randint(0, 2, shape, device="cuda", generator=g).float() * 2 - 1
    m = torch.rand(shape, device="cuda", generator=g) + 0.5
    return (s * m * mag).half().view(torch.int16)


def _experts(case, g):
    """Per class c of n_class: the stacked planes of the experts e with e % n_class == c."""
    H, K, Kd = case["hidden"], case["bits"], case["dn_bits"]
    ws = _widths(case)
    out = []
    for c, W in enumerate(ws):
        n = (case["n_expert"] - c + len(ws) - 1) // len(ws)

        def codes(nbytes):
            return torch.randint(0, 256, (n, nbytes), dtype=torch.uint8, device="cuda", generator=g)
        out.append({"n": n, "W": W, "gu": codes(2 * W * H * K // 8), "dn": codes(H * W * Kd // 8),
                    "suh": _scales(g, (n, H), 1.0), "suh1": _scales(g, (n, H), 1.0),
                    "svh": _scales(g, (n, 2 * W), 1.0 / math.sqrt(H)), "dn_suh": _scales(g, (n, W), 1.0),
                    "dn_svh": _scales(g, (n, H), 1.0 / math.sqrt(W))})
    return out


def _logits(case, g):
    M, E = case["tokens"], case["n_expert"]
    if not case["zipf"]:
        return torch.randn((M, E), device="cuda", generator=g)
    rank = torch.randperm(E, device="cuda", generator=g).float() + 1.0
    u = torch.rand((M, E), device="cuda", generator=g).clamp_(1e-12, 1.0 - 1e-7)
    return -ZIPF_S * torch.log(rank)[None, :] - torch.log(-torch.log(u))


def _inputs(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    s = {"experts": _experts(case, g)}
    x = torch.randn((case["tokens"], case["hidden"]), device="cuda", generator=g)
    s["x_val"] = x.bfloat16() if case["bf16"] else x.half()
    if case["kind"] == "expert":
        s["expert"] = int(torch.randint(0, case["n_expert"], (1,), device="cuda", generator=g))
    else:
        s["logits"] = _logits(case, g)
    return s


def _load_planes(case, seed):
    r = np.random.default_rng(int(seed))
    H, W = case["hidden"], _widths(case)[0]
    return (r.integers(0, 256, (2 * W, (H * case["bits"] + 7) // 8), dtype=np.uint8),
            r.integers(0, 256, (H, (W * case["dn_bits"] + 7) // 8), dtype=np.uint8))


def prepare(case, seed):
    if case["kind"] == "load":
        gu, dn = _load_planes(case, seed)
        return {"kind": "load", "gu": gu, "dn": dn, "H": case["hidden"], "W": _widths(case)[0], "K": case["bits"],
                "Kd": case["dn_bits"]}
    s = _inputs(case, seed)
    M, k, E, H = case["tokens"], case["top_k"], case["n_expert"], case["hidden"]
    T, Wmax, K, Kd, cb = M * k, max(_widths(case)), case["bits"], case["dn_bits"], case["codebook"]
    bf = case["bf16"]
    s.update(kind=case["kind"], k=k, E=E, stream=torch.cuda.current_stream(), x=s["x_val"].view(torch.int16))

    def i32(*shape):
        return torch.zeros(shape, dtype=torch.int32, device="cuda")

    def i16(*shape):
        return torch.zeros(shape, dtype=torch.int16, device="cuda")
    gu = [exl3c4.make_class(2 * c["W"], H, codes=c["gu"], suh=c["suh"], suh1=c["suh1"], svh=c["svh"],
                            dn_suh=c["dn_suh"]) for c in s["experts"]]
    s["st"], s["off"] = i32(T), i32(E + 1)
    s["y"] = i16(T, H)
    if case["kind"] == "expert":
        s["st"].copy_(torch.arange(T, device="cuda"))
        s["off"][s["expert"] + 1:] = T
    else:
        s["ids"], s["row_of"] = i32(M, k), i32(T)
        s["w"] = torch.zeros((M, k), dtype=torch.float32, device="cuda")
    if case["kind"] in ("layer", "expert"):
        dn = [exl3c4.make_class(H, c["W"], codes=c["dn"], svh=c["dn_svh"]) for c in s["experts"]]
        s["op"] = exl3c4.make_op(exl3c4.GU_DN, K, cb, gu, s["x"], s["st"], s["off"], s["y"], M, k, dn=dn, x_bf16=bf,
                                 dn_bits=0 if K == Kd else Kd)
        s["scratch"] = exl3c4.alloc_scratch(s["op"])
        # the counter block a serving loop zeroes once and keeps
        s["ctr"] = torch.zeros(max(exl3c4.ctr_bytes(s["op"]), 256), dtype=torch.uint8, device="cuda")
        s["out"] = i16(M, H)
    else:
        dn = [exl3c4.make_class(H, c["W"], codes=c["dn"], suh=c["dn_suh"], svh=c["dn_svh"]) for c in s["experts"]]
        s["xr"], s["h"] = i16(T, 2 * H), i16(T, Wmax)
        s["ops"] = [
            exl3c4.make_op(exl3c4.PREP_GU, K, cb, gu, s["x"], s["st"], s["off"], s["xr"], M, k, x_bf16=bf),
            exl3c4.make_op(exl3c4.GATE_UP, K, cb, gu, s["xr"], s["st"], s["off"], s["h"], M, k, h_rot=1, a_rot=1),
            exl3c4.make_op(exl3c4.DOWN, K, cb, dn, s["h"], s["st"], s["off"], s["y"], M, k, h_rot=1)]
        s["scratch"] = torch.empty(max([256] + [exl3c4.scratch_bytes(o) for o in s["ops"]]), dtype=torch.uint8,
                                   device="cuda")
        # routed before: the ops alone are the pass
        rc = exl3c4.router_topk_scatter(s["logits"], k, True, s["ids"], s["w"], s["st"], s["off"], None, s["row_of"],
                                        s["stream"])
        if rc:
            raise RuntimeError(f"router_topk_scatter: {exl3c4.STATUS.get(rc, rc)}")
    return s


# ------------------------------------------------------------------------------------------ one pass
def _ok(rc):
    if rc:
        raise RuntimeError(exl3c4.STATUS.get(rc, rc))


def run(s):
    kind = s["kind"]
    if kind == "layer":
        _ok(exl3c4.router_topk_scatter(s["logits"], s["k"], True, s["ids"], s["w"], s["st"], s["off"], None,
                                       s["row_of"], s["stream"]))
        _ok(exl3c4.launch_gather(s["op"], s["scratch"], s["ctr"], s["w"], s["row_of"], s["out"], s["stream"]))
        return {"out": s["out"].view(torch.float16), "y": s["y"].view(torch.bfloat16), "w": s["w"], "ids": s["ids"],
                "sorted_tok": s["st"], "offset": s["off"], "row_of": s["row_of"]}
    if kind == "expert":
        _ok(exl3c4.launch_ctr(s["op"], s["scratch"], s["ctr"], s["stream"]))
        return {"y": s["y"].view(torch.bfloat16)}
    if kind == "chain":
        for o in s["ops"]:
            _ok(exl3c4.launch(o, s["scratch"], s["stream"]))
        return {"xr": s["xr"].view(torch.float16), "h": s["h"].view(torch.float16), "y": s["y"].view(torch.bfloat16)}
    return {"gu": exl3c4.relayout(s["gu"], 2 * s["W"], s["H"], s["K"]),
            "dn": exl3c4.relayout(s["dn"], s["H"], s["W"], s["Kd"])}


# ------------------------------------------------------------------------------------------ what it cannot do without
def _live(case):
    """Experts that hold a row, by expectation."""
    E, M, k = case["n_expert"], case["tokens"], case["top_k"]
    if case["kind"] == "expert":
        return 1.0
    if not case["zipf"]:
        return E * (1.0 - (1.0 - k / E) ** M)
    pop = 1.0 / np.arange(1, E + 1) ** ZIPF_S
    return float(np.sum(1.0 - np.exp(-M * k * pop / pop.sum())))


def work(case):
    H, W = case["hidden"], float(np.mean(_widths(case)))
    K, Kd = case["bits"], case["dn_bits"]
    codes = (2 * W * H * K + H * W * Kd) / 8
    if case["kind"] == "load":
        return {"bytes": 2 * codes, "flops": 0}
    T = case["tokens"] * case["top_k"]
    weights = _live(case) * (codes + 2 * (H + H + 2 * W) + 2 * (W + H))     # live experts' codes and scale planes
    acts = case["tokens"] * H * 2                                            # the hidden states in
    if case["kind"] == "layer":
        acts += case["tokens"] * (case["n_expert"] * 4 + H * 2 + case["top_k"] * 8) + 8 * T
    elif case["kind"] == "expert":
        acts += T * H * 2
    else:
        acts += 2 * T * 2 * H * 2 + 2 * T * W * 2 + T * H * 2                # xr and h written, then read; y
    return {"bytes": weights + acts, "flops": 2.0 * T * 3 * H * W}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    # four times the 1.8e-3 that the outputs differ from 64 bits: the rotated input and h rounded to f16, y to bf16
    return {"rel": 7e-3}


# ------------------------------------------------------------------------------------------ in 64 bits
def _codebook(cb):
    """The f16 weight of each 16-bit state."""
    x = np.arange(65536, dtype=np.uint64)
    if cb == "mul1":
        h = (x * np.uint64(0x83DCD12D)) & np.uint64(0xFFFFFFFF)
        s = sum((h >> np.uint64(8 * i)) & np.uint64(255) for i in range(4)).astype(np.float64)
        kinv, kbias = (float(np.array([v], np.uint16).view(np.float16)[0]) for v in (0x1EEE, 0xC931))
        v = ((1024.0 + s) * kinv + kbias).astype(np.float16)
    else:
        h = x * np.uint64(0xCBAC1FED) if cb == "mcg" else x * np.uint64(89226354) + np.uint64(64248484)
        h = ((h & np.uint64(0x8FFF8FFF)) ^ np.uint64(0x3B603B60)).astype(np.uint32)
        lo, hi = (h & 0xFFFF).astype(np.uint16).view(np.float16), (h >> 16).astype(np.uint16).view(np.float16)
        v = (lo.astype(np.float64) + hi.astype(np.float64)).astype(np.float16)
    return torch.from_numpy(v.astype(np.float64)).cuda()


def _weights(record, rows, cols, bits, table):
    """W [rows, cols] of a stored record (include/exl3c4.h: blocks of one 32-row strip and 64 columns, 64 segments of
    `bits` words each, segment t + 2 s + 16 g the s-th eighth of tile (k tile 4 ks + g, n tile 2 nb + t))."""
    ns, ks = rows // 32, cols // 64
    w = record.view(torch.int32).to(torch.int64) & 0xFFFFFFFF
    w = w.view(ns, ks, 4, 8, 2, bits).permute(0, 4, 1, 2, 3, 5).reshape(2 * ns, 4 * ks, 8 * bits)
    nw = 8 * bits
    start = [(((p + 1) * bits - 16) % (32 * nw)) for p in range(256)]         # each position's 16-bit window
    i0 = torch.tensor([b // 32 for b in start], device=w.device)
    sh = torch.tensor([b % 32 for b in start], device=w.device)
    # a window starts in word i0 and ends there or in the next; both halves shifted into place without 64-bit overflow
    hi, lo = w[:, :, i0], w[:, :, (i0 + 1) % nw]
    state = torch.where(sh <= 16, hi >> (16 - sh).clamp(min=0),
                        (hi << (sh - 16).clamp(min=0)) | (lo >> (48 - sh).clamp(max=32))) & 0xFFFF
    pos = [[8 * (4 * (c & 7) + ((r & 7) >> 1)) + 4 * (c >> 3) + (r & 1) + 2 * (r >> 3) for r in range(16)]
           for c in range(16)]
    v = table[state][:, :, torch.tensor(pos, device=w.device)]                # [n tile, k tile, column, row]
    return v.permute(0, 2, 1, 3).reshape(rows, cols)


def _had(v):
    """The normalised Hadamard over each 128 columns."""
    h = torch.ones((1, 1), dtype=torch.float64, device=v.device)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (v.reshape(v.shape[0], -1, 128) @ (h / math.sqrt(128.0))).reshape(v.shape)


def _f64(bits16):
    return bits16.view(torch.float16).double()


def exact(case, seed):
    if case["kind"] == "load":
        return None
    s = _inputs(case, seed)
    M, k, E, H = case["tokens"], case["top_k"], case["n_expert"], case["hidden"]
    table, ws, x = _codebook(case["codebook"]), _widths(case), s["x_val"].double()
    if case["kind"] == "expert":
        ids = torch.full((M, 1), s["expert"], device="cuda")
    else:
        p = torch.softmax(s["logits"].double(), 1)
        w, ids = torch.sort(p, dim=1, descending=True, stable=True)
        w, ids = w[:, :k], ids[:, :k]
        w = w / w.sum(1, keepdim=True)
    flat = ids.reshape(-1)
    order = torch.argsort(flat, stable=True)                                  # the sorted rows' flat pairs
    T = M * k
    y = torch.zeros((T, H), dtype=torch.float64, device="cuda")
    xr = h_out = None
    if case["kind"] == "chain":
        xr = torch.zeros((T, 2 * H), dtype=torch.float64, device="cuda")
        h_out = torch.zeros((T, max(ws)), dtype=torch.float64, device="cuda")
    counts = torch.bincount(flat, minlength=E).tolist()
    at = 0
    for e in range(E):
        n = counts[e]
        if not n:
            continue
        rows = slice(at, at + n)
        at += n
        c, j = s["experts"][e % len(ws)], e // len(ws)
        W = c["W"]
        xe = x[order[rows] // k]
        g, u = _had(xe * _f64(c["suh"][j])), _had(xe * _f64(c["suh1"][j]))
        wg = _weights(c["gu"][j], 2 * W, H, case["bits"], table)
        svh = _f64(c["svh"][j])
        gate, up = _had(g @ wg[:W].T) * svh[:W], _had(u @ wg[W:].T) * svh[W:]
        h = _had(torch.nn.functional.silu(gate) * up * _f64(c["dn_suh"][j]))
        wd = _weights(c["dn"][j], H, W, case["dn_bits"], table)
        y[rows] = _had(h @ wd.T) * _f64(c["dn_svh"][j])
        if xr is not None:
            xr[rows, :H], xr[rows, H:], h_out[rows, :W] = g, u, h
    if case["kind"] == "chain":
        return {"xr": xr, "h": h_out, "y": y}
    if case["kind"] == "expert":
        return {"y": y}
    back = torch.empty_like(order)
    back[order] = torch.arange(T, device="cuda")
    out = (y[back].view(M, k, H) * w[:, :, None]).sum(1)
    return {"out": out, "y": y, "w": w, "ids": None, "sorted_tok": None, "offset": None, "row_of": None}

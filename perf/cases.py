"""Performance cases: what a program that serves GGUF models has this package do.

Each case is one pass of one kind of work over device-resident weights, called
through the public entry points (``vibeblade_amd.tensor`` and
``vibeblade_amd.sparse``):

* ``gemv``    -- linear layers of a decode step, one activation vector each
* ``ffn``     -- the decode step's FFN blocks (norm, gate/up, act, down, residual)
* ``sparse``  -- TurboSparse decode: neuron prediction on the device, then the
                 sparse FFN block over the predicted set
* ``gemm``    -- linear layers over a batch of tokens: speculative verify
                 (a few rows), chunked and full prefill (up to 1024 rows)
* ``moe``     -- mixture-of-experts FFN layers, from one token to a prefill chunk

``listed()`` names twelve fixed cases, ``draw(rng)`` gives others of the same
ranges.  A decode loop replays a captured graph over its layers, so the cases
of several small calls do (``graph``); prefill and one-off calls are eager.
``exact`` recomputes a case in float64 from the block bytes with plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from vibeblade_amd import ggml
from vibeblade_amd.sparse import DeviceEMAPredictor
from vibeblade_amd.tensor import (ACT_RELU2, ACT_SILU, DOWN_NEURON_MAJOR, QTensor, ffn_block, gemm, gemv,
                                  moe_grouped_ffn, sparse_ffn)

TYPES = {"Q4_0": ggml.GGML_TYPE_Q4_0, "Q8_0": ggml.GGML_TYPE_Q8_0, "Q4_K": ggml.GGML_TYPE_Q4_K,
         "Q5_K": ggml.GGML_TYPE_Q5_K, "Q6_K": ggml.GGML_TYPE_Q6_K}
# elements and bytes of one block
BLOCK = {"Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210)}
EPS = 1e-5
SPARSE_RATIO, THRESHOLD, DECAY, UPDATES = 0.1, 0.3, 0.1, 8


# ---- the cases -------------------------------------------------------------

def listed():
    return [
        # One key projection of a Q8_0 model, called by itself: the smallest call.
        {"name": "gemv_kv_q8_0", "kind": "gemv", "type": "Q8_0", "n": 1024, "k": 4096, "layers": 1, "graph": False},
        # The 4096 x 4096 attention projections (q and o) of eight layers in a decode step's graph.
        {"name": "decode_attn_q4_k", "kind": "gemv", "type": "Q4_K", "n": 4096, "k": 4096, "layers": 16, "graph": True},
        # The output head of a decode step.
        {"name": "decode_head_q6_k", "kind": "gemv", "type": "Q6_K", "n": 128256, "k": 4096, "layers": 1,
         "graph": False},
        # The FFN blocks of four layers of a Q4_K_M model in a decode step's graph, the residual running through.
        {"name": "decode_ffn_q4_k_m", "kind": "ffn", "type": "Q4_K", "down": "Q6_K", "h": 4096, "i": 14336,
         "layers": 4},
        # The same with predicted neuron sets (below the wanted tenth, so each prediction is topped up).
        {"name": "decode_sparse_q4_k", "kind": "sparse", "h": 4096, "i": 14336, "hot": 0.08, "layers": 4},
        # Speculative verify of eight tokens: the up projections of eight layers.
        {"name": "verify_up_q4_k_m8", "kind": "gemm", "type": "Q4_K", "m": 8, "n": 14336, "k": 4096, "x": "f16",
         "layers": 8, "graph": True},
        # Verify of five tokens through the output head (logits of every position).
        {"name": "verify_head_q6_k_m5", "kind": "gemm", "type": "Q6_K", "m": 5, "n": 128256, "k": 4096, "x": "f16",
         "layers": 1, "graph": False},
        # A prompt's ragged last chunk through the down projections of four layers.
        {"name": "chunk_down_q4_k_m100", "kind": "gemm", "type": "Q4_K", "m": 100, "n": 4096, "k": 14336, "x": "f16",
         "layers": 4, "graph": True},
        # A full prefill chunk through one up projection.
        {"name": "prefill_up_q4_k_m512", "kind": "gemm", "type": "Q4_K", "m": 512, "n": 14336, "k": 4096, "x": "f16",
         "layers": 1, "graph": False},
        # A long ragged prompt through a Q6_K down projection, the activations as the FFN leaves them (fp32).
        {"name": "prefill_down_q6_k_m777", "kind": "gemm", "type": "Q6_K", "m": 777, "n": 4096, "k": 14336, "x": "f32",
         "layers": 1, "graph": False},
        # An eight-expert MoE layer over a batch of 16 decode or verify tokens.
        {"name": "moe_verify_t16", "kind": "moe", "type": "Q4_K", "down": "Q4_K", "experts": 8, "topk": 2, "t": 16,
         "h": 4096, "i": 14336},
        # The same layer of a Q4_K_M file over a ragged prefill chunk.
        {"name": "moe_prefill_t500", "kind": "moe", "type": "Q4_K", "down": "Q6_K", "experts": 8, "topk": 2, "t": 500,
         "h": 4096, "i": 14336},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_256(rng, lo, hi):
    """A multiple of 256, log-uniform."""
    return max(lo, min(hi, 256 * _log_int(rng, lo // 256, hi // 256)))


def draw(rng):
    kind = rng.choice(["gemv", "ffn", "sparse", "gemm", "gemm", "gemm", "moe", "moe"])
    kinds = ["Q4_K", "Q4_K", "Q6_K", "Q8_0", "Q5_K", "Q4_0"]
    if kind == "gemv":
        n, k = _log_int(rng, 512, 32768), _log_256(rng, 1024, 14336)
        return {"kind": kind, "type": rng.choice(kinds), "n": n, "k": k, "layers": rng.randint(1, 8),
                "graph": rng.random() < 0.7}
    if kind == "ffn":
        return {"kind": kind, "type": rng.choice(["Q4_K", "Q8_0", "Q6_K", "Q5_K"]),
                "down": rng.choice(["Q4_K", "Q6_K", "Q8_0"]), "h": _log_256(rng, 1024, 8192),
                "i": _log_256(rng, 2048, 16384), "layers": rng.randint(1, 4)}
    if kind == "sparse":
        return {"kind": kind, "h": _log_256(rng, 2048, 4096), "i": _log_256(rng, 4096, 16384),
                "hot": round(rng.uniform(0.05, 0.15), 3), "layers": rng.randint(1, 4)}
    if kind == "gemm":
        m, n, k = _log_int(rng, 2, 1024), _log_int(rng, 512, 32768), _log_256(rng, 1024, 14336)
        n = min(n, (64 << 20) // k)
        return {"kind": kind, "type": rng.choice(kinds), "m": m, "n": n, "k": k,
                "x": rng.choice(["f16", "f16", "f32"]), "layers": 4 if m <= 128 else 1, "graph": m <= 128}
    experts = rng.choice([4, 8, 8, 16, 32])
    h, i = _log_256(rng, 1024, 4096), _log_256(rng, 512, 14336)
    while experts * h * i > 8 * 4096 * 14336:
        i = max(256, i // 512 * 256)
    return {"kind": "moe", "type": rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q8_0"]), "down": rng.choice(["Q4_K", "Q6_K"]),
            "experts": experts, "topk": rng.choice([1, 2, 2, 4]), "t": _log_int(rng, 1, 250), "h": h, "i": i}


# ---- GGUF blocks of roughly N(0, 0.02) weights --------------------------------

def _bytes(g, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g)


def _codes(g, rows, count, levels, middle, spread):
    """Codes 0 .. levels-1 as a quantizer leaves them: normal around `middle`."""
    z = torch.erfinv((torch.arange(256, dtype=torch.float64) + 0.5) / 128 - 1) * math.sqrt(2)
    lut = (middle + spread * z).round().clamp(0, levels - 1).to(torch.uint8).cuda()
    return torch.cat([lut[_bytes(g, min(1 << 17, rows - r), count).to(torch.int32)]
                      for r in range(0, rows, 1 << 17)])


def _half(g, rows, mean):
    """One fp16 scale per block near `mean`, as two bytes."""
    v = mean * (0.9 + 0.2 * torch.rand(rows, 1, device="cuda", generator=g))
    return v.to(torch.float16).view(torch.uint8)


def _pack_scales(sc, mn):
    """Eight 6-bit scales and minimums of a K block in 12 bytes."""
    low = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6)], 1)
    return torch.cat([low, (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)


def _blocks(g, kind, rows, k):
    """Random block bytes of a rows x k tensor."""
    nb = rows * (k // BLOCK[kind][0])
    if kind == "Q4_0":
        q = _codes(g, nb, 32, 16, 8, 2.7)
        return torch.cat([_half(g, nb, 0.0074), q[:, :16] | (q[:, 16:] << 4)], 1).reshape(-1)
    if kind == "Q8_0":
        q = _codes(g, nb, 32, 256, 128, 45).clamp(min=1) ^ 128
        return torch.cat([_half(g, nb, 0.02 / 45), q], 1).reshape(-1)
    if kind == "Q6_K":
        q = _codes(g, nb, 256, 64, 32, 11).view(nb, 2, 4, 32)  # half, quarter, element
        ql = torch.cat([(q[:, :, 0:2] & 15) | ((q[:, :, 2:4] & 15) << 4)], 2).reshape(nb, 128)
        qh = ((q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6))
        sc = _bytes(g, nb, 16) % 48 + 80
        sc = torch.where(_bytes(g, nb, 16) < 128, sc, 256 - sc.to(torch.int32)).to(torch.uint8)  # int8, either sign
        return torch.cat([ql, qh.reshape(nb, 64), sc, _half(g, nb, 0.02 / 11 / 104)], 1).reshape(-1)
    levels = 16 if kind == "Q4_K" else 32
    q = _codes(g, nb, 256, levels, (levels - 1) / 2, 0.19 * levels).view(nb, 4, 2, 32)  # chunk, sub-block, element
    sc = _bytes(g, nb, 8) % 28 + 32
    mn = sc + _bytes(g, nb, 8) % 4
    step = 0.02 / (0.19 * levels) / 46
    head = [_half(g, nb, step), _half(g, nb, step * (levels - 1) / 2), _pack_scales(sc, mn)]
    if kind == "Q5_K":
        hi = q >> 4
        head.append(sum(hi[:, c, s] << (2 * c + s) for c in range(4) for s in range(2)))
    return torch.cat(head + [((q[:, :, 0] & 15) | ((q[:, :, 1] & 15) << 4)).reshape(nb, 128)], 1).reshape(-1)


def _decode64(raw, kind, rows, k):
    """The tensor's values in float64, by the GGUF formulas."""
    b = raw.view(-1, BLOCK[kind][1])
    nb = b.shape[0]

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    if kind == "Q4_0":
        q = torch.cat([b[:, 2:18] & 15, b[:, 2:18] >> 4], 1).double()
        return (half(0) * (q - 8)).view(rows, k)
    if kind == "Q8_0":
        return (half(0) * b[:, 2:34].contiguous().view(torch.int8).double()).view(rows, k)
    if kind == "Q6_K":
        ql, qh = b[:, :128].reshape(nb, 2, 2, 32), b[:, 128:192].reshape(nb, 2, 32)
        q = torch.stack([(ql[:, :, t % 2] >> (4 * (t // 2)) & 15) | ((qh >> (2 * t) & 3) << 4) for t in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = (q.double() - 32).view(nb, 16, 16) * (half(208) * sc)[:, :, None]
        return w.view(rows, k)
    p = b[:, 4:16]
    sc = torch.cat([p[:, :4] & 63, (p[:, 8:] & 15) | ((p[:, :4] >> 6) << 4)], 1).double()
    mn = torch.cat([p[:, 4:8] & 63, (p[:, 8:] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1).double()
    qs = b[:, -128:].reshape(nb, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2)
    if kind == "Q5_K":
        qh = b[:, 16:48]
        hi = torch.stack([torch.stack([qh >> (2 * c + s) & 1 for s in range(2)], 1) for c in range(4)], 1)
        q = q | (hi << 4)
    w = (half(0) * sc)[:, :, None] * q.reshape(nb, 8, 32).double() - (half(2) * mn)[:, :, None]
    return w.view(rows, k)


# ---- inputs ----------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(shape, dtype=torch.float32, device="cuda", generator=g)


def _mat(g, kind, rows, k):
    return QTensor(_blocks(g, kind, rows, k), TYPES[kind], rows, k)


def _batch(g, case):
    """Activations with one value in a thousand twenty times as large."""
    x = _normal(g, case["m"], case["k"])
    x = torch.where(torch.rand(x.shape, device="cuda", generator=g) < 0.001, 20 * x, x)
    return x.to(torch.float16) if case["x"] == "f16" else x


def _masks(g, case):
    """UPDATES observed neuron sets: hot neurons nearly always, the others now and then."""
    i = case["i"]
    often = torch.where(torch.rand(i, device="cuda", generator=g) < case["hot"], 0.97, 0.03)
    return [torch.rand(i, device="cuda", generator=g) < often for _ in range(UPDATES)]


def _inputs(case, seed):
    """What the seed gives: weights, activations and observations."""
    g, kind = _generator(seed), case["kind"]
    if kind in ("gemv", "gemm"):
        x = _normal(g, case["k"]) if kind == "gemv" else _batch(g, case)
        return {"x": x, "w": [_mat(g, case["type"], case["n"], case["k"]) for _ in range(case["layers"])]}
    h, i = case["h"], case["i"]
    if kind == "moe":
        e, t = case["experts"], case["t"]
        return {"x": _normal(g, t, h), "logits": _normal(g, t, e),
                "gate": [_mat(g, case["type"], i, h) for _ in range(e)],
                "up": [_mat(g, case["type"], i, h) for _ in range(e)],
                "down": [_mat(g, case["down"], h, i) for _ in range(e)]}
    made = {"x": _normal(g, h), "layers": []}
    for _ in range(case["layers"]):
        layer = {"norm": 1 + 0.1 * _normal(g, h)}
        if kind == "ffn":
            layer["gate"], layer["up"] = _mat(g, case["type"], i, h), _mat(g, case["type"], i, h)
            layer["down"] = _mat(g, case["down"], h, i)
        else:
            layer["gate"], layer["up"], layer["down"] = (_mat(g, "Q4_K", i, h) for _ in range(3))
            layer["masks"] = _masks(g, case)
        made["layers"].append(layer)
    return made


# ---- the calls ---------------------------------------------------------------------

def _pass(case, s):
    """One pass through the entry points."""
    kind = case["kind"]
    if kind == "gemv":
        return [gemv(w, s["x"]) for w in s["w"]]
    if kind == "gemm":
        return [gemm(w, s["x"]) for w in s["w"]]
    if kind == "moe":
        return moe_grouped_ffn(s["gate"], s["up"], s["down"], s["x"], s["logits"], case["topk"])
    x, out = s["x"], []
    for n, layer in enumerate(s["layers"]):
        if kind == "ffn":
            x = ffn_block(layer["gate"], layer["up"], layer["down"], x, norm_w=layer["norm"], eps=EPS, act=ACT_SILU)
            out.append(x)
        else:
            active, count, mask = s["predictor"].predict_active(n)
            x = sparse_ffn(layer["gate"], layer["up"], layer["down"], x, active, act=ACT_RELU2,
                           down_layout=DOWN_NEURON_MAJOR, norm_w=layer["norm"], eps=EPS, residual=True, count=count)
            out.append([x, mask, count])
    return out


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "sparse":
        s["predictor"] = DeviceEMAPredictor(case["i"], case["layers"], ema_decay=DECAY, sparse_ratio=SPARSE_RATIO,
                                            activation_threshold=THRESHOLD)
        for n, layer in enumerate(s["layers"]):
            for m in layer.pop("masks"):
                s["predictor"].update(n, m)
    s["case"], s["graph"] = case, None
    if case.get("graph", case["kind"] in ("ffn", "sparse")):
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _pass(case, s)
        torch.cuda.current_stream().wait_stream(stream)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["out"] = _pass(case, s)
    return s


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return _pass(state["case"], state)


# ---- what a pass cannot do without ---------------------------------------------------

def _nbytes(kind, rows, k):
    return rows * (k // BLOCK[kind][0]) * BLOCK[kind][1]


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        m, n, k = case.get("m", 1), case["n"], case["k"]
        x = m * k * (2 if case.get("x") == "f16" else 4)
        return {"bytes": case["layers"] * (_nbytes(case["type"], n, k) + 4 * m * n) + x,
                "flops": case["layers"] * 2 * m * n * k}
    h, i = case["h"], case["i"]
    if kind == "ffn":
        one = 2 * _nbytes(case["type"], i, h) + _nbytes(case["down"], h, i) + 12 * h
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 6 * h * i}
    if kind == "sparse":
        # hot neurons pass the threshold; fewer than the wanted share are topped up to it
        active = max(case["hot"], SPARSE_RATIO) * i
        one = 3 * active * _nbytes("Q4_K", 1, h) + 12 * h + 4 * i + i + 4
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 6 * h * active}
    t, e, topk = case["t"], case["experts"], case["topk"]
    hit = e * (1 - (1 - topk / e) ** t)  # experts that some token takes
    one = 2 * _nbytes(case["type"], i, h) + _nbytes(case["down"], h, i)
    return {"bytes": hit * one + 8 * t * h + 4 * t * e + 8 * t * topk, "flops": t * topk * 6 * h * i}


def tolerance(case):
    """About four times what the arithmetic of each path shows against float64: fixed-point activations of 15
    bits in the matrix-vector kernels, fp16 operands in the matrix products and fp16 hidden rows in the MoE."""
    rel = {"gemv": 2e-4, "ffn": 8e-4, "sparse": 6e-4, "gemm": 3e-3, "moe": 5e-3}[case["kind"]]
    return {"rel": rel, "max": 40 * rel}


# ---- the same in float64 -----------------------------------------------------------------

def _dense(w):
    """A weight's values in float64 by chunks of rows: (first row, chunk)."""
    kind = next(name for name, t in TYPES.items() if t == w.qtype)
    step = max(1, (1 << 27) // w.k)
    for r in range(0, w.rows, step):
        rows = min(step, w.rows - r)
        yield r, _decode64(w.data[r:r + rows].reshape(-1), kind, rows, w.k)


def _times(x, w):
    """x (.., k) times the rows of w, in float64."""
    return torch.cat([x.double() @ d.T for _, d in _dense(w)], -1)


def _normed(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean() + EPS) * w.double()


def _predicted(masks, i):
    """The predictor's set after the observations: float32 averages, ties to the lowest index."""
    a = np.float32(DECAY)
    rest = np.float32(1.0 - DECAY)
    p = np.zeros(i, np.float32)
    for m in masks:
        p = a * m.cpu().numpy().astype(np.float32) + rest * p
    k = min(i, max(1, int(i * SPARSE_RATIO)))
    mask = p >= np.float32(THRESHOLD)
    mask[np.argsort(-p, kind="stable")[:k]] = True
    return torch.from_numpy(mask).cuda()


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind in ("gemv", "gemm"):
        return [_times(s["x"], w) for w in s["w"]]
    if kind == "moe":
        logits = s["logits"].double().clamp(-50, 50)
        p, at = torch.softmax(logits, 1).topk(case["topk"], 1)
        p = p / p.sum(1, keepdim=True)
        y = torch.zeros(s["x"].shape, dtype=torch.float64, device="cuda")
        for e in range(case["experts"]):
            rows, slot = torch.where(at == e)
            if len(rows):
                x = s["x"][rows]
                g, u = _times(x, s["gate"][e]), _times(x, s["up"][e])
                y.index_add_(0, rows, _times(g * torch.sigmoid(g) * u, s["down"][e]) * p[rows, slot][:, None])
        return y, None, p
    x, out = s["x"], []
    for layer in s["layers"]:
        n = _normed(x, layer["norm"])
        g, u = _times(n, layer["gate"]), _times(n, layer["up"])
        if kind == "ffn":
            x = x.double() + _times(g * torch.sigmoid(g) * u, layer["down"])
            out.append(x)
        else:
            act = torch.relu(g) * torch.relu(u) * _predicted(layer["masks"], case["i"])
            x = x.double() + sum(act[r:r + len(d)] @ d for r, d in _dense(layer["down"]))
            out.append([x, None, None])
    return out

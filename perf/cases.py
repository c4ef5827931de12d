"""Timing cases of the library's main path: what a program that uses it has it
do, through its public entry points.

A case is a dict of plain values with a "kind":

  products   cq.gemms_dev of one or several matrices on one input: one
             token's projections (1 row) up to long batches of frames
  exact      products of an Exact view (the nibble tables in float32, which
             the text model loads by default) or of its Dense form
  plan       cq.Batch: every matrix of a sweep, one activation each
  memory     a cross-attention memory: int8-input K and V linears over the
             encoder's frames (needle.ApplyShared), then QuantizeRows per head
  attend     AttendInt8Spans: decode rows of many streams, beams sharing one
             memory, prompts of many rows
  hadamard   HadamardMLP.Forward, the Monarch FFN
  mhc        one mHC layer around a block: RMSUnit, the three phi products,
             the heads with the Sinkhorn, the lane mix
  decode     whole greedy decode steps of the synthetic decoder, replayed
             from a captured graph

The library's results are bit for bit the arithmetic it documents (exact
integer sums, every float operation in a fixed order), so the tolerance is
"exact" wherever that holds; HadamardMLP and the Dense products are float32
sums in the kernel's own order and have a relative one.
"""

import importlib
import math

import numpy as np
import torch

_pkg = importlib.import_module("go-whistle_amd")
cq, needle, synth = _pkg.cq, _pkg.needle, _pkg.synth
_decoder = importlib.import_module("go-whistle_amd.decoder")

SWEEP = [(512, 512), (2048, 512), (512, 2048), (16384, 512)]  # the GEMV benchmark's shapes, each at 4 and 2 bits


def listed():
    return [
        # One token's q/k/v/gate projections in a decode step run product by
        # product: the smallest call, all latency and launches.
        {"name": "token_qkvg", "kind": "products", "mats": "512x512x4,512x512x4,512x512x4,512x512x4", "rows": 1,
         "group": 128},
        # An FFN-up product over a long batch of encoder frames: the largest
        # single product.
        {"name": "frames_12000", "kind": "products", "mats": "2048x512x4", "rows": 12000, "group": 128},
        # A prompt's product on an Exact view, the text model's default.
        {"name": "exact_prompt_375", "kind": "exact", "mats": "2048x512x4", "rows": 375, "group": 128, "dense": False},
        # The GEMV sweep: every matrix once with its own activation, as a
        # batch plan (a memory-bound pass over the weights).
        {"name": "gemv_plan", "kind": "plan", "copies": 8, "rows": 1},
        # The cross memory of one long utterance: K and V of 8 heads (48 and
        # 64 wide) over 1500 frames, quantised per head.
        {"name": "memory_1500", "kind": "memory", "frames": 1500, "heads": 8, "qk": 48, "vd": 64, "bits": 2,
         "act8": True},
        # Self-attention of 256 streams at different positions, one row each.
        {"name": "attend_self_256", "kind": "attend", "batch": 256, "t": 1, "heads": 8, "kv_heads": 8, "qk": 64,
         "vd": 64, "keys": 448, "spans": "ragged", "shared": False, "quant_q": True},
        # Cross-attention of 5 beams over the 375 frames of their utterance.
        {"name": "attend_beams_5", "kind": "attend", "batch": 5, "t": 1, "heads": 8, "kv_heads": 8, "qk": 48, "vd": 64,
         "keys": 375, "spans": "full", "shared": True, "quant_q": True},
        # A prompt's rows attending causally over a grouped-query cache.
        {"name": "attend_prompt_4x96", "kind": "attend", "batch": 4, "t": 96, "heads": 8, "kv_heads": 2, "qk": 48,
         "vd": 64, "keys": 448, "spans": "causal", "shared": False, "quant_q": True},
        # The Monarch FFN over the frames of a 30-second clip.
        {"name": "hadamard_375", "kind": "hadamard", "rows": 375, "na": 16, "nb": 32, "dim": 512, "rank": 8},
        # The mHC layer around a block over the same frames.
        {"name": "mhc_375", "kind": "mhc", "rows": 375, "lanes": 4, "dim": 512},
        # Greedy decoding of one stream with every feature of the reference's
        # step (8 tokens), and of 256 streams of the benchmark's decoder (4).
        {"name": "decode_features_b1", "kind": "decode", "batch": 1, "features": True, "steps": 8},
        {"name": "decode_b256", "kind": "decode", "batch": 256, "features": False, "steps": 4},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# Output and input widths of the configurations (projections, FFN, phi,
# tied heads, the encoder's stem) and sizes that are no multiple of anything.
WIDTHS = [(96, 512), (384, 512), (512, 512), (1024, 512), (2048, 512), (8199, 512), (16384, 512), (512, 1280),
          (512, 2048), (128, 2048), (777, 512), (300, 500), (1001, 1000)]


def draw(rng):
    kind = rng.choice(["products", "products", "exact", "plan", "memory", "attend", "attend", "attend", "hadamard", "mhc",
                       "decode"])
    if kind in ("products", "exact"):
        out, inp = rng.choice(WIDTHS)
        n = rng.choice([1, 1, 2, 4])
        if n * out > 16384:
            n = 1
        bits = rng.choice([2, 4])
        cap = (12000 if kind == "products" else 3000) * 2048 * 512 // (n * out * inp)
        rows = _log_int(rng, 1, min(12000 if kind == "products" else 3000, cap))
        case = {"kind": kind, "mats": ",".join([f"{out}x{inp}x{bits}"] * n), "rows": rows,
                "group": rng.choice([128, 128, 128, 128, 64, 32, 256])}
        if kind == "exact":
            case["dense"] = rng.random() < 0.4
        return case
    if kind == "plan":
        return {"kind": kind, "copies": rng.randint(1, 8), "rows": 1}
    if kind == "memory":
        return {"kind": kind, "frames": _log_int(rng, 60, 3000), "heads": rng.choice([2, 8]), "qk": rng.choice([48, 64]),
                "vd": 64, "bits": rng.choice([2, 4]), "act8": rng.random() < 0.7}
    if kind == "attend":
        qk, vd = rng.choice([(48, 64), (64, 64), (64, 64), (64, 128)])
        spans = rng.choice(["ragged", "full", "causal"])
        heads = 8
        kv_heads = rng.choice([2, 8])
        if spans == "causal":
            t = _log_int(rng, 2, 128)
            batch = rng.randint(1, max(1, 512 // t))
            keys = rng.choice([200, 448])
        else:
            t = 1
            batch = _log_int(rng, 1, 256)
            keys = _log_int(rng, 16, 1500 if spans == "full" and batch <= 64 else 448)
        return {"kind": kind, "batch": batch, "t": t, "heads": heads, "kv_heads": kv_heads, "qk": qk, "vd": vd,
                "keys": keys, "spans": spans, "shared": spans == "full" and rng.random() < 0.5,
                "quant_q": rng.random() < 0.8}
    if kind == "hadamard":
        na, nb, dim = rng.choice([(16, 32, 512), (16, 32, 500), (16, 16, 256), (24, 32, 768), (32, 32, 1024)])
        return {"kind": kind, "rows": _log_int(rng, 1, 3000), "na": na, "nb": nb, "dim": dim, "rank": rng.choice([8, 16])}
    if kind == "mhc":
        return {"kind": kind, "rows": _log_int(rng, 1, 3000), "lanes": rng.choice([2, 4, 4, 4]),
                "dim": rng.choice([512, 512, 256, 384, 500])}
    features = rng.random() < 0.5
    return {"kind": "decode", "batch": _log_int(rng, 1, 128 if features else 256), "features": features,
            "steps": rng.randint(1, 4)}


# ---- inputs ----------------------------------------------------------------


def _mats(case):
    return [tuple(int(v) for v in m.split("x")) for m in case["mats"].split(",")]


def _packs(g, shapes, group):
    """Matrices of one model: a codebook per index width, as a weight file
    holds them, N(0, 0.05) levels and uniform indices."""
    books = {b: np.sort(g.standard_normal(1 << b) * 0.05).astype(np.float32) for b in (2, 4)}
    packs = []
    for out, inp, bits in shapes:
        p = synth.random_packed(g, out, inp, group, bits, sigma=0.05)
        p.Codebook = books[bits]
        packs.append(p)
    return packs


def _plan_shapes(case):
    return [(o, i, b) for _ in range(case["copies"]) for b in (4, 2) for o, i in SWEEP]


def _host(case, seed):
    """The case's inputs on the host, from the seed alone."""
    g = np.random.Generator(np.random.PCG64(seed))
    kind = case["kind"]
    if kind in ("products", "exact"):
        shapes = _mats(case)
        packs = _packs(g, shapes, case["group"])
        return packs, g.standard_normal((case["rows"], shapes[0][1]), dtype=np.float32)
    if kind == "plan":
        shapes = _plan_shapes(case)
        packs = _packs(g, shapes, 128)
        return packs, [g.standard_normal((case["rows"], i), dtype=np.float32) for _, i, _ in shapes]
    if kind == "memory":
        h = case["heads"]
        packs = _packs(g, [(h * case["qk"], 512, case["bits"]), (h * case["vd"], 512, case["bits"])], 128)
        return packs, g.standard_normal((case["frames"], 512), dtype=np.float32)
    if kind == "attend":
        return _attend_host(case, g)
    if kind == "hadamard":
        na, nb, dim, rank, n = case["na"], case["nb"], case["dim"], case["rank"], case["na"] * case["nb"]
        w = {k: (1 + 0.2 * g.standard_normal(n)).astype(np.float32) for k in ("d1", "d2", "d3", "d4")}
        w["b2"] = (0.1 * g.standard_normal(n)).astype(np.float32)
        for s in (1, 2, 3):
            w[f"w{s}a"] = (g.standard_normal((na, na)) / math.sqrt(na)).astype(np.float32)
            w[f"w{s}b"] = (g.standard_normal((nb, nb)) / math.sqrt(nb)).astype(np.float32)
        w["cond_v"] = (g.standard_normal((dim, rank)) / math.sqrt(dim)).astype(np.float32)
        w["cond_u"] = (0.5 * g.standard_normal((rank, n))).astype(np.float32)
        w["p1"], w["p2"] = g.permutation(n).astype(np.int32), g.permutation(n).astype(np.int32)
        return w, (g.standard_normal((case["rows"], dim)) * 1.5).astype(np.float32)
    n, dim, rows = case["lanes"], case["dim"], case["rows"]  # mhc
    packs = _packs(g, [(n, n * dim, 4), (n, n * dim, 4), (n * n, n * dim, 4)], 128)
    aff = np.concatenate([0.5 + g.uniform(0, 0.5, 3), g.standard_normal(n) * 0.5, np.full(n, -4.0),
                          g.standard_normal(n) * 0.5, np.full(n, -4.0), g.standard_normal(n * n) * 0.5])
    aff[3 + n], aff[3 + 3 * n] = 4, 0  # the layer's own lane
    return (packs, aff.astype(np.float32), g.standard_normal((rows, n, dim), dtype=np.float32),
            g.standard_normal((rows, dim), dtype=np.float32))


# int8 codes as QuantizeRow leaves N(0, 1) heads: a standard deviation of about
# 48 under a bound of 127, drawn through a table of 256 quantiles.
_CODES = np.clip(np.rint(48 * torch.special.ndtri(torch.from_numpy((np.arange(256) + 0.5) / 256)).numpy()), -127,
                 127).astype(np.int8)


def _attend_host(case, g):
    b, t, h, kvh, qk, vd, keys = (case[k] for k in ("batch", "t", "heads", "kv_heads", "qk", "vd", "keys"))
    caches = 1 if case["shared"] else b
    kc, vc = kvh * qk, kvh * vd
    codes = lambda cols: _CODES[g.integers(0, 256, (caches, keys, cols), dtype=np.uint8)]
    scales = lambda: g.uniform(0.015, 0.03, (caches, keys, kvh)).astype(np.float32)
    kq, vq, ks, vs = codes(kc), codes(vc), scales(), scales()
    spans = np.zeros((b, t, 4), np.int32)
    if case["spans"] == "full":  # a whole memory
        spans[:, :, 3] = keys
    elif case["spans"] == "ragged":  # streams at their own positions
        spans[:, :, 3] = g.integers(1, keys + 1, (b, 1))
    else:  # row i of a prompt at its stream's offset sees the keys up to its own
        t0 = g.integers(0, max(1, keys - t + 1), b)
        spans[:, :, 3] = t0[:, None] + np.arange(t)[None, :] + 1
    q = g.standard_normal((b, t, h * qk), dtype=np.float32)
    return q, kq, ks, vq, vs, spans


def _cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _prepare_decode(case, seed)
    if kind in ("products", "exact", "memory", "plan"):
        packs, x = _host(case, seed)
        ms = [cq.New(p) for p in packs]
        if kind == "plan":
            xs = [_cuda(v) for v in x]
            ys = [_empty(case["rows"], p.Out) for p in packs]
            return {"ys": ys, "plan": cq.Batch(ms, ys, xs, [case["rows"]] * len(ms))}
        if kind == "exact":
            ms = [m.Dense() if case["dense"] else m.Exact() for m in ms]
        rows = case.get("rows", case.get("frames"))
        st = {"ms": ms, "x": _cuda(x), "rows": rows, "ys": [_empty(rows, p.Out) for p in packs]}
        if kind == "memory":
            st["ls"] = [needle.Linear(m, case["act8"]) for m in ms]
            st["widths"] = (case["qk"], case["vd"])
            st["q8"] = [_empty(rows, p.Out, dtype=torch.int8) for p in packs]
            st["s8"] = [_empty(rows, case["heads"]) for _ in packs]
        return st
    if kind == "attend":
        q, kq, ks, vq, vs, spans = _host(case, seed)
        caches, keys, kvh = ks.shape
        cols = max(kq.shape[2], vq.shape[2])  # the caches of K and V lie one stride apart
        pad = lambda a: np.pad(a.reshape(caches, -1), ((0, 0), (0, keys * cols - a[0].size)))
        stride = 0 if case["shared"] else 1
        return {"out": _empty(case["batch"], case["t"], case["heads"] * case["vd"]), "q": _cuda(q), "kq": _cuda(pad(kq)),
                "ks": _cuda(ks), "vq": _cuda(pad(vq)), "vs": _cuda(vs), "spans": _cuda(spans), "case": dict(case),
                "kv_stride": stride * keys * cols, "s_stride": stride * keys * kvh}
    if kind == "hadamard":
        w, x = _host(case, seed)
        return {"mlp": needle.HadamardMLP(w), "x": _cuda(x), "rows": case["rows"], "out": _empty(*x.shape)}
    packs, aff, stream, block_out = _host(case, seed)
    n, dim, rows = case["lanes"], case["dim"], case["rows"]
    return {"phi": [cq.New(p) for p in packs], "aff": _cuda(aff), "stream": _cuda(stream), "block_out": _cuda(block_out),
            "nx": _empty(rows, n * dim), "logits": [_empty(rows, p.Out) for p in packs],
            "h": [_empty(rows, n), _empty(rows, n), _empty(rows, n * n)], "u": _empty(rows, dim),
            "out": _empty(rows, n, dim), "shape": (rows, n, dim)}


def _prepare_decode(case, seed):
    cfg = _decoder.DecoderConfig.whistle() if case["features"] else _decoder.DecoderConfig()
    d = _decoder.Decoder(_decoder.make_model(seed, cfg), case["batch"])
    d.set_memory(seed, generator="device")
    tokens = np.random.Generator(np.random.PCG64(seed)).integers(0, cfg.vocab, case["batch"]).astype(np.int32)
    d.reset(tokens)
    return {"decoder": d, "graph": d.capture(), "tokens": tokens, "steps": case["steps"]}


# ---- one pass --------------------------------------------------------------


def run(state):
    if "plan" in state:
        state["plan"].run()
        return state["ys"]
    if "decoder" in state:
        d, graph = state["decoder"], state["graph"]
        d.reset(state["tokens"])
        for _ in range(state["steps"]):
            graph.replay()
        return {"logits": d.logits, "tokens": d.tok}
    if "mlp" in state:
        state["mlp"].forward_dev(state["out"], state["x"], state["rows"])
        return state["out"]
    if "spans" in state:
        c = state["case"]
        needle.attend_int8_dev(state["out"], state["q"], c["t"], c["heads"], state["kq"], state["ks"],
                               c["kv_heads"] * c["qk"], c["qk"], state["vq"], state["vs"], c["kv_heads"] * c["vd"],
                               c["vd"], state["spans"], c["keys"], math.sqrt(c["qk"]), c["quant_q"], batch=c["batch"],
                               kv_stride=state["kv_stride"], s_stride=state["s_stride"])
        return state["out"]
    if "phi" in state:
        rows, n, dim = state["shape"]
        stream, (pre, post, res), u = state["stream"], state["h"], state["u"]
        needle.rms_unit_dev(state["nx"], stream, rows, n * dim)
        cq.gemms_dev(state["phi"], state["logits"], state["nx"], rows)
        needle.mhc_heads_dev(pre, post, res, u, *state["logits"], stream, rows, n, dim, state["aff"])
        needle.mhc_mix_dev(state["out"], stream, res, post, state["block_out"], u, rows, n, dim)
        return {"nx": state["nx"], "pre": pre, "post": post, "res": res, "u": u, "out": state["out"]}
    if "ls" in state:
        needle.ApplyShared(state["ys"], state["x"], state["rows"], *state["ls"])
        for y, q8, s8, width in zip(state["ys"], state["q8"], state["s8"], state["widths"]):
            needle.quantize_rows_dev(q8, s8, y, state["rows"], y.shape[1], width)
        return {"kv": state["ys"], "codes": state["q8"], "scales": state["s8"]}
    cq.gemms_dev(state["ms"], state["ys"], state["x"], state["rows"])
    return state["ys"]


# ---- what a pass cannot do without -----------------------------------------


def _matrix_bytes(out, inp, bits, group):
    groups = -(-inp // group)
    return out * groups * (group * bits // 8 + 2)


def work(case):
    kind = case["kind"]
    if kind in ("products", "exact"):
        shapes, rows = _mats(case), case["rows"]
        out = sum(o for o, _, _ in shapes)
        return {"bytes": sum(_matrix_bytes(o, i, b, case["group"]) for o, i, b in shapes) +
                4 * rows * (shapes[0][1] + out), "flops": 2 * rows * out * shapes[0][1]}
    if kind == "plan":
        shapes, rows = _plan_shapes(case), case["rows"]
        return {"bytes": sum(_matrix_bytes(o, i, b, 128) + 4 * rows * (o + i) for o, i, b in shapes),
                "flops": sum(2 * rows * o * i for o, i, _ in shapes)}
    if kind == "memory":
        outs, f = [case["heads"] * case["qk"], case["heads"] * case["vd"]], case["frames"]
        return {"bytes": sum(_matrix_bytes(o, 512, case["bits"], 128) for o in outs) + 4 * f * 512 +
                5 * f * sum(outs) + 8 * f * case["heads"], "flops": 2 * f * sum(outs) * 512}
    if kind == "attend":
        b, t, h, kvh, qk, vd, keys = (case[k] for k in ("batch", "t", "heads", "kv_heads", "qk", "vd", "keys"))
        # keys a row sees, and keys of a cache that any row sees, on average
        seen = {"full": keys, "ragged": (keys + 1) / 2, "causal": (keys + 1) / 2}[case["spans"]]
        held = {"full": keys, "ragged": (keys + 1) / 2, "causal": (keys + t) / 2}[case["spans"]]
        caches = 1 if case["shared"] else b
        return {"bytes": int(caches * held * kvh * (qk + vd + 8) + 4 * b * t * (h * (qk + vd) + 4)),
                "flops": int(2 * b * t * h * seen * (qk + vd))}
    if kind == "hadamard":
        n, na, nb, rank, rows = case["na"] * case["nb"], case["na"], case["nb"], case["rank"], case["rows"]
        return {"bytes": 8 * rows * case["dim"] + 4 * (3 * (na * na + nb * nb) + rank * (n + case["dim"]) + 7 * n),
                "flops": rows * (3 * 2 * n * (na + nb) + 2 * rank * (n + case["dim"]))}
    if kind == "mhc":
        n, dim, rows = case["lanes"], case["dim"], case["rows"]
        phi = 2 * n + n * n
        return {"bytes": _matrix_bytes(phi, n * dim, 4, 128) + 4 * rows * (3 * n * dim + 2 * dim + phi),
                "flops": rows * (2 * phi * n * dim + 2 * n * dim + 2 * n * (n + 1) * dim + 3 * n * dim)}
    # decode: per step the weights once, each stream's cross memory and self rows, the logits
    b, steps, c = case["batch"], case["steps"], _decoder.DecoderConfig()
    d, f = c.dim, c.ffn
    layer = 8 * _matrix_bytes(d, d, 4, 128) + _matrix_bytes(f, d, 2, 128) + _matrix_bytes(d, f, 2, 128)
    flops = 2 * (8 * d * d + 2 * d * f)
    if case["features"]:
        layer += _matrix_bytes(24, 4 * d, 4, 128)
        flops += 2 * 24 * 4 * d
    keys = c.frames + (steps + 1) / 2
    kv = keys * (2 * d + 8 * c.heads)
    return {"bytes": int(steps * (c.layers * (layer + b * kv) + _matrix_bytes(c.vocab, d, 4, 128) + 4 * b * c.vocab)),
            "flops": int(steps * b * (c.layers * (flops + 4 * keys * d) + 2 * c.vocab * d))}


def tolerance(case):
    if case["kind"] == "hadamard":
        return {"rel": 1.5e-6}
    if case["kind"] == "exact" and case["dense"]:
        return {"rel": 1.5e-6}
    return "exact"


# ---- the same results in 64 bits -------------------------------------------


def _sylvester(n):
    h = np.ones((1, 1))
    while h.shape[0] < n:
        h = np.block([[h, h], [h, -h]])
    return h


def _product64(p, x):
    """x times the matrix p stands for: the rows' codebook levels times their
    group norms, over the input rotated group by group by H / sqrt(G)."""
    G, groups = p.Group, p.Groups()
    xp = np.zeros((x.shape[0], groups * G))
    xp[:, :p.In] = x
    xh = (xp.reshape(-1, groups, G) @ _sylvester(G) / math.sqrt(G)).reshape(x.shape[0], -1)
    by = p.Index.reshape(p.Out, -1)
    per = 8 // p.Width
    idx = np.stack([(by >> (p.Width * k)) & ((1 << p.Width) - 1) for k in range(per)], axis=2).reshape(p.Out, groups, G)
    norms = np.ascontiguousarray(p.Norms).view("<f2").astype(np.float64).reshape(p.Out, groups, 1)
    w = (p.Codebook.astype(np.float64)[idx] * norms).reshape(p.Out, -1)
    return (torch.from_numpy(xh) @ torch.from_numpy(w).T).numpy()


def _bound(x, axis):
    """QuantizeRow's scale: the largest magnitude over 127, 1 for zeros."""
    s = np.abs(x).max(axis=axis, keepdims=True) / x.dtype.type(127)
    return np.where(s > 0, s, x.dtype.type(1))


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        # every layer quantises what the one before computed (tables, int8
        # rows, the query), so the 64-bit values of a step are not the step's
        # own a few layers on; the layers' pieces have cases of their own
        return None
    if kind in ("products", "exact"):
        packs, x = _host(case, seed)
        return [_product64(p, x.astype(np.float64)) for p in packs]
    if kind == "plan":
        packs, xs = _host(case, seed)
        return [_product64(p, x.astype(np.float64)) for p, x in zip(packs, xs)]
    if kind == "memory":
        packs, x = _host(case, seed)
        if case["act8"]:  # the input's int8 codes times their scale, in float32 as the path defines them
            s = _bound(x, 1)
            x = np.rint(x / s) * s
        kv = [_product64(p, x.astype(np.float64)) for p in packs]
        heads = [y.reshape(y.shape[0], case["heads"], -1) for y in kv]
        scales = [_bound(y, 2) for y in heads]
        return {"kv": kv, "codes": [np.rint(y / s).reshape(y.shape[0], -1) for y, s in zip(heads, scales)],
                "scales": [s[:, :, 0] for s in scales]}
    if kind == "attend":
        return _attend64(case, seed)
    if kind == "hadamard":
        return _hadamard64(case, seed)
    packs, aff, stream, block_out = _host(case, seed)
    n, dim, rows = case["lanes"], case["dim"], case["rows"]
    st, a = stream.astype(np.float64), aff.astype(np.float64)
    flat = st.reshape(rows, n * dim)
    nx = flat / np.sqrt((flat * flat).mean(axis=1, keepdims=True) + 1e-6)
    pre, post, res = (_product64(p, nx) for p in packs)
    sig = lambda v: 1 / (1 + np.exp(-v))
    hp = sig(a[0] * pre + a[3:3 + n] + a[3 + n:3 + 2 * n])
    hq = 2 * sig(a[1] * post + a[3 + 2 * n:3 + 3 * n] + a[3 + 3 * n:3 + 4 * n])
    k = (a[2] * res + a[3 + 4 * n:]).reshape(rows, n, n)
    k = np.exp(k - k.max(axis=(1, 2), keepdims=True))
    for _ in range(20):
        k = k / k.sum(axis=2, keepdims=True)
        k = k / k.sum(axis=1, keepdims=True)
    u = (hp[:, :, None] * st).sum(axis=1)
    out = k @ st + hq[:, :, None] * (block_out.astype(np.float64) - u)[:, None, :]
    return {"nx": nx, "pre": hp, "post": hq, "res": k.reshape(rows, n * n), "u": u, "out": out}


def _attend64(case, seed):
    q, kq, ks, vq, vs, spans = _host(case, seed)
    b, t, h, kvh, qk, vd = (case[k] for k in ("batch", "t", "heads", "kv_heads", "qk", "vd"))
    out = np.zeros((b, t, h, vd))
    rep = h // kvh
    q = q.reshape(b, t, h, qk)
    if case["quant_q"]:  # the query's int8 codes and scale, as the path defines them
        s = _bound(q, 3)
        q = np.rint(q / s).astype(np.float64) * s
    q = q.astype(np.float64)
    for i in range(b):
        c = 0 if case["shared"] else i
        n = int(spans[i, :, 3].max())
        k = kq[c, :n].reshape(n, kvh, qk) * ks[c, :n].astype(np.float64)[:, :, None]
        v = vq[c, :n].reshape(n, kvh, vd) * vs[c, :n].astype(np.float64)[:, :, None]
        k, v = np.repeat(k, rep, axis=1).transpose(1, 2, 0), np.repeat(v, rep, axis=1).transpose(1, 0, 2)
        lg = q[i].transpose(1, 0, 2) @ k / math.sqrt(qk)
        lg = np.where(np.arange(n)[None, None, :] < spans[i, :, 3][None, :, None], lg, -np.inf)
        e = np.exp(lg - lg.max(axis=2, keepdims=True))
        out[i] = ((e / e.sum(axis=2, keepdims=True)) @ v).transpose(1, 0, 2)
    return out.reshape(b, t, h * vd)


def _hadamard64(case, seed):
    w, x = _host(case, seed)
    w = {k: v if k in ("p1", "p2") else v.astype(np.float64) for k, v in w.items()}
    na, nb, dim, rows = case["na"], case["nb"], case["dim"], case["rows"]
    kron = lambda z, a, b: (a.T @ z.reshape(rows, na, nb) @ b).reshape(rows, -1)
    xp = np.zeros((rows, na * nb))
    xp[:, :dim] = x
    e = xp[:, :dim] @ w["cond_v"]
    e = np.exp(e - e.max(axis=1, keepdims=True))
    cond = 1 + e / e.sum(axis=1, keepdims=True) @ w["cond_u"]
    z = kron(w["d1"] * xp, w["w1a"], w["w1b"])[:, w["p1"]]
    a = w["d2"] * cond * z + w["b2"]
    z = kron(a / (1 + np.exp(-a)), w["w2a"], w["w2b"])[:, w["p2"]]
    return (w["d4"] * kron(w["d3"] * z, w["w3a"], w["w3b"]))[:, :dim]

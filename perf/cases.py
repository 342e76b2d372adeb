"""What the framework is timed on: the calls a Gemma 4 engine makes for a token or a prompt.

Every pass goes through the C ABI (include/g4attn.h) as g4hip binds it, with the arguments
made beforehand, as a compiled engine would hold them.  Sizes are those of the E2B model the
framework's own tests and benchmark use: 8 query heads on 1 KV head, sliding layers of head
width 256 and window 512, global layers of head width 512, 35 layers of which 15 keep K/V,
hidden width 1536, a 262,144-row output head.

q and K rows are normal draws with unit RMS per head (the engine's norm, which RoPE keeps),
V rows likewise; raw q/k/v of the layer steps are plain normal draws.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("gemma4-rs_amd"))
import g4hip  # noqa: E402

EPS = 1e-6
LOCAL_BASE, GLOBAL_BASE = 10000.0, 1000000.0
WINDOW = 512
LAYERS, SHARED = 35, 20
CAP = 30.0  # the output head's soft cap


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # One token of a short chat through a sliding layer: the smallest call there is.
        {"name": "decode_sliding_64", "kind": "decode", "heads": 8, "kv": 1, "d": 256, "rows": 64},
        # One token through a global layer at a usual context length.
        {"name": "decode_global_4096", "kind": "decode", "heads": 8, "kv": 1, "d": 512, "rows": 4096},
        # One token through the attention of all 35 layers: norms, RoPE, append, attention.
        {"name": "token_35_layers_8192", "kind": "token", "context": 8192},
        # A serving step over 32 ragged sequences: a global and a sliding layer.
        {"name": "batch_32_ragged", "kind": "batch", "B": 32, "lo": 1024, "hi": 32768, "lens_seed": 2024},
        # A small serving batch through all 35 layers, captured once as a HIP graph, replayed per step.
        {"name": "batch_8_graph_35_layers", "kind": "serve", "B": 8, "lo": 300, "hi": 4096, "lens_seed": 7},
        # A 2048-token prompt chunk, sliding layer.
        {"name": "prefill_sliding_2048", "kind": "prefill", "heads": 8, "kv": 1, "d": 256, "window": WINDOW,
         "pos0": 0, "N": 2048, "exact_products": False},
        # The same chunk, global layer.
        {"name": "prefill_global_2048", "kind": "prefill", "heads": 8, "kv": 1, "d": 512, "window": 0,
         "pos0": 0, "N": 2048, "exact_products": False},
        # A follow-up turn of 256 tokens deep into a long context, global layer.
        {"name": "prefill_chunk_256_at_16384", "kind": "prefill", "heads": 8, "kv": 1, "d": 512, "window": 0,
         "pos0": 16384, "N": 256, "exact_products": False},
        # A prompt of an odd length in two chunks through a sliding and a global layer, from the
        # projected q/k/v on: norms, RoPE, append, attention.
        {"name": "prompt_777", "kind": "prompt", "tokens": 777, "chunk": 512},
        # One token's Q8_0 mat-vecs of five layers (four sliding, one global), captured as a graph.
        {"name": "matvecs_5_layers", "kind": "matvecs", "layers": 5, "hidden": 1536, "ffn": 6144},
        # One token's logits with the soft cap.
        {"name": "logits_262144", "kind": "logits", "rows": 262144, "cols": 1536},
        # A per-token projection kept in BF16 (35 layers x 256 values from the hidden row).
        {"name": "projection_bf16_8960", "kind": "dense", "format": "bf16", "rows": 8960, "cols": 1536},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "token", "batch", "batch", "serve", "prefill", "prefill", "prefill",
                       "prompt", "prompt", "matvecs", "logits", "dense", "dense"])
    if kind == "decode":
        d = rng.choice([256, 512])
        heads, kv = rng.choice([(8, 1), (8, 1), (8, 1), (16, 2)])
        return {"kind": kind, "heads": heads, "kv": kv, "d": d, "rows": _log(rng, 16, 512 if d == 256 else 32768)}
    if kind == "token":
        return {"kind": kind, "context": _log(rng, 64, 8192)}
    if kind == "batch":
        B = _log(rng, 2, 32)
        hi = _log(rng, 512, 32768)
        return {"kind": kind, "B": B, "lo": max(16, hi // 32), "hi": hi, "lens_seed": rng.randrange(1 << 30)}
    if kind == "serve":
        hi = _log(rng, 64, 4096)
        return {"kind": kind, "B": _log(rng, 1, 12), "lo": max(16, hi // 12), "hi": hi,
                "lens_seed": rng.randrange(1 << 30)}
    if kind == "prefill":
        d = rng.choice([256, 512])
        heads, kv = rng.choice([(8, 1), (8, 1), (8, 1), (16, 2)])
        while True:
            case = {"kind": kind, "heads": heads, "kv": kv, "d": d, "window": WINDOW if d == 256 else 0,
                    "pos0": rng.choice([0, _log(rng, 32, 16384)]), "N": _log(rng, 8, 2048),
                    "exact_products": rng.random() < 0.1}
            if work(case)["flops"] <= 4e10:
                return case
    if kind == "prompt":
        tokens = _log(rng, 24, 2048)
        return {"kind": kind, "tokens": tokens, "chunk": rng.choice([tokens, 512, 256])}
    if kind == "matvecs":
        return {"kind": kind, "layers": rng.randint(1, 5), "hidden": 256 * rng.randint(4, 10),
                "ffn": 1024 * rng.randint(4, 10)}
    if kind == "logits":
        return {"kind": kind, "rows": _log(rng, 16384, 262144), "cols": 256 * rng.randint(3, 6)}
    fmt = rng.choice(["bf16", "bf16", "f32", "q8_f32", "q8_f64"])
    return {"kind": "dense", "format": fmt, "rows": _log(rng, 64, 8960), "cols": 32 * _log(rng, 8, 64)}


# -------------------------------------------------------------------- helpers
def _lengths(case):
    return np.random.default_rng(case["lens_seed"]).integers(case["lo"], case["hi"] + 1, size=case["B"])


def _is_global(layer):
    return layer + 1 == LAYERS or layer % 5 == 4


def _source(layer):
    if layer < LAYERS - SHARED:
        return layer
    return 14 if _is_global(layer) else 13


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _unit_rows(g, rows, heads, d):
    x = _normal(g, rows, heads, d)
    x /= x.square().mean(-1, keepdim=True).sqrt()
    return x.view(rows, heads * d)


class _Ctx:
    """A context that goes with its state."""

    def __init__(self):
        self.ctx = g4hip.Context(0)
        self.handle = self.ctx.handle

    def __del__(self):
        try:
            self.ctx.close()
        except Exception:
            pass


class _Cache:
    def __init__(self, widths, capacity):
        self.owner = _shared()  # outlives the cache
        self.cache = g4hip.KvCache(self.owner, widths, capacity)
        self.handle = self.cache.handle

    def __del__(self):
        try:
            self.cache.close()
        except Exception:
            pass


_one = []


def _shared():
    """The program's context: one per device."""
    if not _one:
        _one.append(g4hip.Context(0))
    return _one[0]


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _call(name, *args):
    """A C ABI call with its arguments in hand."""
    fn = getattr(g4hip.lib(), name)
    return fn, tuple(a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args)


def _go(calls, stream):
    for fn, args in calls:
        if fn(*args, stream):
            raise RuntimeError(g4hip.lib().g4_last_error().decode())


def _captured(calls):
    _go(calls, _stream())  # sizes the workspace
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _go(calls, _stream())
    return graph


def _angles(pos, base, d):
    """rope_neox's angles: the engine's f32 recurrence."""
    scale = np.float32(np.float32(base) ** np.float32(-2.0 / d))
    a = np.empty(d // 2, np.float32)
    t = np.float32(pos)
    for i in range(d // 2):
        a[i] = t
        t = np.float32(t * scale)
    return a


def _rope_freqs():
    return torch.tensor(g4hip.proportional_rope_freq_factors(512, 0.25), device="cuda")


# ------------------------------------------------- weights in their GGUF form
def _q8_bytes(g, rows, cols):
    """Q8_0 rows of a normal matrix: blocks of an f16 scale and 32 int8."""
    out = torch.empty(rows * cols // 32, 34, dtype=torch.uint8, device="cuda")
    for at in range(0, out.shape[0], 1 << 21):
        n = min(1 << 21, out.shape[0] - at)
        w = _normal(g, n, 32) * 0.02
        scale = (w.abs().amax(1) / 127.0).to(torch.float16)
        q = (w / scale.float()[:, None]).round().clamp(-127, 127).to(torch.int8)
        out[at:at + n, :2] = scale.view(torch.uint8).view(n, 2)
        out[at:at + n, 2:] = q.view(torch.uint8)
    return out.view(-1)


def _q8_parts(w, rows, cols):
    w = w.view(rows, cols // 32, 34)
    scale = w[..., :2].contiguous().view(torch.float16).view(rows, cols // 32)
    return scale, w[..., 2:].contiguous().view(torch.int8)


def _q8_exact(w, rows, cols, x, quantized):
    """W @ x in 64 bits; the activation quantized first (matvec_q8_0) or as it is."""
    if quantized:
        b = x.view(-1, 32)
        scale = b.abs().amax(1) / 127.0
        inv = torch.where(scale == 0, torch.zeros_like(scale), 1.0 / scale)
        xq = torch.round(b * inv[:, None]).clamp(-128, 127).double()
        x = (xq * scale.to(torch.float16).double()[:, None]).view(-1)
    else:
        x = x.double()
    out = torch.empty(rows, dtype=torch.float64, device="cuda")
    for at in range(0, rows, 16384):
        n = min(16384, rows - at)
        s, q = _q8_parts(w.view(rows, -1)[at:at + n], n, cols)
        out[at:at + n] = (q.double() * s.double()[..., None]).view(n, cols) @ x
    return out


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(float(np.float32(0.7978846)) * x * (1.0 + float(np.float32(0.044715)) * x * x)))


# --------------------------------------------------------------------- inputs
def _layer_shapes(case):
    """(rows, cols) of one layer's projections: q, k, v, o, gate/up, down."""
    h, f = case["hidden"], case["ffn"]
    for i in range(case["layers"]):
        d = 512 if i % 5 == 4 else 256
        yield [("q", 8 * d, h), ("k", d, h), ("v", d, h), ("o", h, 8 * d), ("gate_up", f, h), ("down", h, f)]


def _inputs(case, seed):
    """The tensors of a case, from its seed."""
    g = _generator(seed)
    k = case["kind"]
    if k == "decode":
        n, kv, d = case["rows"], case["kv"], case["d"]
        return {"K": _unit_rows(g, n, kv, d), "V": _unit_rows(g, n, kv, d),
                "q": _unit_rows(g, 1, case["heads"], d).view(-1)}
    if k == "token":
        s = {"layers": [], "freqs": _rope_freqs()}
        T = case["context"]
        owners = {d: [l for l in range(LAYERS - SHARED) if _is_global(l) == (d == 512)] for d in (256, 512)}
        s["rows"] = {d: [_unit_rows(g, len(o) * T, 1, d).view(len(o), T, d) for _ in range(2)]  # K, V
                     for d, o in owners.items()}
        for l in range(LAYERS):
            d = 512 if _is_global(l) else 256
            e = {"q": _normal(g, 8 * d), "k": _normal(g, d), "v": _normal(g, d),
                 "qw": 0.8 + 0.4 * torch.rand(d, device="cuda", generator=g),
                 "kw": 0.8 + 0.4 * torch.rand(d, device="cuda", generator=g), "d": d}
            if _source(l) == l:
                e["K"], e["V"] = (t[owners[d].index(l)] for t in s["rows"][d])
            s["layers"].append(e)
        return s
    if k in ("batch", "serve"):
        lens = _lengths(case)
        s = {"kinds": {}}
        for d, attended in ((512, lens), (256, np.minimum(lens, WINDOW))):
            total = int(attended.sum())
            s["kinds"][d] = {
                "row0": torch.from_numpy(np.concatenate([[0], np.cumsum(attended)[:-1]]).astype(np.int64)).cuda(),
                "begin": torch.zeros(len(lens), dtype=torch.int64, device="cuda"),
                "end": torch.from_numpy(attended.astype(np.int64)).cuda(), "total": total, "lens": attended}
        layers = range(LAYERS) if k == "serve" else (4, 3)
        s["layers"] = []
        for l in layers:
            d = 512 if _is_global(l) else 256
            e = {"d": d, "q": _unit_rows(g, len(lens), 8, d)}
            if k == "batch" or _source(l) == l:
                e["K"], e["V"] = (_unit_rows(g, s["kinds"][d]["total"], 1, d) for _ in range(2))
            else:
                e["K"], e["V"] = s["layers"][_source(l)]["K"], s["layers"][_source(l)]["V"]
            s["layers"].append(e)
        return s
    if k == "prefill":
        n, kv, d = case["pos0"] + case["N"], case["kv"], case["d"]
        return {"K": _unit_rows(g, n, kv, d), "V": _unit_rows(g, n, kv, d),
                "q": _unit_rows(g, case["N"], case["heads"], d)}
    if k == "prompt":
        n = case["tokens"]
        s = {"freqs": _rope_freqs(), "layers": []}
        for l, d in ((0, 256), (4, 512)):
            # One projected row per token: q, k and v side by side in their own runs.
            s["layers"].append({"layer": l, "d": d, "raw": _normal(g, n * 10 * d),
                                "qw": 0.8 + 0.4 * torch.rand(d, device="cuda", generator=g),
                                "kw": 0.8 + 0.4 * torch.rand(d, device="cuda", generator=g)})
        return s
    if k == "matvecs":
        s = {"layers": []}
        for shapes in _layer_shapes(case):
            e = {}
            for name, rows, cols in shapes:
                e[name] = {"rows": rows, "cols": cols, "w": _q8_bytes(g, rows, cols)}
                if name == "gate_up":
                    e[name]["w2"] = _q8_bytes(g, rows, cols)
            e["x"], e["attended"], e["h"], e["act"] = (_normal(g, n) for n in (
                case["hidden"], e["o"]["cols"], case["hidden"], case["ffn"]))
            s["layers"].append(e)
        return s
    if k == "logits":
        return {"w": _q8_bytes(g, case["rows"], case["cols"]), "x": 20.0 * _normal(g, case["cols"])}
    rows, cols = case["rows"], case["cols"]
    x = _normal(g, cols)
    if case["format"].startswith("q8"):
        return {"w": _q8_bytes(g, rows, cols), "x": x}
    w = _normal(g, rows, cols) * 0.02
    return {"w": w.to(torch.bfloat16) if case["format"] == "bf16" else w, "x": x}


def _matvec_plan(e):
    """(weights, input) of one layer's calls, in the order a token makes them."""
    return [("q", "x"), ("k", "x"), ("v", "x"), ("o", "attended"), ("gate_up", "h"), ("down", "act")]


def prepare(case, seed):
    s = _inputs(case, seed)
    k = case["kind"]
    s["kind"] = k
    if k == "decode":
        n, d = case["rows"], case["d"]
        s["out"] = torch.zeros(case["heads"] * d, device="cuda")
        s["calls"] = [_call("g4_attend_decode", _shared().handle, s["q"], s["K"], s["V"], case["kv"] * d, 0, n,
                            case["heads"], case["kv"], d, 1.0, s["out"])]
    elif k == "token":
        pos = case["context"] - 1
        s["out"], s["calls"] = [], []
        for l, e in enumerate(s["layers"]):
            d, own = e["d"], _source(l) == l
            src = s["layers"][_source(l)]
            lo = 0 if _is_global(l) else max(0, pos + 1 - WINDOW)
            out = torch.zeros(8 * d, device="cuda")
            s["out"].append(out)
            row = lambda t, at: t.data_ptr() + at * d * 4  # noqa: E731
            s["calls"].append(_call(
                "g4_decode_step_fused", _shared().handle, e["q"], e["k"] if own else None, e["v"] if own else None,
                e["qw"], e["kw"] if own else None, EPS, GLOBAL_BASE if _is_global(l) else LOCAL_BASE,
                s["freqs"] if _is_global(l) else None, pos, row(src["K"], lo), row(src["V"], lo), d, pos + 1 - lo,
                row(src["K"], pos) if own else None, row(src["V"], pos) if own else None, 8, 1, d, 1.0, out))
        s["out"] += [t[:, pos] for d in (256, 512) for t in s["rows"][d]]  # the appended rows
    elif k in ("batch", "serve"):
        ctx = _shared() if k == "batch" else _Ctx()  # a graph keeps the workspace it was captured with
        s["ctx"], s["out"], s["calls"] = ctx, [], []
        for e in s["layers"]:
            d, at = e["d"], s["kinds"][e["d"]]
            out = torch.zeros(case["B"], 8 * d, device="cuda")
            s["out"].append(out)
            s["calls"].append(_call("g4_attend_decode_batch", ctx.handle, case["B"], e["q"], e["K"], e["V"], d,
                                    at["row0"], at["begin"], at["end"], case["hi"] if d == 512 else WINDOW, 8, 1, d,
                                    1.0, out))
        if k == "serve":
            s["graph"] = _captured(s["calls"])
    elif k == "prefill":
        d = case["d"]
        ctx = _shared()
        if case["exact_products"]:
            ctx = s["ctx"] = _Ctx()
            ctx.ctx.set_prefill_exact(1)
        s["out"] = torch.zeros(case["N"], case["heads"] * d, device="cuda")
        s["calls"] = [_call("g4_attend_prefill", ctx.handle, s["q"], s["K"], s["V"], case["kv"] * d, case["pos0"],
                            case["N"], case["window"], case["heads"], case["kv"], d, 1.0, s["out"])]
    elif k == "prompt":
        n = case["tokens"]
        hp = s["hp"] = g4hip.G4Hparams.e2b()
        s["cache"] = _Cache([256, 0, 0, 0, 512], n)
        s["calls"], s["out"], s["work"] = [], [], []
        for e in s["layers"]:
            d = e["d"]
            work, out = torch.empty_like(e["raw"]), torch.zeros(n, 8 * d, device="cuda")
            q, key, v = work[:n * 8 * d].view(n, -1), work[n * 8 * d:n * 9 * d].view(n, -1), work[n * 9 * d:].view(n, -1)
            s["work"].append(work)
            s["out"].append(out)
            for at in range(0, n, case["chunk"]):
                m = min(case["chunk"], n - at)
                s["calls"].append(_call("g4_layer_prefill", _shared().handle, s["cache"].handle, ctypes.byref(hp),
                                        e["layer"], at, m, q[at], key[at], v[at], e["qw"], e["kw"], s["freqs"],
                                        out[at], None))
    elif k == "matvecs":
        ctx = s["ctx"] = _Ctx()
        s["out"], s["calls"] = [], []
        for e in s["layers"]:
            for name, x in _matvec_plan(e):
                p = e[name]
                out = torch.zeros(p["rows"], device="cuda")
                s["out"].append(out)
                if name == "gate_up":
                    s["calls"].append(_call("g4_gated_ffn_q8_0", ctx.handle, p["w"], p["w2"], p["w"].numel(),
                                            p["rows"], p["cols"], e[x], 0, out))
                else:
                    s["calls"].append(_call("g4_project_q8_0", ctx.handle, p["w"], p["w"].numel(), p["rows"],
                                            p["cols"], e[x], out))
        s["graph"] = _captured(s["calls"])
    else:
        rows, cols = case["rows"], case["cols"]
        s["out"] = torch.zeros(rows, device="cuda")
        h, w, x = _shared().handle, s["w"], s["x"]
        if k == "logits":
            call = _call("g4_logits_q8_0", h, w, w.numel(), rows, cols, x, CAP, s["out"])
        elif case["format"] in ("bf16", "f32"):
            call = _call("g4_matvec_" + case["format"], h, w, w.numel(), rows, cols, x, s["out"])
        else:
            call = _call("g4_matvec_q8_0_f32", h, w, w.numel(), rows, cols, x, int(case["format"] == "q8_f64"),
                         s["out"])
        s["calls"] = [call]
    return s


def run(s):
    if "graph" in s:
        s["graph"].replay()
        return s["out"]
    if s["kind"] == "prompt":
        # A new prompt: the projections leave their rows in the layers' buffers, the cache starts empty.
        for e, work in zip(s["layers"], s["work"]):
            work.copy_(e["raw"])
        s["cache"].cache.clear()
    _go(s["calls"], _stream())
    return s["out"] + s["work"] if s["kind"] == "prompt" else s["out"]


# ----------------------------------------------------------- what it must cost
def _pairs(pos0, N, window):
    p = np.arange(pos0 + 1, pos0 + N + 1)
    return int((np.minimum(p, window) if window else p).sum())


def work(case):
    """Bytes: each input once, each output once.  Operations: 4 per head, dim and (query, key) pair; 2 per weight."""
    k = case["kind"]
    if k == "decode":
        n, d = case["rows"], case["d"]
        return {"bytes": 8 * n * case["kv"] * d + 8 * case["heads"] * d, "flops": 4 * case["heads"] * d * n}
    if k == "token":
        b = f = 0
        T = case["context"]
        for l in range(LAYERS):
            d = 512 if _is_global(l) else 256
            n = T if _is_global(l) else min(T, WINDOW)
            own = _source(l) == l
            b += (8 * n * d if own or l in (LAYERS - 2, LAYERS - 1) else 0) + 4 * d * (16 + (5 if own else 1))
            f += 32 * d * n
        return {"bytes": b, "flops": f}
    if k in ("batch", "serve"):
        lens = _lengths(case)
        b = f = 0
        for l in (range(LAYERS) if k == "serve" else (4, 3)):
            d = 512 if _is_global(l) else 256
            n = int(lens.sum() if _is_global(l) else np.minimum(lens, WINDOW).sum())
            b += (8 * n * d if k == "batch" or _source(l) == l else 0) + 64 * d * case["B"]
            f += 32 * d * n
        return {"bytes": b, "flops": f}
    if k == "prefill":
        d, n = case["d"], case["pos0"] + case["N"]
        first = max(0, case["pos0"] + 1 - case["window"]) if case["window"] else 0
        return {"bytes": 8 * (n - first) * case["kv"] * d + 8 * case["N"] * case["heads"] * d,
                "flops": 4 * case["heads"] * d * _pairs(case["pos0"], case["N"], case["window"])}
    if k == "prompt":
        n = case["tokens"]
        return {"bytes": sum(4 * n * d * (10 + 10 + 2 + 8) for d in (256, 512)),
                "flops": sum(32 * d * _pairs(0, n, w) for d, w in ((256, WINDOW), (512, 0)))}
    if k == "matvecs":
        b = f = 0
        for shapes in _layer_shapes(case):
            for name, rows, cols in shapes:
                m = 2 if name == "gate_up" else 1
                b += m * rows * cols // 32 * 34 + 4 * (rows + cols)
                f += 2 * m * rows * cols
        return {"bytes": b, "flops": f}
    size = {"bf16": 2.0, "f32": 4.0}.get(case.get("format"), 34 / 32)
    return {"bytes": size * case["rows"] * case["cols"] + 4 * (case["rows"] + case["cols"]),
            "flops": 2 * case["rows"] * case["cols"]}


def tolerance(case):
    """f32 results whose sums may be taken in another order; prefill products as split f16 or f32."""
    if case["kind"] in ("prefill", "prompt"):
        return {"rel": 1e-5, "max": 1e-3}
    if case["kind"] in ("decode", "token", "batch", "serve"):
        return {"rel": 1e-5, "max": 4e-4}
    return {"rel": 1.5e-6, "max": 4e-5}


# ------------------------------------------------------------- in 64 bits
def _attend(q, K, V, heads, kv, d, lo=None, hi=None):
    """q [N, heads*d] over rows K/V [n, kv*d]; query i attends rows lo[i]..hi[i]-1."""
    N, n = q.shape[0], K.shape[0]
    out = torch.empty(N, heads * d, dtype=torch.float64, device="cuda")
    mask = None
    if lo is not None:
        at = torch.arange(n, device="cuda")[None, :]
        mask = (at < lo[:, None]) | (at >= hi[:, None])
    for h in range(heads):
        c = h * kv // heads
        Kh, Vh = K[:, c * d:(c + 1) * d].double(), V[:, c * d:(c + 1) * d].double()
        sc = q[:, h * d:(h + 1) * d].double() @ Kh.t().contiguous()
        if mask is not None:
            sc.masked_fill_(mask, -math.inf)
        out[:, h * d:(h + 1) * d] = torch.softmax(sc, -1) @ Vh
    return out


def _causal(q, K, V, heads, kv, d, pos0, window):
    p = torch.arange(pos0 + 1, pos0 + q.shape[0] + 1, device="cuda")
    return _attend(q, K, V, heads, kv, d, (p - window).clamp(min=0) if window else torch.zeros_like(p), p)


def _norm_rope(x, weight, d, angles=None, factors=None):
    """x [N, heads*d] in 64 bits; angles [N, d/2] (f32, the engine's)."""
    N = x.shape[0]
    x = x.double().view(N, -1, d)
    x = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt()
    if weight is not None:
        x = x * weight.double()
    if angles is not None:
        a = angles.cuda()
        if factors is not None:
            a = a / factors
        c, s = a.double().cos()[:, None, :], a.double().sin()[:, None, :]
        u, v = x[..., :d // 2], x[..., d // 2:]
        x = torch.cat([u * c - v * s, u * s + v * c], -1)
    return x.reshape(N, -1)


def exact(case, seed):
    s = _inputs(case, seed)
    k = case["kind"]
    if k == "decode":
        return _attend(s["q"][None], s["K"], s["V"], case["heads"], case["kv"], case["d"])[0]
    if k == "token":
        pos = case["context"] - 1
        outs, rows = [], {}
        for l, e in enumerate(s["layers"]):
            d, glob = e["d"], _is_global(l)
            a = torch.from_numpy(_angles(pos, GLOBAL_BASE if glob else LOCAL_BASE, d))[None]
            f = s["freqs"] if glob else None
            q = _norm_rope(e["q"][None], e["qw"], d, a, f)
            if _source(l) == l:
                rows[l] = (_norm_rope(e["k"][None], e["kw"], d, a, f), _norm_rope(e["v"][None], None, d))
            src = s["layers"][_source(l)]
            lo = 0 if glob else max(0, pos + 1 - WINDOW)
            K = torch.cat([src["K"][lo:pos].double(), rows[_source(l)][0]])
            V = torch.cat([src["V"][lo:pos].double(), rows[_source(l)][1]])
            outs.append(_attend(q, K, V, 8, 1, d)[0])
        return outs + [torch.cat([r[i] for r in rows.values() if r[i].numel() == d])
                       for d in (256, 512) for i in (0, 1)]
    if k in ("batch", "serve"):
        outs = []
        for e in s["layers"]:
            d, at = e["d"], s["kinds"][e["d"]]
            row0, lens = at["row0"].tolist(), at["lens"].tolist()
            outs.append(torch.cat([_attend(e["q"][i:i + 1], e["K"][r:r + n], e["V"][r:r + n], 8, 1, d)
                                   for i, (r, n) in enumerate(zip(row0, lens))]))
        return outs
    if k == "prefill":
        return _causal(s["q"], s["K"], s["V"], case["heads"], case["kv"], case["d"], case["pos0"], case["window"])
    if k == "prompt":
        n = case["tokens"]
        outs, work_rows = [], []
        for e in s["layers"]:
            d, glob = e["d"], e["d"] == 512
            q, key, v = (e["raw"][a * n * d:b * n * d].view(n, -1) for a, b in ((0, 8), (8, 9), (9, 10)))
            a = torch.from_numpy(np.stack([_angles(p, GLOBAL_BASE if glob else LOCAL_BASE, d) for p in range(n)]))
            f = s["freqs"] if glob else None
            q, key, v = _norm_rope(q, e["qw"], d, a, f), _norm_rope(key, e["kw"], d, a, f), _norm_rope(v, None, d)
            outs.append(_causal(q, key, v, 8, 1, d, 0, 0 if glob else WINDOW))
            work_rows.append(torch.cat([q.reshape(-1), key.reshape(-1), v.reshape(-1)]))
        return outs + work_rows
    if k == "matvecs":
        outs = []
        for e in s["layers"]:
            for name, x in _matvec_plan(e):
                p = e[name]
                y = _q8_exact(p["w"], p["rows"], p["cols"], e[x], True)
                if name == "gate_up":
                    y = _gelu(y) * _q8_exact(p["w2"], p["rows"], p["cols"], e[x], True)
                outs.append(y)
        return outs
    if k == "logits":
        y = _q8_exact(s["w"], case["rows"], case["cols"], s["x"], True)
        return torch.tanh(y / CAP) * CAP
    if case["format"].startswith("q8"):
        return _q8_exact(s["w"], case["rows"], case["cols"], s["x"], False)
    x = s["x"].to(torch.bfloat16) if case["format"] == "bf16" else s["x"]
    return s["w"].double() @ x.double()

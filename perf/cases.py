"""The calls whose speed matters to a program that runs a diffusion language
model's denoise loop on this library, over the range of shapes it meets them at.

Kinds of case (a case is a dict of plain values; the sizes of the models are
those of tests/helpers.py, bench.py and the tests):

  step     one layer of a denoise step: the canvas rows' Q/K/V as the QKV
           projection leaves them, stored into the cache with bias, norm and
           RoPE folded in, and the attention of the canvas over prompt and
           canvas.  first=True is the first pass of a generation, where every
           position is active (prompt and canvas, the prompt causal in Gemma).
  scatter  a later step: split_active picks the changed and still masked
           positions on the device, then the layer runs on those rows only.
  pass     all layers of a denoise step, captured once in a HIP graph and
           replayed each step, as a loop over a fixed canvas runs it.
  wo       the projection after the attention on GGUF weights, with the
           residual add and (Gemma) the post-attention norm.
  experts  the expert matmuls of one MoE layer: a few experts, each with the
           rows that were routed to it.
  dropin   attention() on host arrays, the reference's own call.
"""
from __future__ import annotations

import math
import pathlib
import sys

import numpy as np
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "diffuse-rs_amd"))
import dr_attn as dr  # noqa: E402

# name: (query heads, KV heads, head dim)
MODELS = {
    "llada": (32, 32, 128),
    "dream": (28, 4, 128),
    "llada_moe": (16, 16, 128),
    "gemma_sliding": (16, 8, 256),
    "gemma_global": (16, 2, 512),
    "small": (8, 2, 64),
}
GEMMA_WINDOW = 1024
THETA = 10000.0
EPS = 1e-6
# GGML type: (values per block, bytes per block)
BLOCKS = {"q4_k": (256, 144), "q6_k": (256, 210), "q4_0": (32, 18), "q5_0": (32, 22), "q8_0": (32, 34)}
WTYPES = {"q4_k": 12, "q6_k": 14, "q4_0": 2, "q5_0": 6, "q8_0": 8}


# ------------------------------------------------------------------ cases


def _step(model, prompt, canvas, batch=1, first=False, fused=False):
    return {"kind": "step", "model": model, "prompt": prompt, "canvas": canvas, "batch": batch,
            "first": first, "fused": fused}


def listed():
    return [
        # the smallest call: a 64-token chat canvas after a 64-token prompt
        dict(_step("llada", 64, 64), name="step_llada_64"),
        # a whole denoise step of LLaDA-8B: 32 layers, 512 cached prompt rows + 256 canvas rows
        {"kind": "pass", "model": "llada", "layers": 32, "prompt": 512, "canvas": 256, "io": "f32", "name": "pass_llada8b"},
        # LLaDA-MoE, QK-norm and RoPE, rows of a fused QKV projection, a prompt
        # length as tokenizers give it (no multiple of anything)
        dict(_step("llada_moe", 2041, 512, fused=True), name="step_llada_moe"),
        # a late step of LLaDA-8B: 145 still masked or just changed canvas positions among 768
        {"kind": "scatter", "model": "llada", "prompt": 512, "canvas": 256, "masked": 137, "changed": 8, "name": "scatter_llada"},
        # Dream's first pass with classifier-free guidance: 1280 rows of both
        # streams, QKV bias and RoPE, grouped heads
        dict(_step("dream", 1024, 256, batch=2, first=True), name="first_dream_cfg"),
        # DiffusionGemma's two kinds of layer at attention scale 1.0 (hi/lo cache layers)
        dict(_step("gemma_sliding", 4096, 256), name="step_gemma_sliding"),
        dict(_step("gemma_global", 4096, 256), name="step_gemma_global"),
        # DiffusionGemma's first pass over prompt (causal) and canvas, the largest call
        dict(_step("gemma_sliding", 4096, 256, first=True), name="first_gemma_sliding"),
        # Wo of LLaDA-8B for a 256-row canvas, Q4_K, with the residual
        {"kind": "wo", "wtype": "q4_k", "rows": 4096, "cols": 4096, "n": 256, "post_norm": False, "name": "wo_llada_q4k"},
        # Wo of a first pass (2553 rows) on Q6_K weights with the post-attention norm
        {"kind": "wo", "wtype": "q6_k", "rows": 2048, "cols": 4096, "n": 2553, "post_norm": True, "name": "wo_first_q6k"},
        # one MoE layer's experts: 8 experts with up to 96 rows each, Q8_0
        {"kind": "experts", "wtype": "q8_0", "rows": 1024, "cols": 2048, "experts": 8, "n": 96, "name": "experts_q8_0"},
        # the reference's own call on host arrays: LLaDA-8B, 256 queries x 768 keys
        {"kind": "dropin", "model": "llada", "prompt": 512, "canvas": 256, "causal": False, "name": "dropin_llada"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    most = work(_step("gemma_sliding", 4096, 256, first=True))
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= 0.9 * most["flops"] and w["bytes"] <= 1.2e9:
            return c


def _draw(rng):
    kind = rng.choice(["step", "step", "gemma", "first", "scatter", "pass", "wo", "wo", "experts", "dropin"])
    if kind == "step":
        model = rng.choice(["llada", "dream", "llada_moe", "small"])
        return _step(model, _log(rng, 16, 4096), _log(rng, 8, 512), batch=rng.choice([1, 1, 2, 4]),
                     fused=rng.random() < 0.5)
    if kind == "gemma":
        return _step(rng.choice(["gemma_sliding", "gemma_global"]), _log(rng, 64, 6144), _log(rng, 16, 384))
    if kind == "first":
        model = rng.choice(["llada", "dream", "llada_moe", "small", "gemma_sliding", "gemma_global"])
        total = _log(rng, 64, 4096)
        canvas = max(8, total // rng.choice([2, 4, 8]))
        return _step(model, max(8, total - canvas), canvas, batch=rng.choice([1, 1, 2]), first=True)
    if kind == "scatter":
        canvas = _log(rng, 32, 512)
        masked = rng.randint(4, canvas - 12)
        return {"kind": "scatter", "model": rng.choice(["llada", "dream", "llada_moe"]),
                "prompt": _log(rng, 32, 4096), "canvas": canvas, "masked": masked, "changed": rng.randint(0, 8)}
    if kind == "pass":
        return {"kind": "pass", "model": rng.choice(["llada", "dream", "llada_moe"]), "layers": rng.randint(4, 32),
                "prompt": 32 * _log(rng, 2, 64), "canvas": 32 * _log(rng, 1, 16), "io": rng.choice(["f32", "bf16"])}
    if kind == "wo":
        return {"kind": "wo", "wtype": rng.choice(["q4_k", "q4_k", "q6_k", "q4_0"]), "rows": 16 * _log(rng, 32, 256),
                "cols": 256 * _log(rng, 4, 16), "n": _log(rng, 1, 3072), "post_norm": rng.random() < 0.3}
    if kind == "experts":
        return {"kind": "experts", "wtype": rng.choice(["q4_k", "q6_k", "q4_0", "q5_0", "q8_0"]),
                "rows": 16 * _log(rng, 16, 128), "cols": 256 * _log(rng, 2, 8), "experts": rng.randint(2, 16),
                "n": _log(rng, 2, 160)}
    return {"kind": "dropin", "model": rng.choice(["llada", "dream", "llada_moe", "small"]),
            "prompt": _log(rng, 16, 1024), "canvas": _log(rng, 16, 256), "causal": rng.random() < 0.5}


# ------------------------------------------------------------------ geometry


def _geom(c):
    """Heads, masks, epilogue and positions of an attention case."""
    h, hkv, hd = MODELS[c["model"]]
    gemma = c["model"].startswith("gemma")
    n_tot = c["prompt"] + c["canvas"]
    first = bool(c.get("first") or c.get("causal"))  # (a causal prompt: every position asks, as in a first pass)
    return {
        "h": h, "hkv": hkv, "hd": hd, "gemma": gemma, "n_tot": n_tot, "n0": 0 if first else c["prompt"],
        "window": GEMMA_WINDOW if c["model"] == "gemma_sliding" else None,
        "prefix": c["prompt"] if gemma or c.get("causal") else None,
        "scale": 1.0 if gemma else 1.0 / math.sqrt(hd),
        "bias": c["model"] == "dream", "norm": gemma or c["model"] == "llada_moe", "vnorm": gemma,
    }


def _visible(qpos, kpos, window, prefix):
    """[q, k] which keys a query sees."""
    q, k = qpos[:, None], kpos[None, :]
    ok = torch.ones(q.shape[0], k.shape[1], dtype=torch.bool, device=qpos.device)
    if window is not None:
        ok &= (q - k).abs() < window
    if prefix is not None:
        ok &= ~((q < prefix) & (k > q))
    return ok


def _count(q0, n_tot, window, prefix):
    """(sum over queries q0..n_tot-1 of the keys each sees, keys that any sees)."""
    q = np.arange(q0, n_tot)
    lo = np.maximum(0, q - window + 1) if window is not None else np.zeros_like(q)
    hi = np.minimum(n_tot, q + window) if window is not None else np.full_like(q, n_tot)
    if prefix is not None:
        hi = np.where(q < prefix, np.minimum(hi, q + 1), hi)
    return int((hi - lo).sum()), int(hi.max() - lo.min())


def work(case):
    kind = case["kind"]
    if kind in ("wo", "experts"):
        qk, bb = BLOCKS[case["wtype"]]
        rows, cols = case["rows"], case["cols"]
        ns = _expert_rows(case) if kind == "experts" else [case["n"]]
        b = len(ns) * rows * cols // qk * bb + sum(ns) * 4 * (cols + rows)
        if kind == "wo":
            b += 4 * rows * case["n"] + (4 * rows if case["post_norm"] else 0)
        return {"bytes": b, "flops": 2 * sum(ns) * rows * cols}
    g = _geom(case)
    if kind == "scatter":
        n, layers, batch = case["masked"] + case["changed"], 1, 1
        sees, keys = n * g["n_tot"], g["n_tot"]
    else:
        n = g["n_tot"] - g["n0"]
        layers, batch = case.get("layers", 1), case.get("batch", 1)
        sees, keys = _count(g["n0"], g["n_tot"], g["window"], g["prefix"])
    if kind == "dropin":
        b = 4 * g["hd"] * (2 * g["h"] * n + 2 * g["hkv"] * g["n_tot"])
    else:
        kv = 4 if g["gemma"] else 2  # cached bytes of one K or V value (hi + lo halves in Gemma's layers)
        io = 2 if case.get("io") == "bf16" else 4
        b = 2 * io * n * g["h"] * g["hd"]  # Q in, attention out
        b += 2 * (4 + kv) * n * g["hkv"] * g["hd"]  # fresh K and V rows in, their cached form out
        b += 2 * kv * max(0, keys - n) * g["hkv"] * g["hd"]  # the cached rows that were there
    return {"bytes": layers * batch * b, "flops": layers * batch * 4 * g["h"] * g["hd"] * sees}


def tolerance(case):
    """About four times the distance from exact() that the calls show (measured: Wo 1e-7, hi/lo layers 3e-4,
    host arrays 1.6e-3, bf16 layers 3.4e-3)."""
    kind = case["kind"]
    if kind in ("wo", "experts"):
        return {"rel": 5e-7}  # exact integers, f32 sums over the blocks
    if kind == "dropin":
        return {"rel": 6e-3}  # softmax weights in bf16, flat over the keys
    if case["model"].startswith("gemma"):
        return {"rel": 1.5e-3}  # softmax weights in bf16, one or a few keys of each row
    return {"rel": 1.4e-2}  # Q, K, V and the softmax weights in bf16


# ------------------------------------------------------------------ the program's own objects

_DEV = {}


def _dev(io="f32"):
    """The program's context and stream: one of each, and a second context for bf16 rows."""
    if not _DEV:
        _DEV["stream"] = torch.cuda.Stream()
    if io not in _DEV:
        ctx = dr.Context(0)
        ctx.set_stream(_DEV["stream"].cuda_stream)
        if io == "bf16":
            ctx.set_q_dtype(dr.DTYPE_BF16)
            ctx.set_o_dtype(dr.DTYPE_BF16)
        _DEV[io] = ctx
    return _DEV[io], _DEV["stream"]


def _gen(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return g


def _rows_in(case, seed):
    """Per batch slot: the prompt's K and V rows (ready for the cache) and the
    active rows' Q, K and V, as one [n, (h + 2 hkv) hd] block; and the gains and biases."""
    g, gen = _geom(case), _gen(seed)
    h, hkv, hd = g["h"], g["hkv"], g["hd"]
    n = g["n_tot"] - g["n0"]
    slots = []
    for _ in range(case.get("batch", 1)):
        kp = torch.randn(g["n0"], hkv * hd, device="cuda", generator=gen)
        vp = torch.randn(g["n0"], hkv * hd, device="cuda", generator=gen)
        if g["norm"] and g["n0"]:
            kp = _norm(kp, hd, None)
        qkv = torch.randn(n, (h + 2 * hkv) * hd, device="cuda", generator=gen)
        slots.append((kp, vp, qkv))
    epi = {}
    if g["norm"]:
        epi["q_norm_w"] = torch.rand(hd, device="cuda", generator=gen) + 0.5
        epi["k_norm_w"] = torch.rand(hd, device="cuda", generator=gen) + 0.5
    if g["bias"]:
        for name, m, size in (("bq", h, 0.5), ("bk", hkv, 0.5), ("bv", hkv, 0.02)):
            epi[name] = size * torch.randn(m * hd, device="cuda", generator=gen)
    return g, slots, epi


def _norm(x, hd, w):
    y = x.reshape(x.shape[0], -1, hd)
    y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + EPS)
    return (y if w is None else y * w).reshape(x.shape)


def _rope_table(n, hd):
    """[n, hd/2] angles in f32, as the model defines them."""
    f = (np.float32(1.0) / np.power(np.float32(THETA), (2.0 * np.arange(hd // 2, dtype=np.float32) / np.float32(hd)))).astype(np.float32)
    return (np.arange(n, dtype=np.float32)[:, None] * f[None, :]).astype(np.float32)


def _step_call(cache, g, p, slots, epi, rope, out, fused):
    """The arguments of one layer's call; Q, K and V lie side by side in a fused projection's rows."""
    h, hkv, hd = g["h"], g["hkv"], g["hd"]
    kw = dict(sliding_window=g["window"], causal_prefix=g["prefix"], scale=g["scale"], v_norm=g["vnorm"], eps=EPS,
              rope=rope, **epi)
    if fused:
        ld = (h + 2 * hkv) * hd
        items = [(qkv.data_ptr(), o, p, qkv.data_ptr() + 4 * h * hd, qkv.data_ptr() + 4 * (h + hkv) * hd)
                 for (_, _, qkv), o in zip(slots, out)]
        return lambda: cache.step_rows(0, items, h, ld, ld, **kw), slots
    parts = [[x.contiguous() for x in qkv.split([h * hd, hkv * hd, hkv * hd], 1)] for _, _, qkv in slots]
    items = [(q, o, p, k, v) for (q, k, v), o in zip(parts, out)]
    return lambda: cache.step_epi(0, items, h, **kw), parts


def _tokens(case, seed):
    """The step's tokens, the mask, the tokens of the step before, and the
    positions that are active: the masked ones and those that just changed."""
    rng = np.random.default_rng(seed)
    n_tot = case["prompt"] + case["canvas"]
    seq = rng.integers(5, 30000, n_tot).astype(np.int32)
    pick = case["prompt"] + rng.permutation(case["canvas"])
    masked, changed = pick[: case["masked"]], pick[case["masked"]: case["masked"] + case["changed"]]
    mask = np.zeros(n_tot, np.uint8)
    mask[masked] = 1
    seq[masked] = 4
    prev = seq.copy()
    prev[changed] = 4
    return seq, mask, prev, np.sort(np.concatenate([masked, changed]))


def _layer_inputs(case, seed):
    g, gen = _geom(case), _gen(seed)
    kv, nl = g["hkv"] * g["hd"], case["layers"]
    kp, vp = (torch.randn(nl, case["prompt"], kv, device="cuda", generator=gen) for _ in range(2))
    k, v = (torch.randn(nl, case["canvas"], kv, device="cuda", generator=gen) for _ in range(2))
    q = torch.randn(nl, case["canvas"], g["h"] * g["hd"], device="cuda", generator=gen)
    return g, kp, vp, k, v, q.bfloat16() if case["io"] == "bf16" else q


def _expert_rows(case):
    """Rows routed to each expert: uneven, as a router leaves them."""
    return [1 + (case["n"] * (5 * e + 3) // 7) % case["n"] for e in range(case["experts"])]


def _weights(case, seed, rows):
    """[rows, blocks, bytes] GGUF blocks with random quants and scales of a trained layer's size."""
    qk, bb = BLOCKS[case["wtype"]]
    gen, nb = _gen(seed), case["cols"] // qk
    w = torch.randint(0, 256, (rows, nb, bb), device="cuda", dtype=torch.uint8, generator=gen)

    def half(lo, hi):
        d = torch.rand(rows, nb, 1, device="cuda", generator=gen) * (hi - lo) + lo
        return d.to(torch.float16).view(torch.uint8)

    if case["wtype"] == "q4_k":
        w[:, :, 0:2], w[:, :, 2:4] = half(5e-5, 2e-4), half(2e-4, 1.2e-3)
    elif case["wtype"] == "q6_k":
        w[:, :, 208:210] = half(5e-6, 2e-5)
    else:
        w[:, :, 0:2] = half(2e-4, 1e-3) if case["wtype"] == "q8_0" else half(2e-3, 1e-2)
    return w


def _acts(case, seed, n):
    """Rows of attention output: a few dimensions larger than the rest."""
    gen = _gen(seed)
    x = torch.randn(n, case["cols"], device="cuda", generator=gen)
    return x * (0.3 + 2.0 * torch.rand(case["cols"], device="cuda", generator=gen) ** 4)


# ------------------------------------------------------------------ prepare and run


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dropin":
        return _prepare_dropin(case, seed)
    ctx, stream = _dev(case.get("io", "f32"))
    with torch.cuda.stream(stream):
        if kind == "wo":
            n, rows = case["n"], case["rows"]
            gen = _gen(seed + 3)
            return {"kind": kind, "case": case, "ctx": ctx, "w": _weights(case, seed + 1, rows), "x": _acts(case, seed + 2, n),
                    "res": torch.randn(n, rows, device="cuda", generator=gen),
                    "gain": torch.rand(rows, device="cuda", generator=gen) + 0.5,
                    "out": torch.empty(n, rows, device="cuda")}
        if kind == "experts":
            ns = _expert_rows(case)
            return {"kind": kind, "case": case, "ctx": ctx, "ns": ns,
                    "w": _weights(case, seed + 1, case["rows"] * case["experts"]),
                    "x": [x.contiguous() for x in _acts(case, seed + 2, sum(ns)).split(ns)],
                    "out": [torch.empty(m, case["rows"], device="cuda") for m in ns]}
        if kind == "pass":
            return _prepare_pass(case, seed, ctx, stream)
        g, slots, epi = _rows_in(case, seed)
        n_tot = g["n_tot"]
        hilo = [dr.PRECISION_HILO] if g["gemma"] else None
        cache = dr.StepCache(ctx, n_tot, [g["hkv"]], [g["hd"]], n_batch=len(slots), precision=hilo)
        rope = dr.Rope(ctx, n_tot, g["hd"], THETA)
        if g["n0"]:
            before = dr.Pass(ctx, range(g["n0"]))
            for b, (kp, vp, _) in enumerate(slots):
                cache.store(0, before, kp, vp, batch=b)
        if kind == "scatter":
            canvas = dr.Pass(ctx, range(g["n0"], n_tot))  # as the step before left them
            kv = g["hkv"] * g["hd"]
            kc, vc = (x.contiguous() for x in slots[0][2][:, -2 * kv:].split(kv, 1))
            cache.store(0, canvas, kc, vc)
            seq, mask, prev, active = _tokens(case, seed)
            cache.update_seq(prev)
            gen = _gen(seed + 7)
            rows = torch.randn(len(active), (g["h"] + 2 * g["hkv"]) * g["hd"], device="cuda", generator=gen)
            slots = [(None, None, rows)]
            p, rest = dr.Pass(ctx, range(n_tot)), dr.Pass(ctx, range(n_tot))
        else:
            p, rest = dr.Pass(ctx, range(g["n0"], n_tot)), None
        out = torch.empty(len(slots), slots[0][2].shape[0], g["h"] * g["hd"], device="cuda")
        call, keep = _step_call(cache, g, p, slots, epi, rope, list(out), case.get("fused", False))
        s = {"kind": kind, "call": call, "out": out, "keep": (keep, epi, rope, cache, p, rest), "cache": cache}
        if kind == "scatter":
            s.update(n=n_tot, p=p, rest=rest, seq=torch.from_numpy(seq).cuda(), mask=torch.from_numpy(mask).cuda())
        stream.synchronize()
        return s


def _prepare_pass(case, seed, ctx, stream):
    g, kp, vp, k, v, q = _layer_inputs(case, seed)
    nl, h = case["layers"], g["h"]
    cache = dr.StepCache(ctx, g["n_tot"], [g["hkv"]] * nl, [g["hd"]] * nl)
    before, p = dr.Pass(ctx, range(case["prompt"])), dr.Pass(ctx, range(case["prompt"], g["n_tot"]))
    for i in range(nl):
        cache.store(i, before, kp[i], vp[i])
    out = torch.empty_like(q)

    def layers():
        for i in range(nl):
            cache.step(i, [(q[i], out[i], p, k[i], v[i])], h, scale=g["scale"])

    layers()  # (sizes the context's workspace before the capture)
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        layers()
    return {"kind": "pass", "graph": graph, "stream": stream, "out": out, "keep": (cache, before, p, k, v, q)}


def _prepare_dropin(case, seed):
    g, q, k, v = _host_inputs(case, seed)
    n_tot, n0 = g["n_tot"], g["n0"]
    shape = dr.AttnShape(nq=n_tot - n0, nk=n_tot, n_head=g["h"], n_head_kv=g["hkv"], head_dim=g["hd"],
                         causal_prefix=g["prefix"], scale=g["scale"])
    return {"kind": "dropin", "q": q, "k": k, "v": v, "out": np.empty_like(q), "shape": shape,
            "qr": dr.Rows(pos=np.arange(n0, n_tot)), "kr": dr.Rows(pos=np.arange(n_tot))}


def _host_inputs(case, seed):
    g = _geom(case)
    rng = np.random.default_rng(seed)
    q = rng.standard_normal((g["n_tot"] - g["n0"], g["h"] * g["hd"]), dtype=np.float32)
    k, v = (rng.standard_normal((g["n_tot"], g["hkv"] * g["hd"]), dtype=np.float32) for _ in range(2))
    return g, q, k, v


def run(state):
    kind = state["kind"]
    if kind == "step":
        state["call"]()
    elif kind == "scatter":
        state["cache"].split_active_dev(state["seq"], state["mask"], state["n"], 5, state["p"], state["rest"])
        state["call"]()
    elif kind == "pass":
        with torch.cuda.stream(state["stream"]):
            state["graph"].replay()
    elif kind == "wo":
        c = state["case"]
        if c["post_norm"]:
            dr.qmatmul_post_norm(state["ctx"], WTYPES[c["wtype"]], state["w"], c["rows"], c["cols"], state["x"], c["n"],
                                 state["out"], state["gain"], EPS, state["res"])
        else:
            dr.qmatmul(state["ctx"], WTYPES[c["wtype"]], state["w"], c["rows"], c["cols"], state["x"], c["n"],
                       state["out"], state["res"])
    elif kind == "experts":
        c = state["case"]
        for e, m in enumerate(state["ns"]):
            dr.qmatmul_expert(state["ctx"], WTYPES[c["wtype"]], state["w"], c["experts"], e, c["rows"], c["cols"],
                              state["x"][e], m, state["out"][e])
    else:
        dr.attention(state["out"], state["q"], state["k"], state["v"], state["shape"], state["qr"], state["kr"])
    return state["out"]


# ------------------------------------------------------------------ the same in 64 bits


def _attention64(q, k, v, qpos, kpos, g):
    """q [nq, h, hd], k and v [nk, hkv, hd] in 64 bits -> [nq, h * hd]."""
    ok = _visible(qpos, kpos, g["window"], g["prefix"])
    out = torch.empty_like(q)
    for i in range(g["h"]):
        j = i // (g["h"] // g["hkv"])
        s = (q[:, i] @ k[:, j].T) * g["scale"]
        out[:, i] = torch.softmax(s.masked_fill(~ok, float("-inf")), 1) @ v[:, j]
    return out.reshape(q.shape[0], -1)


def _rope64(x, hd, pos):
    """x [n, heads, hd] rotated at positions pos (dim i with dim i + hd/2)."""
    a = torch.from_numpy(_rope_table(int(pos.max()) + 1, hd)).to(x.device)[pos].double()[:, None, :]
    a, b, s, c = x[..., : hd // 2], x[..., hd // 2:], torch.sin(a), torch.cos(a)
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _epilogue64(qkv, g, epi, pos):
    h, hkv, hd = g["h"], g["hkv"], g["hd"]
    q, k, v = qkv.double().split([h * hd, hkv * hd, hkv * hd], 1)
    if g["bias"]:
        q, k, v = q + epi["bq"].double(), k + epi["bk"].double(), v + epi["bv"].double()
    if g["norm"]:
        q, k = _norm(q, hd, epi["q_norm_w"].double()), _norm(k, hd, epi["k_norm_w"].double())
    if g["vnorm"]:
        v = _norm(v, hd, None)
    q, k, v = (x.reshape(x.shape[0], -1, hd) for x in (q, k, v))
    return _rope64(q, hd, pos), _rope64(k, hd, pos), v


def exact(case, seed):
    kind = case["kind"]
    if kind == "dropin":
        g, q, k, v = _host_inputs(case, seed)
        q, k, v = (torch.from_numpy(x).cuda().double().reshape(x.shape[0], -1, g["hd"]) for x in (q, k, v))
        pos = torch.arange(g["n_tot"], device="cuda")
        return _attention64(q, k, v, pos[g["n0"]:], pos, g).cpu().numpy()
    if kind == "wo":
        y = _dot64(case, _weights(case, seed + 1, case["rows"]), _acts(case, seed + 2, case["n"]))
        gen = _gen(seed + 3)
        res = torch.randn(case["n"], case["rows"], device="cuda", generator=gen)
        gain = torch.rand(case["rows"], device="cuda", generator=gen) + 0.5
        if case["post_norm"]:
            y = _norm(y, case["rows"], gain.double())
        return y + res.double()
    if kind == "experts":
        ns = _expert_rows(case)
        w = _weights(case, seed + 1, case["rows"] * case["experts"]).split(case["rows"])
        return [_dot64(case, w[e], x) for e, x in enumerate(_acts(case, seed + 2, sum(ns)).split(ns))]
    if kind == "pass":
        g, kp, vp, k, v, q = _layer_inputs(case, seed)
        pos = torch.arange(g["n_tot"], device="cuda")
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        for i in range(case["layers"]):
            kk, vv = (torch.cat(x).double().reshape(g["n_tot"], -1, g["hd"]) for x in ((kp[i], k[i]), (vp[i], v[i])))
            out[i] = _attention64(q[i].double().reshape(q.shape[1], -1, g["hd"]), kk, vv, pos[case["prompt"]:], pos, g)
        return out
    g, slots, epi = _rows_in(case, seed)
    pos, hd = torch.arange(g["n_tot"], device="cuda"), g["hd"]
    out = []
    for kp, vp, qkv in slots:
        if kind == "scatter":
            kv = g["hkv"] * hd
            k, v = (torch.cat(x).double().reshape(-1, g["hkv"], hd)
                    for x in ((kp, qkv[:, -2 * kv: -kv]), (vp, qkv[:, -kv:])))
            qpos = torch.from_numpy(_tokens(case, seed)[3]).cuda()
            qkv = torch.randn(len(qpos), qkv.shape[1], device="cuda", generator=_gen(seed + 7))
            q, kf, vf = _epilogue64(qkv, g, epi, qpos)
            k[qpos], v[qpos] = kf, vf
        else:
            qpos = pos[g["n0"]:]
            q, kf, vf = _epilogue64(qkv, g, epi, qpos)
            k = torch.cat([kp.double().reshape(g["n0"], g["hkv"], hd), kf])
            v = torch.cat([vp.double().reshape(g["n0"], g["hkv"], hd), vf])
        out.append(_attention64(q, k, v, qpos, pos, g))
    return torch.stack(out)


def _away(x):
    """Rounded to the nearest whole number, halves away from zero (x is f32)."""
    x = x.double()
    return torch.sign(x) * torch.floor(x.abs() + 0.5)


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dot64(case, w, x):
    """The k-quant / legacy block product of quantized weights and activations, in 64 bits."""
    rows, nb, _ = w.shape
    if case["wtype"] in ("q4_k", "q6_k"):
        b = x.reshape(x.shape[0], -1, 256)
        m = b.gather(2, b.abs().argmax(2, keepdim=True))
        i = -128.0 / m
        xq = torch.clamp(_away(i * b), max=127.0) * (1.0 / i).double()
    else:
        b = x.reshape(x.shape[0], -1, 32)
        d = b.abs().amax(2, keepdim=True) / 127.0
        xq = _away(b * (1.0 / d)) * d.to(torch.float16).double()
    if case["wtype"] == "q4_k":
        p = w[:, :, 4:16].to(torch.int32)
        sc = torch.cat([p[..., 0:4] & 63, (p[..., 8:12] & 15) | ((p[..., 0:4] >> 6) << 4)], 2).double()
        mn = torch.cat([p[..., 4:8] & 63, (p[..., 8:12] >> 4) | ((p[..., 4:8] >> 6) << 4)], 2).double()
        q = w[:, :, 16:144].reshape(rows, nb, 4, 32)
        q = torch.stack([q & 15, q >> 4], 3).reshape(rows, nb, 8, 32).double()
        wq = _f16(w[:, :, 0:2])[..., None] * sc[..., None] * q - _f16(w[:, :, 2:4])[..., None] * mn[..., None]
    elif case["wtype"] == "q6_k":
        lo = w[:, :, 0:128].reshape(rows, nb, 2, 2, 32).to(torch.int32)
        hi = w[:, :, 128:192].reshape(rows, nb, 2, 1, 32).to(torch.int32)
        sc = w[:, :, 192:208].contiguous().view(torch.int8).double()
        lo = torch.cat([lo & 15, lo >> 4], 3)  # [.., 2, 4, 32]: values 32 j .. of each half
        hi = torch.cat([(hi >> s) & 3 for s in (0, 2, 4, 6)], 3)
        q = ((lo | (hi << 4)) - 32).reshape(rows, nb, 16, 16).double()
        wq = _f16(w[:, :, 208:210])[..., None] * sc[..., None] * q
    else:
        if case["wtype"] == "q8_0":
            q = w[:, :, 2:34].contiguous().view(torch.int8).double()
        else:
            at = 2 if case["wtype"] == "q4_0" else 6
            q = torch.cat([w[:, :, at:] & 15, w[:, :, at:] >> 4], 2).to(torch.int32)
            if case["wtype"] == "q5_0":
                bit = w[:, :, 2:6].to(torch.int32)[..., None] >> torch.arange(8, device=w.device, dtype=torch.int32)
                q = q | ((bit & 1).reshape(rows, nb, 32) << 4)
            q = (q - (8 if case["wtype"] == "q4_0" else 16)).double()
        wq = _f16(w[:, :, 0:2]) * q
    return xq.reshape(x.shape[0], -1) @ wq.reshape(rows, -1).T

"""The attention calls that a user of this library times: what each is, its inputs, one pass of it, its answer.

A pass runs the layers of one step of a host program through the C ABI's
Python binding: `layers` attention calls one after another on the current
stream, each layer on tensors of its own. A case says

  entry     the entry point: "op" (flash_attn_ext), "implicit" (a causal or
            window descriptor in place of the mask tensor), "append" and
            "rope" (the new K/V rows given in F32 and stored by the call),
            "ring" (a ring-buffer cache and its new row)
  hq hkv hd query heads, kv heads, head dim
  nq past   query rows, and cache rows that precede them (n_kv = past + nq)
  capacity  rows of the cache that the views are cut from
  batch     independent streams along ne[3]
  kv        type of K and V: "f16", or "f32" as the application holds them
  mask      "none", "causal" (with `window` > 0: only the last `window`
            positions), "lengths" (each stream sees its own first rows)
  graph     the step is recorded once into a HIP graph and replayed, as a
            serving loop does with its decode step (launch-bound, and equal
            from step to step); else each call is made directly
"""
import importlib.util
import math
import os
import random
import sys

import torch

ROPE_BASE = 1.0e6


def _package():
    """The package's folder name is not a Python identifier."""
    if "voxtral_cpp_amd" not in sys.modules:
        folder = os.path.abspath("voxtral.cpp_amd")
        spec = importlib.util.spec_from_file_location(
            "voxtral_cpp_amd", os.path.join(folder, "__init__.py"), submodule_search_locations=[folder])
        module = importlib.util.module_from_spec(spec)
        sys.modules["voxtral_cpp_amd"] = module
        spec.loader.exec_module(module)
    return sys.modules["voxtral_cpp_amd"]


PKG = _package()
vxfa, views = PKG.vxfa, PKG.views


def _case(name, **kw):
    c = {"entry": "op", "hq": 32, "hkv": 8, "hd": 128, "nq": 1, "past": 0, "capacity": 0, "batch": 1, "kv": "f16",
         "mask": "none", "window": 0, "layers": 1, "graph": False}
    c.update(kw)
    if not c["capacity"]:
        c["capacity"] = c["past"] + c["nq"]
    return {"name": name, **c} if name else c


def listed():
    return [
        # the first generated token after a 39-token streaming prompt, one
        # layer called directly: nothing but latency
        _case("decode_first", past=39, capacity=8192),
        # a token of an offline transcription (prompt of 383, some text so
        # far), all 30 decoder layers with rotation and append in the call
        _case("decode_rope_token", entry="rope", past=434, capacity=8192, layers=30, graph=True),
        # the same token as the unchanged application asks for it: its own
        # F32 cache, four minutes into a stream
        _case("decode_f32_token", past=2999, capacity=8192, kv="f32", layers=30, graph=True),
        # the full 8192-row cache
        _case("decode_8192_token", past=8191, capacity=8192, layers=30, graph=True),
        # a stream that has outgrown a 2048-row window, kept as a ring
        _case("decode_ring_token", entry="ring", past=2047, capacity=2048, layers=30, graph=True),
        # the same window cut out of a long cache by the mask tensor
        _case("decode_window_token", past=16334, capacity=16384, mask="causal", window=2048, layers=10, graph=True),
        # 32 streams of ragged lengths served together
        _case("decode_32_streams", batch=32, past=8191, capacity=8192, mask="lengths"),
        # the offline encoder on a 30 s window
        _case("encoder_offline", hq=20, hkv=20, hd=64, nq=1500, layers=8),
        # the realtime encoder as the application calls it: F32 K/V and the
        # window of 750 as an F16 mask tensor
        _case("encoder_realtime", hq=32, hkv=32, hd=64, nq=1500, kv="f32", mask="causal", window=750, layers=8),
        # the offline decoder prompt of a 30 s window on the F32 cache
        _case("prefill_prompt", nq=383, capacity=8192, kv="f32", mask="causal", layers=30),
        # a further 600 rows for a session that holds 3000
        _case("prefill_resume", entry="rope", nq=600, past=3000, capacity=8192, mask="causal", layers=4),
        # a prompt that fills the cache
        _case("prefill_8192", entry="implicit", nq=8192, mask="causal", layers=1),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "streams", "encoder", "encoder", "prefill", "prefill"])
    if kind == "decode":
        # full heads, and the heads of one or two kv groups as a tensor-parallel shard holds them
        hq, hkv = rng.choice([(32, 8), (32, 8), (16, 4), (8, 2), (4, 1)])
        entry = rng.choice(["op", "op", "implicit", "append", "rope", "ring"])
        past = _log(rng, 8, 8191)
        kv = rng.choice(["f16", "f16", "f32"]) if entry in ("op", "implicit") else "f16"
        window = 0
        if entry == "implicit":
            window = _log(rng, 64, 4096)
        elif entry == "op" and rng.random() < 0.3:
            window = _log(rng, 64, 4096)
        cap = past + 1 + rng.randrange(0, 64)
        return _case(None, entry=entry, hq=hq, hkv=hkv, past=past, capacity=cap, kv=kv,
                     mask="causal" if window else "none", window=window, layers=rng.choice([8, 16, 30]), graph=True)
    if kind == "streams":
        past = _log(rng, 256, 8191)
        return _case(None, batch=rng.randrange(2, 33), past=past, capacity=past + 1, mask="lengths",
                     kv=rng.choice(["f16", "f16", "f32"]))
    if kind == "encoder":
        heads = rng.choice([20, 32])
        n = _log(rng, 40, 1500)
        kv = rng.choice(["f16", "f32"])
        if heads == 20 or rng.random() < 0.2:
            return _case(None, hq=heads, hkv=heads, hd=64, nq=n, kv=kv, layers=8)
        return _case(None, entry=rng.choice(["op", "implicit"]), hq=heads, hkv=heads, hd=64, nq=n, kv=kv,
                     mask="causal", window=750, layers=8)
    entry = rng.choice(["op", "implicit", "append", "rope"])
    kv = rng.choice(["f16", "f32"]) if entry in ("op", "implicit") else "f16"
    n = _log(rng, 2, 4000)
    past = rng.choice([0, 0, _log(rng, 16, 4096)])
    hq, hkv = rng.choice([(32, 8), (32, 8), (16, 4), (8, 2)])
    return _case(None, entry=entry, hq=hq, hkv=hkv, nq=n, past=past, capacity=past + n + rng.randrange(0, 64), kv=kv,
                 mask="causal", layers=1 if n > 1000 else 4)


def _lengths(c, seed):
    """Live rows of each stream: between a sixteenth of the cache and all of it."""
    r = random.Random(seed * 7919 + 13)
    n = c["past"] + c["nq"]
    return [r.randint(max(1, n // 16), n) for _ in range(c["batch"])]


def _inputs(c, seed):
    """Buffers in the layout of the application's graph builders: q and dst
    [layer][stream][row][head][hd] F32, K and V [layer][stream][cache row][kv
    head][hd], new rows [layer][stream][row][kv head][hd] F32."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    L, B, D = c["layers"], c["batch"], c["hd"]
    n_kv = c["past"] + c["nq"]
    kvt = torch.float32 if c["kv"] == "f32" else torch.float16

    def normal(shape, dtype=torch.float32):
        return torch.randn(shape, generator=g, device="cuda", dtype=dtype)

    x = {"q": normal((L, B, c["nq"], c["hq"], D)),
         "k": normal((L, B, c["capacity"], c["hkv"], D), kvt),
         "v": normal((L, B, c["capacity"], c["hkv"], D), kvt)}
    if c["entry"] in ("append", "rope", "ring"):
        x["k_new"] = normal((L, B, c["nq"], c["hkv"], D))
        x["v_new"] = normal((L, B, c["nq"], c["hkv"], D))
    if c["entry"] == "rope":
        x["positions"] = (c["past"] + torch.arange(c["nq"], device="cuda", dtype=torch.int32)).repeat(B)
    if c["entry"] == "ring":   # where the oldest row lies
        x["start"] = random.Random(seed).randrange(c["capacity"])
    if c["mask"] == "lengths":
        n = torch.tensor(_lengths(c, seed), device="cuda")[:, None, None]
        live = torch.arange(n_kv, device="cuda")[None, None, :] < n
    elif c["mask"] == "causal":
        live = _causal(c, 0, c["nq"])[None]
    if c["mask"] != "none" and c["entry"] != "implicit":
        x["mask"] = torch.where(live, 0.0, float("-inf")).to(torch.float16).contiguous()
    return x


def _causal(c, r0, r1):
    """[r1 - r0, n_kv]: whether query row r0.. sees the position."""
    i = torch.arange(r0, r1, device="cuda")[:, None] + c["past"]
    j = torch.arange(c["past"] + c["nq"], device="cuda")[None, :]
    live = j <= i
    if c["window"]:
        live &= j > i - c["window"]
    return live


def _call(c, ctx, x, dst, layer):
    """The attention call of one layer: a function of the stream."""
    D, B, nq, n_kv = c["hd"], c["batch"], c["nq"], c["past"] + c["nq"]
    ring = c["entry"] == "ring"
    rows = c["capacity"] if ring else n_kv
    f32 = c["kv"] == "f32"
    qne, qnb = views.decoder_q(nq, c["hq"], D)
    q = vxfa.desc(x["q"][layer].data_ptr(), vxfa.F32, (*qne[:3], B), qnb)
    kne, knb = views.kv_cache(rows, c["hkv"], D, c["capacity"], elt=4 if f32 else 2, batch=B)
    k, v = (vxfa.desc(x[t][layer].data_ptr(), vxfa.F32 if f32 else vxfa.F16, kne, knb) for t in "kv")
    out = vxfa.desc(dst[layer].data_ptr(), vxfa.F32, *views.dst(D, c["hq"], nq, B))
    mask = None
    if "mask" in x:
        mask = vxfa.desc(x["mask"].data_ptr(), vxfa.F16, *views.mask(n_kv, nq, 1, x["mask"].shape[0]))
    scale = 1.0 / math.sqrt(D)
    new = ()
    if "k_new" in x:
        w = c["hkv"] * D
        new = tuple(vxfa.desc(x[t][layer].data_ptr(), vxfa.F32, (w, nq, 1, B), (4, 4 * w, 4 * w * nq, 4 * w * nq))
                    for t in ("k_new", "v_new"))
    if c["entry"] == "op":
        return lambda s: ctx.flash_attn_ext(q, k, v, mask, out, scale, stream=s)
    if c["entry"] == "implicit":
        md = vxfa.mask_desc(vxfa.MASK_CAUSAL, c["window"], c["past"])
        return lambda s: ctx.flash_attn_ext_implicit(q, k, v, md, out, scale, stream=s)
    if c["entry"] == "append":
        return lambda s: ctx.flash_attn_ext_append(q, k, v, *new, mask, out, scale, stream=s)
    if c["entry"] == "rope":
        rope = vxfa.rope(x["positions"].data_ptr(), D, ROPE_BASE)
        return lambda s: ctx.flash_attn_ext_rope(q, k, v, *new, rope, mask, out, scale, stream=s)
    rd = vxfa.ring(x["start"], n_kv)
    return lambda s: ctx.flash_attn_ext_ring(q, k, v, rd, *new, out, scale, stream=s)


def prepare(case, seed):
    x = _inputs(case, seed)
    dst = torch.zeros((case["layers"], case["batch"], case["nq"], case["hq"], case["hd"]), device="cuda")
    ctx = vxfa.Context(torch.cuda.current_device())
    calls = [_call(case, ctx, x, dst, i) for i in range(case["layers"])]
    state = {"x": x, "dst": dst, "ctx": ctx, "calls": calls, "graph": None}
    # what a pass leaves behind: the outputs, and the caches if it stores rows in them
    state["out"] = {"dst": dst}
    if "k_new" in x:
        state["out"].update(k=x["k"], v=x["v"])
    if case["graph"]:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):   # kernels are loaded before a capture
            calls[0](stream.cuda_stream)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            for call in calls:
                call(stream.cuda_stream)
        state["graph"] = graph
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        stream = torch.cuda.current_stream().cuda_stream
        for call in state["calls"]:
            call(stream)
    return state["out"]


def _pairs(c, lengths=None):
    """(query row, position) pairs that take part, over the streams of one layer."""
    if lengths is not None:
        return sum(lengths)
    n_kv = c["past"] + c["nq"]
    if c["mask"] != "causal":
        return c["batch"] * c["nq"] * n_kv
    w = c["window"] or n_kv
    return c["batch"] * sum(min(c["past"] + i + 1, w) for i in range(c["nq"]))


def work(case):
    """Q, the live rows of K and V, the mask and the new rows read once; dst
    and the new rows' cache copies written once. Two products of hd
    multiply-adds for every live pair and query head."""
    c = case
    D, B, nq, n_kv = c["hd"], c["batch"], c["nq"], c["past"] + c["nq"]
    size = 4 if c["kv"] == "f32" else 2
    # (the streams' lengths are drawn with the inputs: their mean)
    lengths = [(max(1, n_kv // 16) + n_kv) // 2] * B if c["mask"] == "lengths" else None
    rows = sum(lengths) if lengths else B * n_kv
    if c["mask"] == "causal" and c["window"]:
        rows = B * min(n_kv, c["window"] + nq - 1)
    new = nq * B if c["entry"] in ("append", "rope", "ring") else 0
    by = 2 * B * nq * c["hq"] * D * 4                     # q, dst
    by += 2 * (rows - new) * c["hkv"] * D * size          # K, V
    by += 2 * new * c["hkv"] * D * (4 + 2)                # new rows: read, stored
    if c["mask"] != "none" and c["entry"] != "implicit":
        by += 2 * n_kv * (B if lengths else nq)
    return {"bytes": by * c["layers"], "flops": 4 * D * c["hq"] * _pairs(c, lengths) * c["layers"]}


def tolerance(case):
    """Against an F32 cache a decode step keeps Q, both products and P in
    F32. Everything else rounds Q, K, V and P to f16 (11 bits) before the
    products, whose sums are F32. Measured against exact(): 4.2e-7 and
    2.0e-4 to 4.1e-4; about four times that is allowed."""
    if case["kv"] == "f32" and case["nq"] == 1:
        return {"rel": 2e-6}
    return {"rel": 1.6e-3}


def _rotate(x, positions):
    """x [..., rows, heads, D] in 64 bits: pair j of a row at position p turns by
    p * base^(-2 j / D), the angle held in F32 as the operation defines it
    (each pair's angle is the previous one's times a factor)."""
    D = x.shape[-1]
    ts = torch.tensor(ROPE_BASE, dtype=torch.float32).pow(-2.0 / D).to(x.device)
    th = positions.float()
    angles = []
    for _ in range(D // 2):
        angles.append(th)
        th = th * ts
    a = torch.stack(angles, -1).double()[:, None, :]      # [rows, 1, D / 2]
    c, s = a.cos(), a.sin()
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], -1).flatten(-2)


def exact(case, seed):
    c, x = case, _inputs(case, seed)
    D, n_kv, group = c["hd"], c["past"] + c["nq"], c["hq"] // c["hkv"]
    lengths = _lengths(c, seed) if c["mask"] == "lengths" else None
    dst = torch.zeros((c["layers"], c["batch"], c["nq"], c["hq"], D), device="cuda", dtype=torch.float64)
    out = {"dst": dst}
    stored = "k_new" in x
    if stored:
        out.update(k=x["k"].double(), v=x["v"].double())
    at = torch.arange(n_kv, device="cuda")
    if c["entry"] == "ring":
        at = (at + x["start"]) % c["capacity"]
    for i in range(c["layers"]):
        for b in range(c["batch"]):
            q = x["q"][i, b].double()
            if c["entry"] == "rope":
                q = _rotate(q, x["positions"][b * c["nq"]:(b + 1) * c["nq"]])
            if stored:
                kn = x["k_new"][i, b].double()
                if c["entry"] == "rope":
                    kn = _rotate(kn, x["positions"][b * c["nq"]:(b + 1) * c["nq"]])
                out["k"][i, b, at[c["past"]:]] = kn
                out["v"][i, b, at[c["past"]:]] = x["v_new"][i, b].double()
            src = out if stored else x
            rows = at[:lengths[b]] if lengths else at
            for h in range(c["hkv"]):
                k, v = src["k"][i, b, :, h][rows].double(), src["v"][i, b, :, h][rows].double()
                for r0 in range(0, c["nq"], 2048):        # bounds the score matrix
                    r1 = min(r0 + 2048, c["nq"])
                    qh = q[r0:r1, h * group:(h + 1) * group].reshape(-1, D)
                    s = qh @ k.t().contiguous() / math.sqrt(D)
                    if c["mask"] == "causal":
                        s.masked_fill_(~_causal(c, r0, r1).repeat_interleave(group, 0), float("-inf"))
                    dst[i, b, r0:r1, h * group:(h + 1) * group] = (s.softmax(-1) @ v).view(r1 - r0, group, D)
    return out

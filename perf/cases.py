"""The work that an inference engine has this library do, as cases that can be timed.

A case is one call (or the fixed group of calls that an engine always makes together) of the
C ABI of include/oom_hip.h: decode steps of a routed-expert layer over FP8, NVFP4 and bf16
expert records, the whole decode layer, dense projections, prefill over FP8 and NVFP4
records, and decode attention over the two KV caches. Shapes are those of this repository's
bench and tests, and generic ones between them.

`prepare` builds what an engine keeps (records, address tables, caches, workspaces) and what
a step is handed (activations, router logits, queries) on the GPU from the seed. `run` makes
the C calls on a stream of its own, with arguments bound once, as an engine behind the C ABI
does. `exact` is plain torch in 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

import homelab_amd as hip

DEV = "cuda"
_STREAM = []


def _stream():
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


# ---- the cases ---------------------------------------------------------------------------


def listed():
    return [
        # one token of a batch-1 chat through a routed-expert layer: the library's headline
        {"name": "decode-1", "kind": "decode", "tokens": 1, "experts": 128, "top_k": 8, "hidden": 4096,
         "inter": 1536, "zipf": 0.0, "x": "bf16"},
        # a small batch of a smaller model whose residual stream is kept in f32, widths that
        # end inside a 1024-column chunk
        {"name": "decode-f32-6", "kind": "decode", "tokens": 6, "experts": 64, "top_k": 6, "hidden": 2048,
         "inter": 1408, "zipf": 0.0, "x": "f32"},
        # a whole decode layer (router, routed and shared experts) for 11 concurrent requests
        {"name": "layer-11", "kind": "layer", "tokens": 11, "experts": 128, "top_k": 8, "hidden": 4096,
         "inter": 1536, "x": "bf16"},
        # the released NVFP4 records: one token, then eight (speculative or concurrent decode)
        {"name": "nvfp4-decode-1", "kind": "nvfp4", "tokens": 1, "experts": 512, "top_k": 10, "hidden": 2560,
         "inter": 640, "x": "bf16"},
        {"name": "nvfp4-decode-8", "kind": "nvfp4", "tokens": 8, "experts": 512, "top_k": 10, "hidden": 2560,
         "inter": 640, "x": "f32"},
        # one dense FP8 projection per layer of a decode step, 24 layers
        {"name": "dense-1", "kind": "dense", "layers": 24, "tokens": 1, "n": 4096, "k": 4096, "weights": "fp8",
         "layout": 0, "x": "bf16", "y": "bf16"},
        # unquantised experts, four tokens
        {"name": "bf16-experts-4", "kind": "bf16", "tokens": 4, "experts": 128, "top_k": 8, "hidden": 4096,
         "inter": 1536, "x": "bf16"},
        # a full prefill chunk with skewed expert popularity, and a ragged one over NVFP4
        {"name": "prefill-2048", "kind": "prefill", "tokens": 2048, "experts": 128, "top_k": 8, "hidden": 4096,
         "inter": 1536, "zipf": 1.1, "x": "bf16", "precision": "exact"},
        {"name": "nvfp4-prefill-500", "kind": "tiled", "tokens": 500, "experts": 512, "top_k": 10, "hidden": 2560,
         "inter": 640, "precision": "exact"},
        # decode attention of a long context, and of a short chat (the smallest call)
        {"name": "attn-32k", "kind": "attn", "kv_len": 32768, "heads": 64, "kv_heads": 8, "page": 16, "q": "bf16"},
        {"name": "attn-700", "kind": "attn", "kv_len": 700, "heads": 32, "kv_heads": 8, "page": 16, "q": "bf16"},
        # a decode step over the compressed KV cache: the new token's rows appended, then
        # attention over a block-sparse selection of 9001 keys
        {"name": "turbo-9001", "kind": "turbo", "kv_len": 9001, "kv_heads": 2, "k_bits": 8, "v_bits": 6,
         "mask": "sparse"},
    ]


def _log(rng, lo, hi, step=1):
    """An integer spread over the logarithm of [lo, hi], a multiple of `step`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, round(v / step) * step)))


def draw(rng):
    kind = rng.choice(["decode", "layer", "nvfp4", "dense", "bf16", "prefill", "tiled", "attn", "turbo"])
    c = {"kind": kind}
    if kind in ("decode", "layer", "bf16"):
        e = rng.choice([16, 32, 60, 64, 96, 128, 160, 256])
        c.update(tokens=_log(rng, 1, 16), experts=e, top_k=rng.choice([2, 4, 6, 8]), hidden=_log(rng, 768, 4096, 16),
                 inter=_log(rng, 256, 1536, 16), x=rng.choice(["bf16", "f32"]))
        if kind == "decode":
            c["tokens"] = _log(rng, 1, 40)
            c["zipf"] = rng.choice([0.0, 1.1])
    elif kind == "nvfp4":
        c.update(tokens=_log(rng, 1, 24), experts=rng.choice([64, 128, 256, 512]), top_k=rng.choice([4, 8, 10]),
                 hidden=_log(rng, 1024, 4096, 16), inter=_log(rng, 256, 1536, 16), x=rng.choice(["bf16", "f32"]))
    elif kind == "dense":
        w = rng.choice(["fp8", "fp8", "bf16"])
        c.update(layers=rng.choice([8, 12, 16]), tokens=_log(rng, 1, 16), n=_log(rng, 128, 8192),
                 k=_log(rng, 640, 6144, 16), weights=w, layout=rng.choice([0, 1, 2]) if w == "fp8" else 0,
                 x=rng.choice(["bf16", "f32"]), y=rng.choice(["bf16", "f32"]))
    elif kind == "prefill":
        c.update(tokens=_log(rng, 48, 2048), experts=rng.choice([32, 64, 128]), top_k=rng.choice([4, 6, 8]),
                 hidden=_log(rng, 1024, 4096, 128), inter=_log(rng, 512, 1536, 128), zipf=rng.choice([0.0, 1.1]),
                 x=rng.choice(["bf16", "f32"]), precision=rng.choice(["exact", "exact", "bf16"]))
    elif kind == "tiled":
        c.update(tokens=_log(rng, 48, 1200), experts=rng.choice([64, 128, 512]), top_k=rng.choice([4, 8, 10]),
                 hidden=_log(rng, 1024, 2560, 64), inter=_log(rng, 320, 1024, 64),
                 precision=rng.choice(["exact", "exact", "bf16"]))
    elif kind == "attn":
        hk = rng.choice([1, 2, 4, 8])
        c.update(kv_len=_log(rng, 200, 65536), heads=hk * rng.choice([1, 4, 6, 8]), kv_heads=hk,
                 page=rng.choice([16, 32, 64]), q=rng.choice(["bf16", "f32"]))
    else:
        kb, vb = rng.choice([(8, 6), (8, 6), (4, 3), (4, 4), (0, 0)])
        c.update(kv_len=_log(rng, 200, 65536), kv_heads=rng.choice([1, 2, 4]), k_bits=kb, v_bits=vb,
                 mask=rng.choice(["all", "sparse"]))
    return c


# ---- inputs ------------------------------------------------------------------------------


def _gen(seed, n=0):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + n * 7919 + 17) & 0x7FFFFFFF)
    return g


def _dt(name):
    return torch.bfloat16 if name == "bf16" else torch.float32


def _al(v, a=256):
    return (v + a - 1) // a * a


def _cdiv(a, b):
    return (a + b - 1) // b


def _randn(g, shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=DEV).to(dtype)


def _logits(c, seed):
    """Router logits N(0, 1), with a Zipf popularity prior over a shuffled order when asked."""
    g = _gen(seed, 1)
    lg = _randn(g, (c["tokens"], c["experts"]))
    if c.get("zipf"):
        rank = torch.randperm(c["experts"], generator=g, device=DEV).float() + 1.0
        lg = lg - c["zipf"] * torch.log(rank)[None, :]
    return lg.contiguous()


def _fp8_parts(H, I):
    """(weight, scale, rows, cols) of gate, up, down in an fp8-e4m3-b128 record, and its stride."""
    at, parts = 0, []
    for n, k in ((I, H), (I, H), (H, I)):
        w = at
        s = _al(w + n * k)
        at = _al(s + _cdiv(n, 128) * _cdiv(k, 128) * 4)
        parts.append((w, s, n, k))
    return parts, _al(at, 4096)


def _quantize(w, layout):
    """e4m3 codes and fp32 scales (absmax / 448) of [.., n, k] weights: one scale a row, one
    per 1 x 128 piece, or one per 128 x 128 block."""
    *b, n, k = w.shape
    if layout == 0:
        s = w.abs().amax(-1).clamp_min(1e-30) / 448.0
        return (w / s[..., None]).to(torch.float8_e4m3fn).view(torch.uint8), s
    r = 1 if layout == 1 else 128
    nb, kb = _cdiv(n, r), _cdiv(k, 128)
    p = torch.nn.functional.pad(w, (0, kb * 128 - k, 0, nb * r - n)).view(*b, nb, r, kb, 128)
    s = p.abs().amax((-3, -1)).clamp_min(1e-30) / 448.0
    q = (p / s[..., :, None, :, None]).to(torch.float8_e4m3fn).view(torch.uint8)
    return q.reshape(*b, nb * r, kb * 128)[..., :n, :k].contiguous(), s.contiguous()


def _fp8_records(E, H, I, g):
    parts, stride = _fp8_parts(H, I)
    buf = torch.zeros((E, stride), dtype=torch.uint8, device=DEV)
    step = max(1, (64 << 20) // (H * I))
    for e0 in range(0, E, step):
        ne = min(step, E - e0)
        for w, s, n, k in parts:
            q, sc = _quantize(torch.randn((ne, n, k), generator=g, device=DEV) * 0.02, 2)
            buf[e0:e0 + ne, w:w + n * k] = q.view(ne, -1)
            sc = sc.reshape(ne, -1).contiguous().view(torch.uint8)
            buf[e0:e0 + ne, s:s + sc.shape[1]] = sc
    return buf


def _nvfp4_parts(H, I):
    """(codes, scales, scale_2 float index, rows, cols) of gate, up, down, and the stride."""
    at, parts = 256, []
    for i, (n, k) in enumerate(((I, H), (I, H), (H, I))):
        w = at
        s = _al(w + n * k // 2)
        at = _al(s + n * k // 16)
        parts.append((w, s, 2 * i, n, k))
    return parts, _al(at, 4096)


def _nvfp4_records(E, H, I, g):
    parts, stride = _nvfp4_parts(H, I)
    buf = torch.zeros((E, stride), dtype=torch.uint8, device=DEV)
    scal = torch.zeros((E, 64), dtype=torch.float32, device=DEV)
    for w, s, s2, n, k in parts:
        buf[:, w:w + n * k // 2] = torch.randint(0, 256, (E, n * k // 2), generator=g, device=DEV, dtype=torch.uint8)
        buf[:, s:s + n * k // 16] = torch.randint(0x28, 0x50, (E, n * k // 16), generator=g, device=DEV,
                                                  dtype=torch.uint8)
        scal[:, s2] = 0.01 + 0.02 * torch.rand((E,), generator=g, device=DEV)
    buf[:, :256] = scal.view(torch.uint8)
    return buf


def _bf16_parts(H, I):
    gw = 0
    uw = _al(gw + I * H * 2)
    dw = _al(uw + I * H * 2)
    return ((gw, I, H), (uw, I, H), (dw, H, I)), _al(dw + I * H * 2, 4096)


def _bf16_records(E, H, I, g):
    parts, stride = _bf16_parts(H, I)
    buf = torch.zeros((E, stride), dtype=torch.uint8, device=DEV)
    for w, n, k in parts:
        for e0 in range(0, E, 16):
            ne = min(16, E - e0)
            v = (torch.randn((ne, n * k), generator=g, device=DEV) * 0.02).to(torch.bfloat16)
            buf[e0:e0 + ne, w:w + n * k * 2] = v.view(torch.uint8)
    return buf


def _addresses(buf):
    return buf.data_ptr() + torch.arange(buf.shape[0], dtype=torch.int64, device=DEV) * buf.shape[1]


def _route(logits, k):
    """Top-k ids (ties to the lower id do not occur in random logits) and renormalised weights, f64."""
    p = torch.softmax(logits.double(), -1)
    w, ids = torch.topk(p, k, dim=-1)
    return ids, w / w.sum(-1, keepdim=True)


def _plan(ids):
    """A step's slots grouped by expert, ids ascending: experts, off, assign_tok, slot_assign."""
    T, k = ids.shape
    flat = ids.reshape(-1)
    order = torch.sort(flat, stable=True).indices
    experts, counts = torch.unique(flat, return_counts=True)
    off = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), counts.cumsum(0)])
    slot = torch.empty_like(order)
    slot[order] = torch.arange(T * k, device=DEV)
    return experts, off.int(), (order // k).int(), slot.view(T, k).int()


def _sign(d):
    i = torch.arange(d, dtype=torch.int64, device=DEV)
    return 1.0 - 2.0 * (((i * 2654435761) & 0xFFFFFFFF) >> 31).double()


def _wht(x):
    """Unnormalised Walsh-Hadamard transform of the last dimension."""
    d, h = x.shape[-1], 1
    while h < d:
        y = x.reshape(*x.shape[:-1], d // (2 * h), 2, h)
        x = torch.stack((y[..., 0, :] + y[..., 1, :], y[..., 0, :] - y[..., 1, :]), -2).reshape(*x.shape[:-1], d)
        h *= 2
    return x


def _encode_rows(x, bits, levels):
    """Cache rows of [rows, 256] vectors: f32 as they are, or rotated codes with fp16 block RMS."""
    if not bits:
        return x.contiguous().view(torch.uint8).reshape(x.shape[0], -1)
    rows, d = x.shape
    y = (_wht(x.double() * _sign(d)) / math.sqrt(d)).view(rows, d // 32, 32)
    sc = (y * y).mean(-1).sqrt().to(torch.float16)
    lv = levels[(1 << bits) - 4:(2 << bits) - 4].double()
    idx = torch.bucketize((y / sc.double()[..., None]).contiguous(), ((lv[1:] + lv[:-1]) / 2).contiguous())
    lane = torch.arange(32, device=DEV, dtype=torch.int64)
    words = torch.stack([(((idx >> j) & 1) << lane).sum(-1) for j in range(bits)], -1)  # [rows, blocks, bits]
    words = torch.where(words >= 1 << 31, words - (1 << 32), words).int().contiguous()
    return torch.cat([sc.contiguous().view(torch.uint8).reshape(rows, -1), words.view(torch.uint8).reshape(rows, -1)],
                     1).contiguous()


def _decode_rows(rows, bits, levels, d=256):
    """[n, row bytes] to [n, d] f64 (in the rotated space for codes)."""
    if not bits:
        return rows.contiguous().view(torch.float32).double()
    n = rows.shape[0]
    nb = d // 32
    sc = rows[:, :2 * nb].contiguous().view(torch.float16).double()
    words = rows[:, 2 * nb:].contiguous().view(torch.int32).view(n, nb, bits).long()
    lane = torch.arange(32, device=DEV, dtype=torch.int64)
    idx = sum((((words[:, :, j, None] >> lane) & 1) << j) for j in range(bits))
    lv = levels[(1 << bits) - 4:(2 << bits) - 4].double()
    return (lv[idx] * sc[..., None]).reshape(n, d)


# ---- what a step is handed, and what an engine keeps ---------------------------------------


def _inputs(c, seed):
    """The case's tensors, from the seed alone."""
    kind, g = c["kind"], _gen(seed)
    t = {}
    if kind in ("decode", "layer", "prefill"):
        t["recs"] = _fp8_records(c["experts"] + (kind == "layer"), c["hidden"], c["inter"], g)
        t["x"] = _randn(g, (c["tokens"], c["hidden"]), _dt(c["x"]))
        if kind == "layer":
            t["router"] = _randn(g, (c["experts"], c["hidden"]), torch.bfloat16) * 0.02
            t["gate"] = _randn(g, (1, c["hidden"]), torch.bfloat16) * 0.02
        else:
            t["logits"] = _logits(c, seed)
    elif kind in ("nvfp4", "tiled"):
        t["recs"] = _nvfp4_records(c["experts"], c["hidden"], c["inter"], g)
        t["x"] = _randn(g, (c["tokens"], c["hidden"]), _dt(c.get("x", "f32")))
        t["logits"] = _logits(c, seed)
    elif kind == "bf16":
        t["recs"] = _bf16_records(c["experts"], c["hidden"], c["inter"], g)
        t["x"] = _randn(g, (c["tokens"], c["hidden"]), _dt(c["x"]))
        t["logits"] = _logits(c, seed)
    elif kind == "dense":
        L, n, k = c["layers"], c["n"], c["k"]
        t["x"] = _randn(g, (c["tokens"], k), _dt(c["x"]))
        if c["weights"] == "bf16":
            t["w"] = torch.stack([(_randn(g, (n, k)) * 0.02).to(torch.bfloat16) for _ in range(L)])
        else:
            qs = [_quantize(_randn(g, (n, k)) * 0.02, c["layout"]) for _ in range(L)]
            t["w"], t["s"] = torch.stack([q for q, _ in qs]), torch.stack([s for _, s in qs])
    elif kind == "attn":
        pages = _cdiv(c["kv_len"], c["page"])
        shape = (pages + 3, c["kv_heads"], c["page"], 128)
        t["q"] = _randn(g, (c["heads"], 128), _dt(c["q"]))
        t["k"] = _randn(g, shape, torch.bfloat16)
        t["v"] = _randn(g, shape, torch.bfloat16)
        t["table"] = torch.randperm(pages + 3, generator=g, device=DEV)[:pages].int()
    else:
        n, hk = c["kv_len"], c["kv_heads"]
        t["levels"] = torch.from_numpy(hip.kv_codebooks()).to(DEV)
        t["k"] = _encode_rows(_randn(g, (n * hk, 256)), c["k_bits"], t["levels"])
        t["v"] = _encode_rows(_randn(g, (n * hk, 256)), c["v_bits"], t["levels"])
        t["q"] = _randn(g, (12 * hk, 256))
        t["k_new"], t["v_new"] = _randn(g, (1, hk, 256)), _randn(g, (1, hk, 256))
        mask = torch.ones(n, dtype=torch.uint8, device=DEV)
        if c["mask"] == "sparse":
            # the first keys, the latest 256, and about 3840 more in blocks of 16
            nb = _cdiv(n, 16)
            pick = torch.zeros(nb, dtype=torch.uint8, device=DEV)
            pick[torch.randperm(nb, generator=g, device=DEV)[:240]] = 1
            mask = pick.repeat_interleave(16)[:n].contiguous()
            mask[:4] = 1
            mask[-256:] = 1
        t["mask"] = mask
    return t


def _fp8_geo(H, I):
    (g, u, d), _ = _fp8_parts(H, I)
    return hip.Fp8Record(H, I, g[0], g[1], u[0], u[1], d[0], d[1])


def _nvfp4_geo(H, I):
    (g, u, d), _ = _nvfp4_parts(H, I)
    geo = hip.Nvfp4Record(H, I, g[0], g[1], u[0], u[1], d[0], d[1])
    geo.scale2[0], geo.scale2[1], geo.scale2[2] = g[2], u[2], d[2]
    return geo


def _code(t):
    return hip.BF16 if t.dtype == torch.bfloat16 else hip.F32


def _bound(name, *args):
    """A C entry point with its arguments converted once: tensors to their addresses, geometries
    by reference, the stream last."""
    fn = getattr(hip.lib(), name)
    out = []
    for a, ty in zip(args + (_stream(),), hip.SIGNATURES[name][1]):
        if isinstance(a, torch.Tensor):
            a = ctypes.c_void_p(a.data_ptr())
        elif isinstance(a, ctypes.Structure):
            a = ctypes.byref(a)
        elif isinstance(a, torch.cuda.Stream):
            a = ctypes.c_void_p(a.cuda_stream)
        elif a is not None:
            a = ty(a)
        out.append(a)
    return fn, tuple(out)


def _zeros(n):
    return torch.zeros(max(int(n), 256), dtype=torch.uint8, device=DEV)


def prepare(case, seed):
    c, t = case, _inputs(case, seed)
    kind = c["kind"]
    calls, out = [], None
    if "tokens" in c and kind != "dense":
        T, E, k, H, I = c["tokens"], c["experts"], c["top_k"], c["hidden"], c["inter"]
        t["addr"] = _addresses(t["recs"])
        t["ids"] = torch.empty((T, k), dtype=torch.int32, device=DEV)
        t["weights"] = torch.empty((T, k), dtype=torch.float32, device=DEV)
        odt = _dt(c.get("x", "bf16"))
        t["out"] = torch.empty((T, H), dtype=odt, device=DEV)
        out = [t["ids"], t["weights"], t["out"]]
    if kind in ("decode", "nvfp4", "prefill"):
        geo = _nvfp4_geo(H, I) if kind == "nvfp4" else _fp8_geo(H, I)
        name = {"decode": "oom_moe_decode_fp8", "nvfp4": "oom_moe_decode_nvfp4", "prefill": "oom_moe_prefill_fp8"}[kind]
        size = getattr(hip.lib(), name + "_workspace_size")(T, E, k, ctypes.byref(geo))
        t["ws"], t["geo"] = _zeros(size), geo
        more = ()
        if kind == "prefill":
            more = (hip.EXPERT_EXACT if c["precision"] == "exact" else hip.EXPERT_BF16,)
        calls.append(_bound(name, t["logits"], t["x"], _code(t["x"]), t["addr"], T, E, k, geo, *more, t["ids"],
                            t["weights"], t["out"], _code(t["out"]), t["ws"], size))
    elif kind == "layer":
        geo = _fp8_geo(H, I)
        size = hip.moe_layer_decode_fp8_workspace_size(T, E, k, geo, geo)
        t["ws"], t["geo"], t["shared"] = _zeros(size), geo, t["addr"][E:E + 1].clone()
        calls.append(_bound("oom_moe_layer_decode_fp8", t["x"], _code(t["x"]), t["router"], t["addr"], T, E, k, geo,
                            t["shared"], geo, t["gate"], t["ids"], t["weights"], t["out"], _code(t["out"]), t["ws"],
                            size))
    elif kind in ("bf16", "tiled"):
        ids, w = _route(t["logits"], k)
        experts, t["off"], t["tok"], t["slot"] = _plan(ids)
        n_e, t["w"] = int(experts.numel()), w.float().contiguous()
        most = int((t["off"][1:] - t["off"][:-1]).max())
        t["sel"] = t["addr"][experts].contiguous()
        t["h"] = torch.empty((T * k, I), dtype=torch.float32, device=DEV)
        t["y"] = torch.empty((T * k, H), dtype=torch.float32, device=DEV)
        if kind == "bf16":
            (gw, _, _), (uw, _, _), (dw, _, _) = _bf16_parts(H, I)[0]
            geo = t["geo"] = hip.Bf16Record(H, I, gw, uw, dw)
            calls.append(_bound("oom_moe_gate_up_bf16", t["sel"], t["off"], t["tok"], n_e, t["x"], _code(t["x"]),
                                t["h"], geo))
            calls.append(_bound("oom_moe_down_bf16", t["sel"], t["off"], n_e, t["h"], t["y"], geo))
        else:
            t["g"], t["u"] = torch.empty_like(t["h"]), torch.empty_like(t["h"])
            prec = hip.EXPERT_EXACT if c["precision"] == "exact" else hip.EXPERT_BF16
            for (wo, so, s2, n, kk), rows, src, dst in zip(_nvfp4_parts(H, I)[0], (t["tok"], t["tok"], None),
                                                           (t["x"], t["x"], t["h"]), (t["g"], t["u"], t["y"])):
                calls.append(_bound("oom_moe_tiled_nvfp4", t["sel"], t["off"], rows, n_e, most, src, dst, n, kk, wo,
                                    so, s2, prec))
            calls.insert(2, _bound("oom_moe_swiglu_range", t["g"], t["u"], t["h"], 0, T * k * I))
        calls.append(_bound("oom_moe_combine_slots", t["y"], t["slot"], t["w"], t["out"], _code(t["out"]), T, H, k))
        out = [t["out"]]
    elif kind == "dense":
        T, n, k = c["tokens"], c["n"], c["k"]
        t["y"] = torch.empty((c["layers"], T, n), dtype=_dt(c["y"]), device=DEV)
        bf = c["weights"] == "bf16"
        size = hip.gemv_bf16_workspace_size(T, n, k) if bf else hip.gemv_fp8_workspace_size(T, n, k)
        t["ws"] = _zeros(size)
        for i in range(c["layers"]):
            if bf:
                calls.append(_bound("oom_gemv_bf16", t["x"], _code(t["x"]), t["w"][i], t["y"][i], _code(t["y"]), T, n,
                                    k, t["ws"], t["ws"].numel()))
            else:
                calls.append(_bound("oom_gemv_fp8", t["x"], _code(t["x"]), t["w"][i], t["s"][i], c["layout"],
                                    t["y"][i], _code(t["y"]), T, n, k, t["ws"], t["ws"].numel()))
        out = [t["y"]]
    elif kind == "attn":
        H, hk, n = c["heads"], c["kv_heads"], c["kv_len"]
        t["out"] = torch.empty((H, 128), dtype=_dt(c["q"]), device=DEV)
        size = hip.attn_decode_workspace_size(n, H, hk, 128)
        t["ws"] = _zeros(size)
        calls.append(_bound("oom_attn_decode_paged", t["q"], _code(t["q"]), t["k"], t["v"], t["table"],
                            t["k"].shape[0], c["page"], n, H, hk, 128, 1.0 / math.sqrt(128.0), t["out"],
                            _code(t["out"]), t["ws"], t["ws"].numel()))
        out = [t["out"]]
    else:
        hk, n = c["kv_heads"], c["kv_len"]
        t["out"] = torch.empty((12 * hk, 256), dtype=torch.float32, device=DEV)
        t["ws"] = _zeros(hip.attn_decode_turbo_workspace_size(12 * hk, hk, 256, n))
        for src, dst, bits in ((t["k_new"], t["k"], c["k_bits"]), (t["v_new"], t["v"], c["v_bits"])):
            calls.append(_bound("oom_kv_append", src, dst, n - 1, 1, hk, 256, bits, t["levels"]))
        calls.append(_bound("oom_attn_decode_turbo", t["q"], t["k"], t["v"], c["k_bits"], c["v_bits"], t["levels"],
                            t["mask"], 12 * hk, hk, 256, n, 1.0 / 16.0, t["out"], t["ws"], t["ws"].numel()))
        out = [t["k"][-hk:], t["v"][-hk:], t["out"]]
    torch.cuda.synchronize()  # inputs were made on torch's stream, the steps run on their own
    return {"calls": calls, "out": out, "keep": t}


def run(state):
    for fn, args in state["calls"]:
        rc = fn(*args)
        if rc:
            hip.check(rc)
    return state["out"]


# ---- what a pass cannot do without ---------------------------------------------------------


def _distinct(c):
    """Distinct experts of a typical step."""
    r = np.random.default_rng(5)
    lg = r.standard_normal((c["tokens"], c["experts"]))
    if c.get("zipf"):
        lg -= c["zipf"] * np.log(r.permutation(c["experts"]) + 1.0)
    return len(np.unique(np.argpartition(-lg, c["top_k"] - 1, axis=1)[:, :c["top_k"]]))


def work(case):
    c, kind = case, case["kind"]
    es = {"bf16": 2, "f32": 4}
    if kind == "dense":
        T, n, k, L = c["tokens"], c["n"], c["k"], c["layers"]
        sc = {0: n, 1: n * _cdiv(k, 128), 2: _cdiv(n, 128) * _cdiv(k, 128)}[c["layout"]] * 4
        w = n * k * 2 if c["weights"] == "bf16" else n * k + sc
        return {"bytes": L * (w + T * n * es[c["y"]]) + T * k * es[c["x"]], "flops": 2.0 * L * T * n * k}
    if kind == "attn":
        n = c["kv_len"]
        return {"bytes": 4 * n * c["kv_heads"] * 128 + 4 * _cdiv(n, c["page"]) + 2 * c["heads"] * 128 * es[c["q"]],
                "flops": 4.0 * c["heads"] * n * 128}
    if kind == "turbo":
        n, hk = c["kv_len"], c["kv_heads"]
        seen = n if c["mask"] == "all" else min(n, 4100)
        rb = sum(16 + 32 * b if b else 1024 for b in (c["k_bits"], c["v_bits"]))
        return {"bytes": seen * hk * rb + n + 2 * 12 * hk * 1024 + hk * (rb + 2048), "flops": 4.0 * 12 * hk * seen * 256}
    T, k, H, I = c["tokens"], c["top_k"], c["hidden"], c["inter"]
    d = _distinct(c)
    per = 3 * H * I
    per = {"nvfp4": per / 2 + per / 16, "tiled": per / 2 + per / 16, "bf16": per * 2}.get(kind, per + per / 4096)
    io = T * H * 2 * es[c.get("x", "f32")] + T * k * 8
    rows = T * k
    if kind == "layer":
        d, rows, io = d + 1, rows + T, io + (c["experts"] + 1) * H * 2
    elif kind in ("decode", "nvfp4", "prefill"):
        io += T * c["experts"] * 4
    return {"bytes": d * per + io, "flops": 6.0 * rows * H * I}


# ---- tolerances and the exact results -------------------------------------------------------


def tolerance(case):
    """Sums in fp32 in another order, and where the result is bf16 its rounding (unit 2^-9),
    which another order of summation moves for a few outputs."""
    c = case
    if c["kind"] == "prefill":
        # e4m3 matrix-core block sums keep about 13 bits of a group's largest product; h in
        # two bf16 terms (16 bits), or one
        return {"rel": 4e-3 if c["precision"] == "bf16" or c["x"] == "bf16" else 1.2e-3, "max": 0.05}
    kind_out = c.get("y") or c.get("x") or c.get("q") or ("bf16" if c["kind"] == "tiled" else "f32")
    if kind_out == "bf16":
        return {"rel": 2e-3, "max": 0.02}
    if c["kind"] == "tiled" and c["precision"] == "bf16":
        return {"rel": 2e-3, "max": 0.02}
    return {"rel": 1e-5, "max": 2e-4}


def _fp8_weight(rec, w, s, n, k, r=128):
    q = rec[w:w + n * k].view(torch.float8_e4m3fn).double().view(n, k)
    nb, kb = _cdiv(n, r), _cdiv(k, 128)
    sc = rec[s:s + nb * kb * 4].view(torch.float32).double().view(nb, kb)
    return q * sc.repeat_interleave(r, 0)[:n].repeat_interleave(128, 1)[:, :k]


_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _nvfp4_weight(rec, w, s, s2, n, k):
    lut = torch.tensor(_E2M1 + [-v for v in _E2M1], dtype=torch.float64, device=DEV)
    b = rec[w:w + n * k // 2].view(n, k // 2).long()
    v = torch.stack((lut[b & 15], lut[b >> 4]), -1).view(n, k)
    sc = rec[s:s + n * k // 16].view(torch.float8_e4m3fn).double().view(n, k // 16)
    return v * sc.repeat_interleave(16, 1) * rec[4 * s2:4 * s2 + 4].view(torch.float32).double()


def _weights(c, rec):
    H, I = c["hidden"], c["inter"]
    if c["kind"] in ("nvfp4", "tiled"):
        return [_nvfp4_weight(rec, *p) for p in _nvfp4_parts(H, I)[0]]
    if c["kind"] == "bf16":
        return [rec[w:w + n * k * 2].view(torch.bfloat16).double().view(n, k) for w, n, k in _bf16_parts(H, I)[0]]
    return [_fp8_weight(rec, *p) for p in _fp8_parts(H, I)[0]]


def _ffn(c, rec, x, h_of=lambda h: h):
    g, u, d = _weights(c, rec)
    gv, uv = x @ g.T, x @ u.T
    return h_of(gv * torch.sigmoid(gv) * uv) @ d.T


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    kind = c["kind"]
    if kind == "dense":
        x, ys = t["x"].double(), []
        for i in range(c["layers"]):
            if c["weights"] == "bf16":
                w = t["w"][i].double()
            else:
                n, k, sc = c["n"], c["k"], t["s"][i].double()
                if c["layout"] == 0:
                    sc = sc[:, None]
                else:
                    sc = sc.repeat_interleave(1 if c["layout"] == 1 else 128, 0)[:n].repeat_interleave(128, 1)[:, :k]
                w = t["w"][i].view(torch.float8_e4m3fn).double() * sc
            ys.append(x @ w.T)
        return [torch.stack(ys)]
    if kind == "attn":
        n, hk = c["kv_len"], c["kv_heads"]
        j = torch.arange(n, device=DEV)
        page, at = t["table"][j // c["page"]].long(), j % c["page"]
        outs, G = [], c["heads"] // hk
        for h in range(hk):
            q = t["q"][h * G:(h + 1) * G].double()
            p = torch.softmax(q @ t["k"][page, h, at].double().T / math.sqrt(128.0), -1)
            outs.append(p @ t["v"][page, h, at].double())
        return [torch.cat(outs)]
    if kind == "turbo":
        n, hk = c["kv_len"], c["kv_heads"]
        t["k"][-hk:] = _encode_rows(t["k_new"].view(hk, 256), c["k_bits"], t["levels"])
        t["v"][-hk:] = _encode_rows(t["v_new"].view(hk, 256), c["v_bits"], t["levels"])
        rot = c["k_bits"] != 0
        q = t["q"].double()
        if rot:
            q = _wht(q * _sign(256)) / 16.0
        seen = t["mask"].nonzero()[:, 0]
        k = t["k"].view(n, hk, -1)
        v = t["v"].view(n, hk, -1)
        outs = []
        for h in range(hk):
            kd = _decode_rows(k[seen, h], c["k_bits"], t["levels"])
            vd = _decode_rows(v[seen, h], c["v_bits"], t["levels"])
            outs.append(torch.softmax(q[12 * h:12 * h + 12] @ kd.T / 16.0, -1) @ vd)
        o = torch.cat(outs)
        if rot:
            o = _wht(o) * _sign(256) / 16.0
        return [None, None, o]
    E, k = c["experts"], c["top_k"]
    x = t["x"].double()
    logits = x @ t["router"].double().T if kind == "layer" else t["logits"]
    ids, w = _route(logits, k)
    h_of = lambda h: h  # noqa: E731
    if kind == "prefill":
        s = t["x"].float().abs().amax(-1, keepdim=True) / 448.0
        x = (t["x"].float() / s).to(torch.float8_e4m3fn).double() * s.double()
    if c.get("precision") == "bf16":
        h_of = lambda h: h.float().to(torch.bfloat16).double()  # noqa: E731
        if kind == "tiled":
            x = t["x"].to(torch.bfloat16).double()
    out = torch.zeros_like(x)
    for e in range(E):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        if tok.numel():
            out[tok] += w[tok, slot, None] * _ffn(c, t["recs"][e], x[tok], h_of)
    if kind == "layer":
        gate = torch.sigmoid(x @ t["gate"].double().T)
        out = out + gate * _ffn(c, t["recs"][E], x)
    return [out] if kind in ("bf16", "tiled") else [None, w, out]

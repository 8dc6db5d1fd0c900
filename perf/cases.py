"""Performance cases of the attention path: what its callers run, at their sizes and around them.

Every case goes through the Python front end (sam_hip, sam_encoder). Seven kinds of work:

    relpos   attention_relpos over q, kT, v and the rel-pos table (SAM's windowed and global layers)
    memory   rope_attention (SAM 2.1 memory attention: self over one frame, cross over up to 7 and pointers)
    sam3     qkv_rope and flash_attn, a SAM 3 ViT layer between its linears
    flash    flash_attn on the q, k, v slices of a packed projection (Hiera's windows)
    sdpa     sdpa with an additive mask (DETR's text padding, TinyViT's biases)
    deform   deform_core (Grounding DINO's encoder and decoder layers)
    block    sam_encoder.block, a whole ViT block with its linears

listed() holds the sizes that the models have; draw() gives others of the same ranges.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.abspath("sam-rs_amd"))
import sam_encoder  # noqa: E402
import sam_hip  # noqa: E402

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
DEV = "cuda"


def listed():
    return [
        # DETR's cross-attention to the text tokens: one prompt, 200 queries. The smallest call, latency.
        {"name": "detr_text_f16", "kind": "sdpa", "dtype": "f16", "b": 1, "h": 8, "lq": 200, "lk": 32, "d": 32,
         "mask": "padding"},
        # Grounding DINO-tiny's decoder layer at 800 x 1333: 900 queries with box references.
        {"name": "dino_decoder_f32", "kind": "deform", "dtype": "f32", "ih": 800, "iw": 1333, "queries": 900},
        # Its encoder layer: every one of the 22 223 positions samples around itself.
        {"name": "dino_encoder_f32", "kind": "deform", "dtype": "f32", "ih": 800, "iw": 1333, "queries": 0},
        # SAM ViT-H, one image: a windowed layer (25 windows x 16 heads) and a global one. 28 + 4 make an encoder.
        {"name": "vit_h_window_f16", "kind": "relpos", "dtype": "f16", "bh": 400, "gh": 14, "gw": 14, "hd": 80},
        {"name": "vit_h_global_f16", "kind": "relpos", "dtype": "f16", "bh": 16, "gh": 64, "gw": 64, "hd": 80},
        # An 800 x 592 image at patch 16 without padding: a grid that no dedicated kernel has.
        {"name": "grid_37x50_f16", "kind": "relpos", "dtype": "f16", "bh": 16, "gh": 37, "gw": 50, "hd": 80},
        # SAM ViT-B in f32, the reference's exact mode: both layer types.
        {"name": "vit_b_window_f32", "kind": "relpos", "dtype": "f32", "bh": 300, "gh": 14, "gw": 14, "hd": 64},
        {"name": "vit_b_global_f32", "kind": "relpos", "dtype": "f32", "bh": 12, "gh": 64, "gw": 64, "hd": 64},
        # Hiera-L's 14 x 14 windows at head dim 72.
        {"name": "hiera_window_bf16", "kind": "flash", "dtype": "bf16", "b": 64, "l": 196, "h": 4, "d": 72},
        # SAM 3 ViT, one 1008 x 1008 image: a windowed layer, 9 windows of 24 x 24.
        {"name": "sam3_window_f16", "kind": "sam3", "dtype": "f16", "nw": 9, "side": 24, "h": 16, "d": 64},
        # SAM 2.1 video step: cross-attention over the full memory of 7 frames and 16 object pointers of 4 tokens.
        {"name": "memory_cross_f16", "kind": "memory", "dtype": "f16", "side": 64, "frames": 7, "pointers": 64},
        # A whole windowed block of the ViT-B encoder, one image.
        {"name": "vit_b_block_f16", "kind": "block", "dtype": "f16", "batch": 1, "grid": 64, "heads": 12, "hd": 64,
         "window": 14},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _drawn(rng):
    kind = rng.choice(["relpos", "relpos", "relpos", "memory", "sam3", "flash", "sdpa", "deform", "block"])
    if kind == "relpos":
        dtype = rng.choice(["f16", "f16", "bf16", "f32"])
        gh = _log(rng, 7, 64)
        gw = gh if rng.random() < 0.4 else _log(rng, 7, 64)
        heads = rng.choice([12, 16])
        # a few thousand tokens in all, as an image or a small batch of them has
        n = max(1, int(round(_log(rng, 1000, 10000) / (gh * gw))))
        return {"kind": kind, "dtype": dtype, "bh": n * heads, "gh": gh, "gw": gw, "hd": rng.choice([64, 80])}
    if kind == "memory":
        return {"kind": kind, "dtype": rng.choice(["f16", "f16", "bf16"]), "side": rng.choice([32, 48, 57, 64]),
                "frames": rng.randint(1, 7), "pointers": 4 * rng.randint(0, 16)}
    if kind == "sam3":
        side = rng.randint(12, 72)
        nw = max(1, int(round(_log(rng, 600, 10000) / (side * side))))
        return {"kind": kind, "dtype": rng.choice(["f16", "bf16"]), "nw": nw, "side": side, "h": 16, "d": 64}
    if kind == "flash":
        l = _log(rng, 16, 1024)
        b = max(1, int(round(_log(rng, 1024, 16384) / l)))
        return {"kind": kind, "dtype": rng.choice(["f16", "bf16"]), "b": b, "l": l, "h": rng.choice([1, 2, 4, 8]),
                "d": rng.choice([64, 72, 96])}
    if kind == "sdpa":
        if rng.random() < 0.5:
            return {"kind": kind, "dtype": rng.choice(["f16", "bf16"]), "b": rng.randint(1, 4), "h": 8,
                    "lq": _log(rng, 1, 900), "lk": _log(rng, 4, 300), "d": 32, "mask": "padding"}
        side = rng.choice([7, 14])
        return {"kind": kind, "dtype": rng.choice(["f16", "f32"]), "b": _log(rng, 1, 80), "h": rng.choice([4, 5, 10]),
                "lq": side * side, "lk": side * side, "d": 32, "mask": "bias"}
    if kind == "deform":
        ih = _log(rng, 320, 800)
        iw = min(1333, max(320, int(ih * rng.uniform(0.75, 1.7))))
        return {"kind": kind, "dtype": "f32", "ih": ih, "iw": iw, "queries": rng.choice([0, rng.randint(100, 900)])}
    heads = rng.choice([12, 16])
    return {"kind": "block", "dtype": rng.choice(["f16", "bf16"]), "batch": rng.choice([1, 2]),
            "grid": rng.randint(28, 64), "heads": heads, "hd": 64 if heads == 12 else rng.choice([64, 80]),
            "window": rng.choice([14, 14, 0])}


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / (1e14 if case["dtype"] == "f32" else 1e15))


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _drawn(rng)
        if _cost(case) <= most:
            return case


# ------------------------------------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _rn(g, dtype, *shape, std=1.0):
    return (std * torch.randn(*shape, device=DEV, generator=g)).to(dtype)


def _levels(case):
    """The four feature levels of a Grounding DINO image: strides 8, 16, 32, 64."""
    h, w = -(-case["ih"] // 8), -(-case["iw"] // 8)
    out = []
    for _ in range(4):
        out.append((h, w))
        h, w = -(-h // 2), -(-w // 2)
    return out


def _axial_tables(w, n, d, theta=10000.0):
    """cos and sin [n, d] of 2-D axial RoPE over a grid of row length w: half the pairs by column, half by row."""
    pairs = d // 4
    inv = torch.tensor([theta ** (-i / pairs) for i in range(pairs)], dtype=torch.float64)
    t = torch.arange(n)
    ang = torch.cat([(t % w).double()[:, None] * inv, torch.div(t, w, rounding_mode="floor").double()[:, None] * inv], 1)
    ang = ang.repeat_interleave(2, 1)
    return torch.cos(ang).float().to(DEV), torch.sin(ang).float().to(DEV)


def _refs(case, levels, g):
    """Encoder: the centre of each position, level by level. Decoder: boxes (cx, cy, w, h)."""
    if case["queries"]:
        xy = torch.rand(1, case["queries"], 1, 2, device=DEV, generator=g)
        wh = 0.02 + 0.4 * torch.rand(1, case["queries"], 1, 2, device=DEV, generator=g)
        return torch.cat([xy, wh], 3).expand(1, case["queries"], 4, 4).contiguous()
    pts = []
    for h, w in levels:
        ys = (torch.arange(h, device=DEV, dtype=torch.float32) + 0.5) / h
        xs = (torch.arange(w, device=DEV, dtype=torch.float32) + 0.5) / w
        pts.append(torch.stack([xs[None, :].expand(h, w), ys[:, None].expand(h, w)], 2).reshape(h * w, 2))
    p = torch.cat(pts)
    return p[None, :, None, :].expand(1, p.shape[0], 4, 2).contiguous()


def _mask(case, g, dtype):
    if case["mask"] == "bias":
        return _rn(g, dtype, 1, case["h"], case["lq"], case["lk"], std=0.5)
    keep = torch.ones(case["b"], 1, 1, case["lk"], device=DEV, dtype=torch.bool)
    keep[..., 1:] = torch.rand(case["b"], 1, 1, case["lk"] - 1, device=DEV, generator=g) < 0.8
    zero = torch.zeros((), device=DEV, dtype=dtype)
    return torch.where(keep, zero, torch.full_like(zero, float("-inf")))


BLOCK_NAMES = ("norm1_w", "norm1_b", "qkv_w", "qkv_b", "proj_w", "proj_b", "rel", "norm2_w", "norm2_b", "lin1_w",
               "lin1_b", "lin2_w", "lin2_b")


def _block_tensors(case, g, dtype):
    c, hd = case["heads"] * case["hd"], case["hd"]
    inp = case["window"] or case["grid"]
    shapes = {"norm1_w": (c,), "norm1_b": (c,), "qkv_w": (3 * c, c), "qkv_b": (3 * c,), "proj_w": (c, c),
              "proj_b": (c,), "rel": (2 * (2 * inp - 1), hd), "norm2_w": (c,), "norm2_b": (c,),
              "lin1_w": (4 * c, c), "lin1_b": (4 * c,), "lin2_w": (c, 4 * c), "lin2_b": (c,)}
    p = {n: _rn(g, dtype, *shapes[n], std=0.02) for n in BLOCK_NAMES}
    p["norm1_w"] = (1 + p["norm1_w"]).to(dtype)
    p["norm2_w"] = (1 + p["norm2_w"]).to(dtype)
    return p


def _inputs(case, seed):
    g, dt, kind = _gen(seed), DTYPES[case["dtype"]], case["kind"]
    if kind == "relpos":
        bh, h, w, hd = case["bh"], case["gh"], case["gw"], case["hd"]
        n = h * w
        return {"q": _rn(g, dt, bh, n, hd), "kt": _rn(g, dt, bh, hd, n), "v": _rn(g, dt, bh, n, hd),
                "table": _rn(g, dt, 2 * h - 1 + 2 * w - 1, hd, std=0.02)}
    if kind == "memory":
        n = case["side"] ** 2
        m = case["frames"] * n + case["pointers"]
        cos, sin = _axial_tables(case["side"], n, 256)
        return {"q": _rn(g, dt, 1, n, 256), "k": _rn(g, dt, 1, m, 256), "v": _rn(g, dt, 1, m, 256), "cos": cos,
                "sin": sin}
    if kind == "sam3":
        n, c = case["side"] ** 2, case["h"] * case["d"]
        cos, sin = _axial_tables(case["side"], n, case["d"])
        return {"y": _rn(g, dt, case["nw"] * n, 3 * c), "bias": _rn(g, dt, 3 * c, std=0.02), "cos": cos, "sin": sin}
    if kind == "flash":
        return {"qkv": _rn(g, dt, case["b"], case["l"], 3, case["h"], case["d"])}
    if kind == "sdpa":
        b, h, d = case["b"], case["h"], case["d"]
        q, k, v = (_rn(g, dt, b, h, n, d) for n in (case["lq"], case["lk"], case["lk"]))
        return {"q": q, "k": k, "v": v, "mask": _mask(case, g, dt)}
    if kind == "deform":
        levels = _levels(case)
        s = sum(h * w for h, w in levels)
        n = case["queries"] or s
        # encoder offsets of about two pixels, decoder ones of about a quarter of the box over 4 points
        return {"value": _rn(g, dt, 1, s, 8, 32), "offsets": _rn(g, dt, 1, n, 8, 4, 4, 2, std=2.0),
                "logits": _rn(g, dt, 1, n, 8, 4, 4), "refs": _refs(case, levels, g)}
    t = _block_tensors(case, g, dt)
    c = case["heads"] * case["hd"]
    t["x"] = _rn(g, dt, case["batch"], case["grid"], case["grid"], c)
    t["next_w"] = (1 + _rn(g, dt, c, std=0.02)).to(dt)
    t["next_b"] = _rn(g, dt, c, std=0.02)
    return t


def prepare(case, seed):
    t = _inputs(case, seed)
    state = {"case": case, "t": t}
    if case["kind"] == "deform":
        state["levels"] = _levels(case)
    elif case["kind"] == "flash":
        state["qkv"] = tuple(t["qkv"][:, :, i] for i in range(3))
    elif case["kind"] == "block":
        window = case["window"]
        p = sam_encoder.BlockWeights(*[t[n] for n in BLOCK_NAMES], window)
        nxt = sam_encoder.BlockWeights(t["next_w"], t["next_b"], *[t[n] for n in BLOCK_NAMES[2:]], window)
        xn = F.layer_norm(t["x"], (t["x"].shape[3],), t["norm1_w"], t["norm1_b"], 1e-6)
        state.update(p=p, nxt=nxt, xn=xn)
    return state


def run(state):
    case, t = state["case"], state["t"]
    kind = case["kind"]
    if kind == "relpos":
        return sam_hip.attention_relpos(t["q"], t["kt"], t["v"], t["table"], case["gh"], case["gw"],
                                        case["hd"] ** -0.5)
    if kind == "memory":
        return sam_hip.rope_attention(t["q"], t["k"], t["v"], t["cos"], t["sin"], case["pointers"])
    if kind == "sam3":
        nw, n, h, d = case["nw"], case["side"] ** 2, case["h"], case["d"]
        qkv = sam_hip.qkv_rope(t["y"], t["bias"], t["cos"], t["sin"], n, h, d)
        return sam_hip.flash_attn(*(qkv[i].view(nw, n, h, d) for i in range(3)))
    if kind == "flash":
        return sam_hip.flash_attn(*state["qkv"])
    if kind == "sdpa":
        return sam_hip.sdpa(t["q"], t["k"], t["v"], t["mask"])
    if kind == "deform":
        return sam_hip.deform_core(t["value"], t["offsets"], t["logits"], t["refs"], state["levels"])
    return sam_encoder.block(t["x"], state["xn"], state["p"], case["heads"], state["nxt"])


# --------------------------------------------------------------------------------- work and tolerances


def work(case):
    e = 4 if case["dtype"] == "f32" else 2
    kind = case["kind"]
    if kind == "relpos":
        bh, n, hd = case["bh"], case["gh"] * case["gw"], case["hd"]
        table = 2 * (case["gh"] + case["gw"]) * hd
        return {"bytes": e * (4 * bh * n * hd + table), "flops": 4.0 * bh * n * n * hd}
    if kind == "memory":
        n = case["side"] ** 2
        m = case["frames"] * n + case["pointers"]
        return {"bytes": e * 256 * (2 * n + 2 * m) + 8 * n * 256, "flops": 4.0 * n * m * 256}
    if kind == "sam3":
        n, c = case["side"] ** 2, case["h"] * case["d"]
        return {"bytes": e * case["nw"] * n * 4 * c + e * 3 * c + 8 * n * case["d"],
                "flops": 4.0 * case["nw"] * n * n * c}
    if kind == "flash":
        b, l, c = case["b"], case["l"], case["h"] * case["d"]
        return {"bytes": e * 4 * b * l * c, "flops": 4.0 * b * l * l * c}
    if kind == "sdpa":
        b, h, lq, lk, d = (case[k] for k in ("b", "h", "lq", "lk", "d"))
        mask = b * lk if case["mask"] == "padding" else h * lq * lk
        return {"bytes": e * (2 * b * h * d * (lq + lk) + mask), "flops": 4.0 * b * h * lq * lk * d}
    if kind == "deform":
        s = sum(h * w for h, w in _levels(case))
        n = case["queries"] or s
        return {"bytes": e * (256 * s + n * (8 * 16 * 3 + 256 + (16 if case["queries"] else 8))),
                "flops": 8.0 * n * 256 * 16}
    c, g, b, ws = case["heads"] * case["hd"], case["grid"], case["batch"], case["window"] or case["grid"]
    tokens = b * g * g
    keys = b * (-(-g // ws) * ws) ** 2 * ws * ws
    return {"bytes": e * (4 * tokens * c + 12 * c * c), "flops": 24.0 * tokens * c * c + 4.0 * keys * c}


def tolerance(case):
    """About four times the largest error against 64 bits that was measured over each kind's range."""
    kind, half = case["kind"], case["dtype"] == "f16"
    if kind == "deform":  # sampling locations in f32: 3.9e-6
        return {"rel": 1.6e-5}
    if case["dtype"] == "f32":  # 1.2e-6 over 4096 keys
        return {"rel": 5e-6}
    if kind == "sam3":  # q and k rounded after the rotation: 1.0e-3 in f16, 8 times that in bf16
        return {"rel": 4e-3 if half else 3.2e-2}
    if kind == "block":  # 3.9e-4 in f16, 3.3e-3 in bf16
        return {"rel": 1.6e-3 if half else 1.3e-2}
    if kind == "memory":  # the same rotation: 4.3e-4 in f16
        return {"rel": 1.8e-3 if half else 1.4e-2}
    return {"rel": 1.2e-3 if half else 7e-3}  # 2.9e-4 and 1.7e-3


# ------------------------------------------------------------------------------------------- in 64 bits


def _attend(q, k, v, scale, bias=None):
    """softmax(scale q k^T + bias) v in float64 on [N, L, D], a slice of heads at a time; bias(i, j) gives a slice's."""
    out = []
    step = max(1, int(2e8 // (q.shape[1] * k.shape[1])))
    for i in range(0, q.shape[0], step):
        j = min(q.shape[0], i + step)
        s = torch.bmm(q[i:j].double() * scale, k[i:j].double().transpose(1, 2).contiguous())
        if bias is not None:
            s += bias(i, j)
        out.append(torch.bmm(torch.softmax(s, 2), v[i:j].double().contiguous()))
    return torch.cat(out)


def _rel_bias(q, table, h, w):
    """q . Th[i - kh + h - 1] + q . Tw[j - kw + w - 1] in float64, [N, h*w, h*w]."""
    t = table.double()
    r = torch.arange(h, device=DEV)
    c = torch.arange(w, device=DEV)
    th = t[: 2 * h - 1][r[:, None] - r[None, :] + h - 1]
    tw = t[2 * h - 1:][c[:, None] - c[None, :] + w - 1]
    q5 = q.double().reshape(q.shape[0], h, w, q.shape[2])
    bh = torch.einsum("nijd,ikd->nijk", q5, th)
    bw = torch.einsum("nijd,jkd->nijk", q5, tw)
    n = q.shape[0]
    return (bh[..., :, None] + bw[..., None, :]).reshape(n, h * w, h * w)


def _relpos64(q, k, v, table, h, w, scale):
    return _attend(q, k, v, scale, lambda i, j: _rel_bias(q[i:j], table, h, w))


def _rotate(x, cos, sin):
    """(x0 c - x1 s, x1 c + x0 s) over the pairs of the last dimension."""
    x = x.double()
    c, s = cos.double(), sin.double()
    turned = torch.stack([-x[..., 1::2], x[..., 0::2]], -1).reshape(x.shape)
    return x * c + turned * s


def _deform64(case, t):
    levels = _levels(case)
    value = t["value"].double()[0]
    s, h, d = value.shape
    outs, n = [], t["logits"].shape[1]
    sizes = torch.tensor([[w_, h_] for h_, w_ in levels], device=DEV, dtype=torch.float64)
    starts = [sum(a * b for a, b in levels[:i]) for i in range(4)]
    head = torch.arange(h, device=DEV)[None, :, None]
    for i in range(0, n, 4096):
        j = min(n, i + 4096)
        attn = torch.softmax(t["logits"][0, i:j].double().reshape(j - i, h, 16), 2).reshape(j - i, h, 4, 4)
        off, refs = t["offsets"][0, i:j].double(), t["refs"][0, i:j].double()
        xy = refs[:, None, :, None, :2]
        loc = xy + off / sizes[:, None, :] if refs.shape[2] == 2 else xy + off / 4 * refs[:, None, :, None, 2:] * 0.5
        acc = torch.zeros(j - i, h, d, device=DEV, dtype=torch.float64)
        for level, (lh, lw) in enumerate(levels):
            x, y = loc[:, :, level, :, 0] * lw - 0.5, loc[:, :, level, :, 1] * lh - 0.5
            x0, y0 = torch.floor(x), torch.floor(y)
            for dy in (0, 1):
                for dx in (0, 1):
                    cx, cy = x0 + dx, y0 + dy
                    wt = (1 - (x - cx).abs()) * (1 - (y - cy).abs()) * attn[:, :, level]
                    inside = (cx >= 0) & (cx < lw) & (cy >= 0) & (cy < lh)
                    at = starts[level] + cy.clamp(0, lh - 1).long() * lw + cx.clamp(0, lw - 1).long()
                    acc += ((wt * inside)[..., None] * value[at, head]).sum(2)
        outs.append(acc.reshape(j - i, h * d))
    return torch.cat(outs)[None]


def _block64(case, t):
    heads, hd, ws = case["heads"], case["hd"], case["window"]
    p = {n: t[n].double() for n in t}
    # the state holds the norm as the framework's dtype has it, as the caller's previous block returned it
    x = p["x"]
    b, g, _, c = x.shape
    xn = F.layer_norm(t["x"], (c,), t["norm1_w"], t["norm1_b"], 1e-6).double()
    wsz = ws or g
    pad = (-g) % wsz
    m = (g + pad) // wsz
    xw = F.pad(xn, (0, 0, 0, pad, 0, pad)).reshape(b, m, wsz, m, wsz, c).permute(0, 1, 3, 2, 4, 5)
    n = wsz * wsz
    qkv = (xw.reshape(-1, c) @ p["qkv_w"].t().contiguous() + p["qkv_b"]).reshape(b * m * m, n, 3, heads, hd)
    q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3).reshape(-1, n, hd) for i in range(3))
    o = _relpos64(q, k, v, t["rel"], wsz, wsz, hd ** -0.5)
    o = o.reshape(b, m, m, heads, wsz, wsz, hd).permute(0, 1, 4, 2, 5, 3, 6).reshape(b, m * wsz, m * wsz, c)
    o = o[:, :g, :g].reshape(-1, c) @ p["proj_w"].t().contiguous()
    x = x + o.reshape(b, g, g, c) + p["proj_b"]
    y = F.layer_norm(x, (c,), p["norm2_w"], p["norm2_b"], 1e-6).reshape(-1, c)
    y = F.gelu(y @ p["lin1_w"].t().contiguous() + p["lin1_b"]) @ p["lin2_w"].t().contiguous()
    x = x + y.reshape(b, g, g, c) + p["lin2_b"]
    return x, F.layer_norm(x, (c,), p["next_w"], p["next_b"], 1e-6)


def exact(case, seed):
    """run()'s outputs in 64 bits, in plain torch, of the same inputs."""
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "relpos":
        return _relpos64(t["q"], t["kt"].transpose(1, 2), t["v"], t["table"], case["gh"], case["gw"],
                         case["hd"] ** -0.5)
    if kind == "memory":
        n = case["side"] ** 2
        rot = case["frames"] * n
        q = _rotate(t["q"], t["cos"], t["sin"])
        c, s = t["cos"].repeat(case["frames"], 1), t["sin"].repeat(case["frames"], 1)
        k = torch.cat([_rotate(t["k"][:, :rot], c, s), t["k"][:, rot:].double()], 1)
        return torch.cat([_attend(q[:, i : i + 1024], k, t["v"], 1 / 16) for i in range(0, n, 1024)], 1)
    if kind == "sam3":
        nw, n, h, d = case["nw"], case["side"] ** 2, case["h"], case["d"]
        y = (t["y"].double() + t["bias"].double()).reshape(nw, n, 3, h, d)
        cos, sin = t["cos"][:, None, :], t["sin"][:, None, :]
        q, k = _rotate(y[:, :, 0], cos, sin), _rotate(y[:, :, 1], cos, sin)
        q, k, v = (a.permute(0, 2, 1, 3).reshape(nw * h, n, d) for a in (q, k, y[:, :, 2]))
        return _attend(q, k, v, d ** -0.5).reshape(nw, h, n, d).permute(0, 2, 1, 3).contiguous()
    if kind == "flash":
        b, l, h, d = (case[k] for k in ("b", "l", "h", "d"))
        q, k, v = (t["qkv"][:, :, i].permute(0, 2, 1, 3).reshape(b * h, l, d) for i in range(3))
        return _attend(q, k, v, d ** -0.5).reshape(b, h, l, d).permute(0, 2, 1, 3).contiguous()
    if kind == "sdpa":
        b, h, lq, lk, d = (case[k] for k in ("b", "h", "lq", "lk", "d"))
        m = t["mask"].double().expand(b, h, lq, lk).reshape(b * h, lq, lk)
        q, k, v = (t[n].reshape(b * h, -1, d) for n in ("q", "k", "v"))
        return _attend(q, k, v, d ** -0.5, lambda i, j: m[i:j]).reshape(b, h, lq, d)
    if kind == "deform":
        return _deform64(case, t)
    return _block64(case, t)

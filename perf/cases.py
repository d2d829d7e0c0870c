"""The workloads whose time this framework is judged by, through its public entry points.

A case is a dict of plain values.  ``listed()`` names the ones that are
tracked, ``draw()`` makes further ones of the same ranges, ``prepare()`` builds
what a program holds before the call (weights bound to a native block or
model, prepared text, KV pools, inputs), ``run()`` is one call, ``exact()`` the
same result in float64 by plain torch.

Kinds of case:
  block      one DiT block (WholeLayerBlock, or TransformerBlock.forward when
             the text is not prepared): the unit every forward repeats
  model      the whole transformer over its layers, action or video path
  attention  ops.attention, self attention over a cached prefix
  ffn        norm3, FFN1 + GELU and FFN2 + gated residual (ops)
  norms      the row passes of a block on their own (ops)
  prompt     text embedder and one layer's cross K/V for a new prompt
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "wam-egale_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from wam_ops import TransformerBlock, TransformerModel, WholeLayerBlock, WholeModel, ops  # noqa: E402

DEV = "cuda"
EPS = 1e-6
HD = 128
TEXT_DIM = 4096
# FFN width of a block by its width: the Wan2.2-5B and the Wan-1.3B block.
FFN = {3072: 14336, 1536: 8960}


def _block(name, B, grid, prefix=0, mode="none", rows=1, gap=0, ctx=512, dim=3072, prepared=True, ffn=0,
           temb="sample", **more):
    f, h, w = grid
    return dict(kind="block", name=name, dim=dim, B=B, f=f, h=h, w=w, prefix=prefix, mode=mode, rows=rows, gap=gap,
                ctx=ctx, prepared=prepared, ffn=ffn, temb=temb, **more)


def listed():
    return [
        # The draft step of action prediction: 16 action tokens, the
        # conditional and unconditional branch, over a short cached episode.
        # The smallest call; a policy makes it at every denoising step.
        _block("action_b2", 2, (2, 8, 1), prefix=288, mode="temp", temb="frame", action=True),
        # Verification of seven action candidates with CFG (14 x 16 tokens),
        # each over its branch's cached episode, read only.
        _block("action_verify_b14", 14, (2, 8, 1), prefix=1152, mode="candidates", rows=2, temb="frame",
               action=True),
        # One predicted video latent (128 tokens) with CFG over a long episode
        # whose oldest chunk was evicted; its K/V enter the pool and are
        # cleared again as predictions.
        _block("video_q128_pred", 2, (1, 8, 16), prefix=2160, mode="pred", gap=128, temb="frame"),
        # The 1.3B-shaped block on 1024 tokens, its text not prepared: every
        # call projects the context.
        _block("wan13b_1024", 1, (4, 16, 16), dim=1536, prepared=False),
        # A dense forward over six latent frames of 26 x 30 tokens.
        _block("video_4680", 1, (6, 26, 30)),
        # Speculative verification of four video chunks over one shared
        # cached prefix.
        _block("video_verify_4x1560", 4, (2, 26, 30), prefix=6240, mode="candidates", rows=1),
        # Three frames of an odd size with both FFN GEMMs on e4m3 (MX hidden
        # layer), per-token timesteps as the reference passes them.
        _block("video_2325_fp8", 1, (3, 25, 31), ffn=3, temb="token"),
        # One 1560-token chunk over four cached ones.
        dict(kind="attention", name="attention_1560_over_6240", B=1, heads=24, Mq=1560, Mk=1560, prefix=6240, gap=0),
        # The FFN of one latent frame.
        dict(kind="ffn", name="ffn_780", dim=3072, B=1, tokens=780, fp8=False),
        # The row passes of a block at 4680 rows (HBM-bound).
        dict(kind="norms", name="norms_4680", dim=3072, B=1, f=6, h=26, w=30),
        # A new prompt: text embedder and a layer's cross K/V, conditional
        # and unconditional.
        dict(kind="prompt", name="prompt_2x512", dim=3072, B=2, ctx=512),
        # The whole 30-layer model on seven action candidates with CFG:
        # what one verification costs a policy.
        dict(kind="model", name="model_action_verify_b14", layers=30, B=14, f=2, h=8, w=1, prefix=720, rows=2,
             action=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block"] * 6 + ["attention", "ffn", "norms", "prompt", "model"])
    dim = rng.choice([3072, 3072, 3072, 1536])
    if kind == "block":
        if rng.random() < 0.5:  # action tokens: few per sample, several samples
            B, f, h, w, action = rng.choice([1, 2, 4, 7, 14]), rng.choice([1, 2, 4]), rng.randint(3, 16), 1, True
        else:  # video latents, up to the verify batch's 6240 rows
            tokens = _log(rng, 60, 5000)
            f = rng.randint(1, 6)
            h = max(2, int(round(math.sqrt(tokens / f) * rng.uniform(0.8, 1.1))))
            w = max(2, tokens // (f * h))
            B, action = (rng.choice([1, 2, 4]) if f * h * w <= 1500 else 1), False
        M = f * h * w
        mode = rng.choice(["none", "temp", "pred", "candidates"])
        prefix = 0 if mode == "none" else _log(rng, 100, 6000)
        return dict(kind="block", dim=dim, B=B, f=f, h=h, w=w, prefix=prefix, mode=mode,
                    rows=rng.choice([1, 2]) if mode == "candidates" else 1,
                    gap=rng.choice([0, rng.randint(1, 200)]) if prefix else 0, ctx=rng.choice([512, rng.randint(40, 512)]),
                    prepared=rng.random() < 0.8, ffn=rng.choice([0, 0, 0, 1, 2, 3]),
                    temb=rng.choice(["sample", "frame", "token"]) if M < 3000 else "frame", action=action)
    if kind == "attention":
        Mq = _log(rng, 16, 2400)
        return dict(kind=kind, B=rng.choice([1, 2, 4]) if Mq < 1200 else 1, heads=dim // HD, Mq=Mq,
                    Mk=rng.choice([Mq, _log(rng, 16, 2400)]), prefix=_log(rng, 100, 6000),
                    gap=rng.choice([0, rng.randint(1, 200)]))
    if kind == "ffn":
        return dict(kind=kind, dim=dim, B=rng.choice([1, 2]), tokens=_log(rng, 16, 2600), fp8=rng.random() < 0.3)
    if kind == "norms":
        return dict(kind=kind, dim=dim, B=rng.choice([1, 2]), f=rng.randint(1, 6), h=rng.randint(4, 26),
                    w=rng.randint(4, 30))
    if kind == "prompt":
        return dict(kind=kind, dim=dim, B=rng.choice([1, 2]), ctx=rng.randint(40, 512))
    action = rng.random() < 0.7
    if action:
        B, f, h, w = rng.choice([1, 2, 7, 14]), rng.choice([1, 2]), rng.randint(4, 16), 1
    else:
        B, f, h, w = rng.choice([1, 2]), rng.choice([1, 2]), rng.randint(4, 20), rng.randint(4, 20)
    return dict(kind=kind, layers=rng.randint(2, 6), B=B, f=f, h=h, w=w, prefix=_log(rng, 100, 3000),
                rows=rng.choice([1, 2]), action=action)


# ------------------------------------------------------------------ inputs
class _Source:
    """Seeded tensors, each from the next values of one generator."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        t = torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float32).mul_(std).add_(mean)
        return t.to(dtype)

    def weights(self, shapes):
        """state_dict values by name: projections and biases N(0, 0.02), norm
        weights N(1, 0.02), the modulation tables N(0, 1) / sqrt(D) in fp32."""
        out = {}
        for name, shape in shapes.items():
            if name.endswith("scale_shift_table"):
                out[name] = self.normal(shape, 1.0 / math.sqrt(shape[-1]), dtype=torch.float32)
            elif "norm" in name:
                mean = 1.0 if name.endswith("weight") else 0.0
                out[name] = self.normal(shape, 0.02, mean, torch.float32 if "norm2" in name else torch.bfloat16)
            else:
                out[name] = self.normal(shape, 0.02, dtype=torch.float32 if "time_embedder" in name else torch.bfloat16)
        return out


def _shapes(module):
    return {n: tuple(p.shape) for n, p in module.named_parameters()}


def _grid_ids(f, h, w, action):
    """[4, f*h*w] (frame, row, column, 0): video latents in raster order;
    action tokens at fractions of their frame with row and column -1."""
    ff, hh, ww = torch.meshgrid(torch.arange(f), torch.arange(h), torch.arange(w), indexing="ij")
    ff, hh, ww = ff.float(), hh.float(), ww.float()
    if action:
        ff = ff + (hh + 1) / (h + 1)
        hh, ww = torch.full_like(hh, -1), torch.full_like(ww, -1)
    g = torch.stack([ff.flatten(), hh.flatten(), ww.flatten()])
    return torch.cat([g, torch.zeros_like(g[:1])]).to(DEV)


def _rope(grid):
    """complex64 [B, L, 1, 64] of grid ids [B, >=3, L] (44 / 42 / 42 split)."""
    ang = []
    for i, d in enumerate((44, 42, 42)):
        base = 10000.0 ** (-torch.arange(0, d, 2, device=DEV).double() / d)
        ang.append(grid[:, i, :, None].double() * base)
    ang = torch.cat(ang, -1).float()
    return torch.polar(torch.ones_like(ang), ang)[:, :, None]


def _pool(src, batch, slots, heads, prefix, gap):
    """A KV pool holding `prefix` committed rows in its first slots; a gap in
    their middle is what an evicted chunk leaves."""
    mask = torch.zeros(slots, dtype=torch.bool, device=DEV)
    head = prefix // 2 if gap else prefix
    mask[:head] = True
    mask[head + gap:prefix + gap] = True
    ids = torch.where(mask, torch.arange(slots, device=DEV) // 128, -1)
    return {"k": src.normal((batch, slots, heads, HD)), "v": src.normal((batch, slots, heads, HD)), "id": ids,
            "mask": mask, "is_pred": torch.zeros(slots, dtype=torch.bool, device=DEV)}


def _rows(B, rows):
    return (torch.arange(B, device=DEV) * rows) // B


def _temb_rows(kind, c):
    return {"sample": 1, "frame": c["f"], "token": c["f"] * c["h"] * c["w"]}[kind]


def _block_inputs(c, seed):
    src = _Source(seed)
    B, M, D = c["B"], c["f"] * c["h"] * c["w"], c["dim"]
    with torch.device("meta"):
        blk = TransformerBlock(D, FFN[D], D // HD, cross_attn_norm=True, eps=EPS)
    s = {"params": src.weights(_shapes(blk))}
    s["x"] = src.normal((B, M, D))
    s["ctx"] = src.normal((1, c["ctx"], D))
    s["temb"] = src.normal((B, _temb_rows(c["temb"], c), 6, D), 0.1, dtype=torch.float32)
    s["freqs"] = _rope(_grid_ids(c["f"], c["h"], c["w"], c.get("action", False))[None])
    if c["mode"] != "none":
        batch = c["rows"] if c["mode"] == "candidates" else B
        s["cache"] = _pool(src, batch, c["prefix"] + max(c["gap"], M), D // HD, c["prefix"], c["gap"])
        s["cand"] = _rows(B, batch) if c["mode"] == "candidates" else None
    return blk, s


def _model_inputs(c, seed):
    src = _Source(seed)
    with torch.device("meta"):
        model = TransformerModel(num_layers=c["layers"])
    s = {"params": src.weights(_shapes(model))}
    B, f, h, w = c["B"], c["f"], c["h"], c["w"]
    lat = (B, 30, f, h, w) if c["action"] else (B, 48, f, 2 * h, 2 * w)
    s["input"] = {
        "noisy_latents": src.normal(lat),
        "text_emb": src.normal((1, 512, TEXT_DIM)),
        "grid_id": _grid_ids(f, h, w, c["action"])[None].repeat(B, 1, 1),
        "timesteps": torch.rand((B, f), generator=src.g, device=DEV) * 1000.0,
    }
    s["caches"] = [_pool(src, c["rows"], c["prefix"] + f * h * w, 24, c["prefix"], 0) for _ in range(c["layers"])]
    s["cand"] = _rows(B, c["rows"])
    return model, s


def _ffn_inputs(c, seed):
    src = _Source(seed)
    D, N = c["dim"], FFN[c["dim"]]
    return {"x": src.normal((c["B"], c["tokens"], D), dtype=torch.float32),
            "w1": src.normal((N, D), 0.02), "b1": src.normal((N,), 0.02),
            "w2": src.normal((D, N), 0.02), "b2": src.normal((D,), 0.02),
            "table": src.normal((1, 6, D), 1 / math.sqrt(D), dtype=torch.float32),
            "temb": src.normal((c["B"], 1, 6, D), 0.1, dtype=torch.float32)}


def _norm_inputs(c, seed):
    src = _Source(seed)
    D, B, M = c["dim"], c["B"], c["f"] * c["h"] * c["w"]
    return {"x": src.normal((B, M, D)), "res": src.normal((B, M, D), 1.2, dtype=torch.float32),
            "q": src.normal((B, M, D)), "k": src.normal((B, M, D)),
            "gq": src.normal((D,), 0.02, 1.0), "gk": src.normal((D,), 0.02, 1.0),
            "g2": src.normal((D,), 0.02, 1.0, torch.float32), "b2": src.normal((D,), 0.02, dtype=torch.float32),
            "table": src.normal((1, 6, D), 1 / math.sqrt(D), dtype=torch.float32),
            "temb": src.normal((B, c["f"], 6, D), 0.1, dtype=torch.float32),
            "freqs": _rope(_grid_ids(c["f"], c["h"], c["w"], False)[None])}


def _attention_inputs(c, seed):
    src = _Source(seed)
    s = {n: src.normal((c["B"], m, c["heads"], HD)) for n, m in (("q", c["Mq"]), ("k", c["Mk"]), ("v", c["Mk"]))}
    s["cache"] = _pool(src, c["B"], c["prefix"] + max(c["gap"], c["Mk"]), c["heads"], c["prefix"], c["gap"])
    return s


def _prompt_inputs(c, seed):
    src = _Source(seed)
    D = c["dim"]
    with torch.device("meta"):
        blk = TransformerBlock(D, FFN[D], D // HD, cross_attn_norm=True, eps=EPS)
    return blk, {"params": src.weights(_shapes(blk)), "text": src.normal((c["B"], c["ctx"], TEXT_DIM)),
                 "t1": src.normal((D, TEXT_DIM), 0.02), "tb1": src.normal((D,), 0.02),
                 "t2": src.normal((D, D), 0.02), "tb2": src.normal((D,), 0.02)}


# ------------------------------------------------------------- the program
def prepare(case, seed):
    c = case
    with torch.no_grad():
        if c["kind"] == "block":
            blk, s = _block_inputs(c, seed)
            blk.load_state_dict(s.pop("params"), assign=True)
            if c["mode"] != "none":
                blk.attn1.attn_caches["pos"] = s["cache"]
            call = blk
            if c["prepared"] or c["ffn"]:
                call = WholeLayerBlock(blk, ffn_fp8=c["ffn"] > 0, ffn_act_fp8=max(0, c["ffn"] - 1))
                if c["prepared"]:
                    call.prepare_context(s["ctx"], precompute=True)
                call.bound()
            s.update(block=blk, call=call)
        elif c["kind"] == "model":
            model, s = _model_inputs(c, seed)
            model.load_state_dict(s.pop("params"), assign=True)
            for b, cache in zip(model.blocks, s["caches"]):
                b.attn1.attn_caches["pos"] = cache
            s["call"] = WholeModel(model)
            s["call"].prepare_text(s["input"]["text_emb"])
        elif c["kind"] == "ffn":
            s = _ffn_inputs(c, seed)
            if c["fp8"]:
                s["w1"], s["s1"] = ops.quantize_fp8_rows(s["w1"])
                s["w2"], s["s2"] = ops.quantize_fp8_rows(s["w2"])
        elif c["kind"] == "norms":
            s = _norm_inputs(c, seed)
        elif c["kind"] == "attention":
            s = _attention_inputs(c, seed)
            P = s["cache"]["mask"].numel()
            s["slots"] = torch.zeros(P, dtype=torch.int32, device=DEV)
            valid = s["cache"]["mask"].nonzero().squeeze(-1).int()
            s["slots"][:valid.numel()] = valid
            s["n"] = torch.tensor([valid.numel()], dtype=torch.int32, device=DEV)
            s["base"] = torch.tensor([-1 if c["gap"] else 0], dtype=torch.int32, device=DEV)
        else:
            blk, s = _prompt_inputs(c, seed)
            blk.load_state_dict(s.pop("params"), assign=True)
            s["call"] = WholeLayerBlock(blk)
            s["call"].bound()
    s["case"] = c
    return s


def run(state):
    s, c = state, state["case"]
    with torch.no_grad():
        if c["kind"] == "block":
            if c["mode"] == "none":
                return s["call"](s["x"], s["ctx"], s["temb"], s["freqs"])
            if c["mode"] == "candidates":
                return s["call"](s["x"], s["ctx"], s["temb"], s["freqs"], update_cache=0,
                                 candidate_cache_rows=s["cand"])
            if c["mode"] == "temp":
                return s["call"](s["x"], s["ctx"], s["temb"], s["freqs"], update_cache=0)
            # a prediction: its K/V are committed, then its slots are freed
            out = s["call"](s["x"], s["ctx"], s["temb"], s["freqs"], update_cache=1)
            s["block"].attn1.clear_pred_cache("pos")
            cache = s["cache"]
            return {"out": out, "k": cache["k"], "v": cache["v"], "mask": cache["mask"]}
        if c["kind"] == "model":
            return s["call"](s["input"], update_cache=0, action_mode=c["action"], candidate_cache_rows=s["cand"])
        if c["kind"] == "attention":
            return ops.attention(s["q"], s["k"], s["v"], pool_k=s["cache"]["k"], pool_v=s["cache"]["v"],
                                 slots=s["slots"], n_hist=s["n"], hist_base=s["base"])
        if c["kind"] == "ffn":
            h = ops.ln_modulate(s["x"], s["table"], s["temb"], 3, EPS)
            u = ops.linear(h, s["w1"], s["b1"], epilogue=ops.EPI_BIAS_GELU, w_scale=s.get("s1"))
            return ops.linear(u, s["w2"], s["b2"], epilogue=ops.EPI_BIAS_GATE_RES, residual=s["x"], table=s["table"],
                              temb=s["temb"], tokens=c["tokens"], gate_index=5, w_scale=s.get("s2"))
        if c["kind"] == "norms":
            h1 = ops.ln_modulate(s["x"], s["table"], s["temb"], 0, EPS)
            q, k = ops.rms_rope([s["q"], s["k"]], [s["gq"], s["gk"]], EPS, s["freqs"])
            h2 = ops.layer_norm_affine(s["res"], s["g2"], s["b2"], EPS)
            h3 = ops.ln_modulate(s["res"], s["table"], s["temb"], 3, EPS)
            return {"h1": h1, "q": q, "k": k, "h2": h2, "h3": h3}
        h = ops.linear(s["text"], s["t1"], s["tb1"], epilogue=ops.EPI_BIAS_GELU)
        ctx = ops.linear(h, s["t2"], s["tb2"])
        s["call"].prepare_context(ctx, precompute=True)
        k, v = s["call"].context_kv
        return {"ctx": ctx, "k": k, "v": v}


# -------------------------------------------------------------------- work
def _block_work(c, hist, ctx_proj, out_bytes=2):
    """One block: its weights and pool rows read once, input and output; two
    flops per multiply-add."""
    D = c["dim"]
    N, M = FFN[D], c["f"] * c["h"] * c["w"]
    R = c["B"] * M
    ffn_bytes = 1 if c.get("ffn", 0) else 2
    flops = 2 * R * D * 6 * D + 4 * R * D * N + 4 * R * (hist + M) * D + 4 * R * c["ctx"] * D
    byts = 6 * D * D * 2 + 2 * D * N * ffn_bytes + R * D * (2 + out_bytes)
    pools = c.get("rows", 1) if c.get("mode") == "candidates" else c["B"]
    byts += pools * hist * D * 4
    if ctx_proj:
        flops += 2 * c["ctx"] * D * 2 * D
        byts += 2 * D * D * 2 + c["ctx"] * D * 2
    else:
        byts += c["ctx"] * D * 4
    if c.get("mode") == "pred":
        byts += R * D * 4
    return byts, flops


def work(case):
    c = case
    if c["kind"] == "block":
        b, f = _block_work(c, c["prefix"], not c["prepared"])
    elif c["kind"] == "model":
        D, R = 3072, c["B"] * c["f"] * c["h"] * c["w"]
        k = 30 if c["action"] else 192
        n = 30 if c["action"] else 192
        b, f = _block_work(dict(c, dim=D, ctx=512, mode="candidates"), c["prefix"], False, 0)
        b, f = (b - R * D * 2) * c["layers"], f * c["layers"]
        b += 2 * (k + n) * D + 2 * R * (k + n) + D * 256 * 4 + D * D * 4 + D * 6 * D * 2
        f += 2 * R * D * (k + n) + 2 * c["B"] * c["f"] * (D * 256 + 7 * D * D)
    elif c["kind"] == "attention":
        D, keys = c["heads"] * HD, c["prefix"] + c["Mk"]
        b, f = c["B"] * D * 2 * (2 * c["Mq"] + 2 * keys), 4 * c["B"] * c["Mq"] * keys * D
    elif c["kind"] == "ffn":
        D, R = c["dim"], c["B"] * c["tokens"]
        N = FFN[D]
        b, f = 2 * D * N * (1 if c["fp8"] else 2) + R * D * 6, 4 * R * D * N
    elif c["kind"] == "norms":
        D, R = c["dim"], c["B"] * c["f"] * c["h"] * c["w"]
        b, f = R * D * (2 + 4 + 4 + 10), R * D * 40
    else:
        D, R = c["dim"], c["B"] * c["ctx"]
        b = 2 * (D * TEXT_DIM + 3 * D * D) + 2 * R * (TEXT_DIM + 3 * D)
        f = 2 * R * (D * TEXT_DIM + 3 * D * D)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Four times what float64 says the path is off by (a bf16 result is off
    by 1.7e-3 from its rounding alone)."""
    c = case
    if c["kind"] == "model":
        return {"rel": 0.03, "max": 0.3}
    if c["kind"] == "block" and c["ffn"] >= 2:
        return {"rel": 0.02, "max": 0.2}
    if c["kind"] == "prompt":  # three roundings, one after the other
        return {"rel": 1.3e-2, "max": 0.13}
    return {"rel": 9e-3, "max": 0.09}


# ------------------------------------------------------------------- exact
def _ln(x):
    return F.layer_norm(x, (x.shape[-1],), eps=EPS)


def _rms(x, g):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * g.double()


def _rotate(x, freqs):
    """[B, M, D] with the (2j, 2j+1) pairs of every head rotated."""
    B, M, D = x.shape
    z = torch.view_as_complex(x.reshape(B, M, D // HD, HD // 2, 2)) * freqs.to(torch.complex128)
    return torch.view_as_real(z).reshape(B, M, D)


def _sdpa(q, k, v, chunk=2048):
    """[B, Mq, D] over [B, Mk, D], by batch row, head and query chunk."""
    out = torch.empty_like(q)
    for b in range(q.shape[0]):
        for h in range(0, q.shape[2], HD):
            kt, vh = k[b, :, h:h + HD].t().contiguous(), v[b, :, h:h + HD].contiguous()
            for i in range(0, q.shape[1], chunk):
                p = torch.softmax(q[b, i:i + chunk, h:h + HD] @ kt / math.sqrt(HD), -1)
                out[b, i:i + chunk, h:h + HD] = p @ vh
    return out


def _lin(x, p, name):
    return F.linear(x, p[name + ".weight"].double(), p[name + ".bias"].double())


def _exact_block(p, x, ctx, temb, freqs, pool_k=None, pool_v=None):
    """One block in float64; pool_k / pool_v [B, n, D] are the history rows."""
    B, M, _ = x.shape
    mod = p["scale_shift_table"].double()[None] + temb.double()
    mod = mod.repeat_interleave(M // mod.shape[1], dim=1)
    sh, sc, gate, csh, csc, cgate = mod.unbind(2)
    h = _ln(x) * (1 + sc) + sh
    q = _rotate(_rms(_lin(h, p, "attn1.to_q"), p["attn1.norm_q.weight"]), freqs)
    k = _rotate(_rms(_lin(h, p, "attn1.to_k"), p["attn1.norm_k.weight"]), freqs)
    v = _lin(h, p, "attn1.to_v")
    kk, vv = (k, v) if pool_k is None else (torch.cat([pool_k, k], 1), torch.cat([pool_v, v], 1))
    x = x + _lin(_sdpa(q, kk, vv), p, "attn1.to_out.0") * gate
    n2 = _ln(x) * p["norm2.weight"].double() + p["norm2.bias"].double()
    q = _rms(_lin(n2, p, "attn2.to_q"), p["attn2.norm_q.weight"])
    ck = _rms(_lin(ctx, p, "attn2.to_k"), p["attn2.norm_k.weight"]).expand(B, -1, -1)
    cv = _lin(ctx, p, "attn2.to_v").expand(B, -1, -1)
    x = x + _lin(_sdpa(q, ck, cv), p, "attn2.to_out.0")
    u = F.gelu(_lin(_ln(x) * (1 + csc) + csh, p, "ffn.net.0.proj"), approximate="tanh")
    return x + _lin(u, p, "ffn.net.2") * cgate, k, v


def _history(cache, rows):
    """[B, n, D] float64 K and V of the valid slots, pool row rows[b] for b."""
    return [cache[n][:, cache["mask"]].flatten(2).double()[rows] for n in ("k", "v")]


def _exact_model(c, s):
    p, inp = s["params"], s["input"]
    B, f, h, w = c["B"], c["f"], c["h"], c["w"]
    lat, M = inp["noisy_latents"].double(), f * h * w
    if c["action"]:
        x = _lin(lat.permute(0, 2, 3, 4, 1).reshape(B, M, 30), p, "action_embedder")
    else:
        x = lat.reshape(B, 48, f, h, 2, w, 2).permute(0, 2, 3, 5, 1, 4, 6).reshape(B, M, 192)
        x = _lin(x, p, "patch_embedding_mlp")
    text = "condition_embedder.text_embedder."
    ctx = _lin(F.gelu(_lin(inp["text_emb"].double(), p, text + "linear_1"), approximate="tanh"), p, text + "linear_2")
    cond = "condition_embedder_action." if c["action"] else "condition_embedder."
    ang = inp["timesteps"].double()[..., None] * torch.exp(-math.log(10000.0) * torch.arange(128, device=DEV) / 128).double()
    e = torch.cat([ang.cos(), ang.sin()], -1)
    temb = _lin(F.silu(_lin(e, p, cond + "time_embedder.linear_1")), p, cond + "time_embedder.linear_2")
    proj = _lin(F.silu(temb), p, cond + "time_proj").unflatten(2, (6, -1))
    freqs = _rope(inp["grid_id"])
    for i in range(c["layers"]):
        pre = f"blocks.{i}."
        pk, pv = _history(s["caches"][i], s["cand"])
        x = _exact_block({n[len(pre):]: t for n, t in p.items() if n.startswith(pre)}, x, ctx, proj, freqs, pk, pv)[0]
    mod = p["scale_shift_table"].double()[None] + temb[:, :, None]
    mod = mod.repeat_interleave(M // f, dim=1)
    x = _ln(x) * (1 + mod[:, :, 1]) + mod[:, :, 0]
    if c["action"]:
        return _lin(x, p, "action_proj_out")
    return _lin(x, p, "proj_out").reshape(B, M * 4, 48)


def exact(case, seed):
    c = case
    with torch.no_grad():
        if c["kind"] == "block":
            s = _block_inputs(c, seed)[1]
            hist = [None, None]
            if c["mode"] != "none":
                hist = _history(s["cache"], s["cand"] if s["cand"] is not None else torch.arange(c["B"], device=DEV))
            out, k, v = _exact_block(s["params"], s["x"].double(), s["ctx"].double(), s["temb"], s["freqs"], *hist)
            if c["mode"] != "pred":
                return out
            free = (~s["cache"]["mask"]).nonzero().squeeze(-1)[:k.shape[1]]
            pk, pv = s["cache"]["k"].double(), s["cache"]["v"].double()
            pk[:, free], pv[:, free] = k.unflatten(2, (-1, HD)), v.unflatten(2, (-1, HD))
            return {"out": out, "k": pk, "v": pv, "mask": None}
        if c["kind"] == "model":
            return _exact_model(c, _model_inputs(c, seed)[1])
        if c["kind"] == "attention":
            s = _attention_inputs(c, seed)
            pk, pv = _history(s["cache"], torch.arange(c["B"], device=DEV))
            k, v = (torch.cat([a, s[n].flatten(2).double()], 1) for a, n in ((pk, "k"), (pv, "v")))
            return _sdpa(s["q"].flatten(2).double(), k, v).unflatten(2, (-1, HD))
        if c["kind"] == "ffn":
            s = _ffn_inputs(c, seed)
            x, mod = s["x"].double(), s["table"].double()[None] + s["temb"].double()
            w1, w2 = s["w1"], s["w2"]
            if c["fp8"]:
                w1, w2 = (q.double() * sc.double()[:, None] for q, sc in map(_e4m3_rows, (w1, w2)))
            u = F.gelu(F.linear(_ln(x) * (1 + mod[:, :, 4]) + mod[:, :, 3], w1.double(), s["b1"].double()),
                       approximate="tanh")
            return x + F.linear(u, w2.double(), s["b2"].double()) * mod[:, :, 5]
        if c["kind"] == "norms":
            s = _norm_inputs(c, seed)
            mod = s["table"].double()[None] + s["temb"].double()
            mod = mod.repeat_interleave(s["x"].shape[1] // c["f"], dim=1)
            res = s["res"].double()
            return {"h1": _ln(s["x"].double()) * (1 + mod[:, :, 1]) + mod[:, :, 0],
                    "q": _rotate(_rms(s["q"].double(), s["gq"]), s["freqs"]),
                    "k": _rotate(_rms(s["k"].double(), s["gk"]), s["freqs"]),
                    "h2": _ln(res) * s["g2"].double() + s["b2"].double(),
                    "h3": _ln(res) * (1 + mod[:, :, 4]) + mod[:, :, 3]}
        s = _prompt_inputs(c, seed)[1]
        p = s["params"]
        ctx = F.gelu(F.linear(s["text"].double(), s["t1"].double(), s["tb1"].double()), approximate="tanh")
        ctx = F.linear(ctx, s["t2"].double(), s["tb2"].double())
        return {"ctx": ctx, "k": _rms(_lin(ctx, p, "attn2.to_k"), p["attn2.norm_k.weight"]),
                "v": _lin(ctx, p, "attn2.to_v")}


def _e4m3_rows(w):
    """Per-row e4m3 values and scales (max / 448) of a weight matrix."""
    amax = w.float().abs().amax(1)
    f = torch.full_like(amax, 448.0) / amax
    return (w.float() * f[:, None]).to(torch.float8_e4m3fn), amax / torch.full_like(amax, 448.0)

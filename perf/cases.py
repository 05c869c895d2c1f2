"""The measured workloads of the framework: what a program that serves a Palu-compressed model calls.

Each case is one call path through the public entry points of ``palu_tt`` at Llama-3.1-8B's attention shape
(32 query and 8 KV heads of 128, hidden 4096, FFN 14336, vocabulary 128256), the shape of the benchmark and
of the tests. Weights and inputs are random-init; the low-rank factors are scaled so that rebuilt keys and
values have the spread of an uncompressed layer's. ``exact`` restates every path in 64-bit torch.

Kinds:
  op       palu_sdpa_decode over tiled, row-major or paged latent caches: one decode step of one layer
  grouped  the same op over grouped latents (G-LRD), V rebuilt per head
  prefill  PaluAttention.forward(mode="prefill"): a layer's attention over whole prompts, caches written
  layer    PaluAttention.forward(mode="decode"): a layer's decode step, fused op or naive path
  mlp      the decode step's FFN: gate / up with the RMSNorm folded in, then the down projection
  model    Transformer.prefill or one decode_graph step of a two-layer decoder, logits out
"""
import math
import random
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "tt-cadlab_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

HD, NQ, NKV, DIM, FFN, VOCAB = 128, 32, 8, 4096, 14336, 128256
REP = NQ // NKV
THETA = 500000.0
LLAMA3 = {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
          "original_max_position_embeddings": 8192}
EPS = 1e-5
SCALE = HD ** -0.5
BF = torch.bfloat16
DEV = "cuda:0"


# ------------------------------------------------------------------------------------------------
# Cases

def listed():
    return [
        # one chat user's decode step: the smallest call, where launches and latency count
        dict(name="op_b1_ctx1024", kind="op", layout="tiled", batch=1, ctx=1024, rank_k=64, rank_v=64, lengths="full",
             table="f32", out="bf16"),
        # the benchmark's headline: a full serving batch at a long context
        dict(name="op_b32_ctx8192", kind="op", layout="tiled", batch=32, ctx=8192, rank_k=64, rank_v=64, lengths="full",
             table="f32", out="bf16"),
        # the reference's own row-major caches and bf16 table, ragged rows, a capacity that is no whole block
        dict(name="op_rows_b5_ragged", kind="op", layout="rows", batch=5, ctx=3001, rank_k=96, rank_v=128,
             lengths="mixed", table="bf16", out="f32"),
        # paged serving of mixed lengths (the benchmark's paged line)
        dict(name="op_paged_b8_mixed", kind="op", layout="paged", batch=8, ctx=32768, rank_k=128, rank_v=64,
             lengths="mixed", table="f32", out="bf16"),
        # grouped latents of unequal ranks in compact caches (the benchmark's grouped line)
        dict(name="grouped_b16_ctx16384", kind="grouped", layout="compact", batch=16, ctx=16384, ranks_k="128,512",
             ranks_v="192,384", lengths="full"),
        # the prompt of one user, a long one
        dict(name="prefill_s4096", kind="prefill", users=1, seq=4096, group=1, rank_k=64, rank_v=64, layout="tiled"),
        # two users' prompts of an odd length, grouped latents
        dict(name="prefill_grouped_u2_s777", kind="prefill", users=2, seq=777, group=4, rank_k=256, rank_v=384,
             layout="tiled"),
        # a layer's decode step at the decoder's serving batch
        dict(name="layer_b64_ctx2048", kind="layer", fused=True, batch=64, ctx=2048, rank_k=64, rank_v=80, layout="tiled"),
        # a layer's decode step on the path that PaluRuntime() selects by default, ragged rows
        dict(name="layer_naive_b4_ctx2000", kind="layer", fused=False, batch=4, ctx=2000, rank_k=64, rank_v=64,
             layout="tiled"),
        # the FFN of a decode step for a handful of users
        dict(name="mlp_b12", kind="mlp", rows=12),
        # a single user's decode step of a whole (two-layer) model, one graph replay, logits
        dict(name="model_decode_b1", kind="model", mode="decode", batch=1, ctx=700, rank_k=64, rank_v=64),
        # four users' prompts through a whole (two-layer) model, as the generation loop prefills
        dict(name="model_prefill_u4_s512", kind="model", mode="prefill", batch=4, ctx=512, rank_k=64, rank_v=96),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["op", "op", "op", "grouped", "prefill", "prefill", "layer", "layer", "mlp", "model_decode",
                       "model_prefill"])
    step16, step32 = [32, 48, 64, 80, 96, 112, 128], [32, 64, 96, 128]
    if kind == "op":
        layout = rng.choice(["tiled", "rows", "paged"])
        ranks = step32 if layout == "rows" else step16
        batch = _log(rng, 1, 64)
        ctx = _log(rng, 50, min(32768, 32 * 8192 // batch))
        return dict(kind="op", layout=layout, batch=batch, ctx=ctx, rank_k=rng.choice(ranks), rank_v=rng.choice(ranks),
                    lengths=rng.choice(["full", "mixed"]), table=rng.choice(["f32", "f32", "bf16"]),
                    out=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "grouped":
        batch = _log(rng, 1, 32)
        ctx = _log(rng, 100, min(32768, 16 * 16384 // batch))
        pick = lambda: str(rng.choice([128, 192, 256, 384, 512]))
        return dict(kind="grouped", layout=rng.choice(["compact", "tiled", "rows"]), batch=batch, ctx=ctx,
                    ranks_k=pick() + "," + pick(), ranks_v=pick() + "," + pick(),
                    lengths=rng.choice(["full", "mixed"]))
    if kind == "prefill":
        users = rng.choice([1, 1, 1, 2, 3, 4])
        seq = _log(rng, 17, 4096 // users)
        group = rng.choice([1, 1, 4])
        ranks = [128, 192, 256, 384, 512] if group > 1 else step16
        layout = "tiled" if group > 1 else rng.choice(["tiled", "tiled", "rows"])
        if layout == "rows":
            ranks = step32
        return dict(kind="prefill", users=users, seq=seq, group=group, rank_k=rng.choice(ranks),
                    rank_v=rng.choice(ranks), layout=layout)
    if kind == "layer":
        fused = rng.choice([True, True, False])
        batch = _log(rng, 1, 64 if fused else 8)
        ctx = _log(rng, 50, min(8192, (64 if fused else 8) * 2048 // batch))
        layout = rng.choice(["tiled", "tiled", "rows"])
        ranks = step32 if layout == "rows" else step16
        return dict(kind="layer", fused=fused, batch=batch, ctx=ctx, rank_k=rng.choice(ranks), rank_v=rng.choice(ranks),
                    layout=layout)
    if kind == "mlp":
        return dict(kind="mlp", rows=_log(rng, 1, 64))
    if kind == "model_decode":
        batch = _log(rng, 1, 64)
        return dict(kind="model", mode="decode", batch=batch, ctx=_log(rng, 50, 2048), rank_k=rng.choice(step16),
                    rank_v=rng.choice(step16))
    batch = rng.choice([1, 2, 3, 4])
    return dict(kind="model", mode="prefill", batch=batch, ctx=_log(rng, 17, 2048 // batch), rank_k=rng.choice(step16),
                rank_v=rng.choice(step16))


# ------------------------------------------------------------------------------------------------
# Inputs, made from the case and the seed alone (plain torch; shared by prepare and exact)

def _up(n, m):
    return -(-n // m) * m


def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 16 + salt)


def _randn(g, *shape, std=1.0, dtype=BF):
    return torch.randn(*shape, device=DEV, generator=g).mul_(std).to(dtype)


def _spectrum(r):
    """Standard deviations of a latent's components: the decaying spectrum that an SVD leaves, unit mean square."""
    s = torch.linspace(1.3, 0.6, r, device=DEV)
    return s / s.square().mean().sqrt()


def _latents(g, *shape):
    return (torch.randn(*shape, device=DEV, generator=g) * _spectrum(shape[-1])).to(BF)


def _lengths(case):
    """Row lengths (a property of the case, so that its work is the same for every seed)."""
    B, S = case["batch"], case["ctx"]
    if case.get("lengths", "full") == "full":
        return [S] * B
    r = random.Random(1000003 * B + S)
    return [S if b == 0 else r.randint(max(1, S // 32), S) for b in range(B)]


def _tables(n, dtype=torch.float32):
    """Meta-interleaved cos, sin [n, 128]: fp32 angles with Llama-3.1's frequency scaling."""
    f = 1.0 / (THETA ** (torch.arange(0, HD, 2).float() / HD))
    wave = 2 * math.pi / f
    factor, low, high, orig = (LLAMA3[k] for k in ("factor", "low_freq_factor", "high_freq_factor",
                                                   "original_max_position_embeddings"))
    slow = torch.where(wave > orig / low, f / factor, f)
    smooth = (orig / wave - low) / (high - low)
    mid = ~(wave < orig / high) & ~(wave > orig / low)
    f = torch.where(mid, (1 - smooth) * slow / factor + smooth * slow, slow).float()
    ang = torch.outer(torch.arange(n, dtype=torch.float32), f)
    return (torch.repeat_interleave(ang.to(dtype).cos(), 2, dim=1).to(DEV),
            torch.repeat_interleave(ang.to(dtype).sin(), 2, dim=1).to(DEV))


def _pair_swap(x):
    """(x0, x1) -> (-x1, x0) on the last dim's pairs."""
    p = x.unflatten(-1, (-1, 2))
    return torch.stack((-p[..., 1], p[..., 0]), dim=-1).flatten(-2)


def _rope(x, cos, sin):
    return x * cos + _pair_swap(x) * sin


def _ranks(case):
    return [[int(r) for r in case[k].split(",")] for k in ("ranks_k", "ranks_v")]


def _op_inputs(case, seed):
    """q, latents as rows [B, G, S, r], u_k, u_v, table, positions of an op or grouped case."""
    g = _gen(seed)
    B, S = case["batch"], case["ctx"]
    if case["kind"] == "grouped":
        (gk, gv), G = _ranks(case), 2
    else:
        G = NKV
        gk, gv = [case["rank_k"]] * G, [case["rank_v"]] * G
    rk, rv = max(gk), max(gv)
    cap = _up(S, 64) if case["layout"] == "paged" else S if case["layout"] == "rows" else _up(S, 32)
    k, v = _latents(g, B, G, cap, rk), _latents(g, B, G, cap, rv)
    u_k = _randn(g, NKV, rk, HD, std=rk ** -0.5)
    u_v = _randn(g, NKV, rv, HD, std=rv ** -0.5) if case["kind"] == "grouped" else None
    for i, (a, b) in enumerate(zip(gk, gv)):
        if case["kind"] == "grouped":
            heads = slice(i * NKV // G, (i + 1) * NKV // G)
            u_k[heads, a:] = 0
            u_v[heads, b:] = 0
            k[:, i, :, a:] = 0
            v[:, i, :, b:] = 0
    q = _randn(g, 1, B, NQ, HD, std=1.3)
    cos, sin = _tables(cap)
    cs = torch.cat([cos, sin], -1)
    cs = cs.to(BF) if case.get("table") == "bf16" else cs
    pos = torch.tensor(_lengths(case), dtype=torch.int32, device=DEV) - 1
    return dict(q=q, k=k, v=v, u_k=u_k, u_v=u_v, cs=cs.contiguous(), pos=pos, cap=cap)


def _pages(case, seed, rows):
    """rows [B, G, cap, r] -> a shuffled pool of 64-position pages and its table [B, cap / 64]."""
    B, G, cap, r = rows.shape
    n = cap // 64
    order = torch.randperm(B * n, generator=torch.Generator().manual_seed(int(seed))).to(DEV)
    pool = torch.empty(B * n, G, 64, r, dtype=rows.dtype, device=DEV)
    pool[order] = rows.reshape(B, G, n, 64, r).transpose(1, 2).reshape(B * n, G, 64, r)
    return pool, order.reshape(B, n).to(torch.int32)


def _attn_weights(g, rank_k, rank_v, group):
    """One attention layer's state-dict tensors in bf16: wq, wo and the converter's Palu tensors. At full
    per-head rank the K or V rows are the projection itself."""
    G = NKV // group
    w = {"wq": _randn(g, NQ * HD, DIM, std=0.02), "wo": _randn(g, DIM, NQ * HD, std=0.02)}
    for name, r in (("wk_lat_pad", rank_k), ("wv_lat_pad", rank_v)):
        pad = torch.zeros(G, group * HD, DIM, dtype=BF, device=DEV)
        pad[:, :r] = (torch.randn(G, r, DIM, device=DEV, generator=g) * 0.02 * _spectrum(r)[:, None]).to(BF)
        w[name] = pad.reshape(NKV * HD, DIM)
    w["u_k"] = _randn(g, NKV, rank_k, HD, std=rank_k ** -0.5)
    w["u_v"] = _randn(g, NKV, rank_v, HD, std=rank_v ** -0.5)
    if group == 1 and rank_v == HD:
        w["u_v"] = torch.eye(HD, device=DEV, dtype=BF).repeat(NKV, 1, 1)
    w["w_rot"] = torch.cat([w["u_k"], _pair_swap(w["u_k"])], -1)
    w["wo_fused"] = w["wo"].clone()
    if group == 1:
        fold = w["wo"].float().reshape(DIM, NKV, REP, HD).permute(1, 2, 0, 3).reshape(NKV, REP * DIM, HD)
        fold = torch.bmm(fold, w["u_v"].float().transpose(1, 2).contiguous())
        fold = fold.reshape(NKV, REP, DIM, rank_v).permute(2, 0, 1, 3).reshape(DIM, NQ, rank_v)
        fused = torch.zeros(DIM, NQ, HD, device=DEV)
        fused[:, :, :rank_v] = fold
        w["wo_fused"] = fused.reshape(DIM, NQ * HD).to(BF)
    return w


def _attn_sd(w, layer=0):
    p = f"layers.{layer}.attention"
    return {(f"{p}.{k}.weight" if k in ("wq", "wo") else f"{p}.palu.{k}"): t for k, t in w.items()}


def _cache_rows(case, seed, layer=0):
    """A decode case's filled caches as rows [B, G, cap, width] (the row at the step's position is rewritten)."""
    g = _gen(seed, 3 + 2 * layer)
    B, cap = case["batch"], _up(case["ctx"], 32)
    kw, rv = case["rank_k"], case["rank_v"]
    return _latents(g, B, NKV, cap, kw), _latents(g, B, NKV, cap, rv)


def _decode_pos(case):
    """Ragged positions of a decode step: every row in the last quarter of the context."""
    r = random.Random(7919 * case["batch"] + case["ctx"])
    S = case["ctx"]
    return torch.tensor([S - 1 if b == 0 else r.randint(3 * S // 4, S - 1) for b in range(case["batch"])],
                        dtype=torch.int32, device=DEV)


def _model_weights(case, seed):
    g = _gen(seed, 1)
    m = {"tok": _randn(g, VOCAB, DIM, std=1.0), "out": _randn(g, VOCAB, DIM, std=0.02),
         "norm": (1 + 0.1 * torch.randn(DIM, device=DEV, generator=g)).to(BF), "layers": []}
    for _ in range(2):
        m["layers"].append({
            "attn": _attn_weights(g, case["rank_k"], case["rank_v"], 1),
            "attention_norm": (1 + 0.1 * torch.randn(DIM, device=DEV, generator=g)).to(BF),
            "ffn_norm": (1 + 0.1 * torch.randn(DIM, device=DEV, generator=g)).to(BF),
            "w1": _randn(g, FFN, DIM, std=0.02), "w3": _randn(g, FFN, DIM, std=0.02), "w2": _randn(g, DIM, FFN, std=0.01)})
    return m


def _tokens(case, seed, *shape):
    return torch.randint(0, VOCAB, shape, generator=torch.Generator().manual_seed(int(seed) + 5)).to(DEV)


class _Args:
    """The configuration object that PaluAttention takes."""

    def __init__(self, max_seq, max_batch, palu):
        self.dim, self.n_heads, self.n_kv_heads, self.head_dim = DIM, NQ, NKV, HD
        self.max_seq_len, self.max_batch_size = max_seq, max_batch
        self.rope_theta, self.rope_scaling, self.palu = THETA, LLAMA3, palu


# ------------------------------------------------------------------------------------------------
# prepare / run

def prepare(case, seed):
    from palu_tt import convert, decoder_ops, model
    from palu_tt.attention import PaluAttention
    from palu_tt.cache import GroupedLatentCache, LatentCache
    kind = case["kind"]
    if kind in ("op", "grouped"):
        x = _op_inputs(case, seed)
        k, v, layout, s = x["k"], x["v"], case["layout"], {"kind": kind}
        s["ranks"] = s["pages"] = None
        if kind == "grouped":
            s["ranks"] = tuple(_ranks(case))
        if layout == "paged":
            k, s["pages"] = _pages(case, seed, k)
            v, _ = _pages(case, seed, v)
        if layout == "compact":
            k, v = GroupedLatentCache.from_rows(k, s["ranks"][0], "k"), GroupedLatentCache.from_rows(v, s["ranks"][1], "v")
        elif layout != "rows":
            k, v = LatentCache.from_rows(k, "k"), LatentCache.from_rows(v, "v")
        s.update(q=x["q"], k=k, v=v, cs=x["cs"][None, None], pos=x["pos"], u_v=None if x["u_v"] is None else x["u_v"][None],
                 w_rot=torch.cat([x["u_k"], _pair_swap(x["u_k"])], -1)[None].contiguous(),
                 width=HD if kind == "grouped" else case["rank_v"],
                 out=torch.float32 if case.get("out") == "f32" else BF)
        return s
    if kind == "mlp":
        g = _gen(seed)
        w = _mlp_weights(g)
        return {"kind": kind, "rows": case["rows"], "x": _randn(g, case["rows"], DIM),
                "w13": decoder_ops.DecodeLinear(None, case["rows"], gate_up=(w["w1"], w["w3"]), in_scale=w["norm"]),
                "w2": decoder_ops.DecodeLinear(w["w2"], case["rows"])}
    if kind in ("prefill", "layer"):
        prefill = kind == "prefill"
        group, B = (case["group"], case["users"]) if prefill else (1, case["batch"])
        cap = _up(case["seq"] if prefill else case["ctx"], 32)
        palu = convert.PaluConfig(rank_k=[case["rank_k"]], rank_v=[case["rank_v"]], cache_id="cases", group_size=group,
                                  runtime=convert.PaluRuntime(use_fused_k=prefill or case["fused"]))
        att = PaluAttention(DEV, None, _Args(cap, B, palu), _attn_sd(_attn_weights(_gen(seed), case["rank_k"], case["rank_v"], group)),
                            None, 0, cache_layout=case["layout"])
        if prefill:
            return {"kind": kind, "att": att, "x": _randn(_gen(seed, 2), B, case["seq"], DIM)}
        _fill(att, *_cache_rows(case, seed), LatentCache)
        return {"kind": kind, "att": att, "x": _randn(_gen(seed, 2), B, DIM), "pos": _decode_pos(case)}
    m = _model_weights(case, seed)
    sd = {"tok_embeddings.weight": m["tok"], "output.weight": m["out"], "norm.weight": m["norm"]}
    for i, L in enumerate(m["layers"]):
        sd.update(_attn_sd(L["attn"], i))
        sd[f"layers.{i}.attention_norm.weight"], sd[f"layers.{i}.ffn_norm.weight"] = L["attention_norm"], L["ffn_norm"]
        sd.update({f"layers.{i}.feed_forward.{k}.weight": L[k] for k in ("w1", "w2", "w3")})
    palu = convert.PaluConfig(rank_k=[case["rank_k"]] * 2, rank_v=[case["rank_v"]] * 2, cache_id="cases",
                              runtime=convert.PaluRuntime(use_fused_k=True))
    args = model.ModelArgs(n_layers=2, max_seq_len=_up(case["ctx"], 32), max_batch_size=case["batch"], palu=palu)
    del m
    net = model.Transformer(args, sd, DEV)
    s = {"kind": case["mode"], "net": net}
    if case["mode"] == "prefill":
        s["tokens"] = _tokens(case, seed, case["batch"], case["ctx"])
        return s
    for i, L in enumerate(net.layers):
        _fill(L["attn"], *_cache_rows(case, seed, i), LatentCache)
    s.update(tokens=_tokens(case, seed, case["batch"]), pos=_decode_pos(case))
    return s


def _fill(att, k, v, LatentCache):
    for i, rows in enumerate((k, v)):
        if isinstance(att.layer_past[i], LatentCache):
            att.layer_past[i] = LatentCache.from_rows(rows, "kv"[i])
        else:
            att.layer_past[i] = rows


def _stores(att):
    return [c if isinstance(c, torch.Tensor) else c.data for c in att.layer_past]


def run(state):
    kind = state["kind"]
    if kind in ("op", "grouped"):
        from palu_tt import fused
        return fused.palu_sdpa_decode(state["q"], state["k"], state["w_rot"], state["cs"], state["v"], state["width"],
                                      state["pos"], u_v=state["u_v"], scale=SCALE, out_dtype=state["out"],
                                      page_table_tensor=state["pages"], group_ranks=state["ranks"])
    if kind == "prefill" and "att" in state:
        return [state["att"].forward(state["x"], mode="prefill", user_id=0)] + _stores(state["att"])
    if kind == "layer":
        return [state["att"].forward(state["x"], state["pos"], mode="decode")] + _stores(state["att"])
    if kind == "mlp":
        a = state["w13"].swiglu_rmsnorm(state["x"], EPS)
        return state["w2"](a, x_tiled=True, rows=state["rows"])
    net = state["net"]
    if kind == "prefill":
        logits = net.prefill(state["tokens"])
    else:
        logits = net.decode_graph(state["tokens"], state["pos"])
    return [logits] + [c for L in net.layers for c in _stores(L["attn"])]


# ------------------------------------------------------------------------------------------------
# work / tolerance

def work(case):
    kind = case["kind"]
    if kind in ("op", "grouped"):
        if kind == "grouped":
            (gk, gv), G = _ranks(case), 2
        else:
            gk, gv, G = [case["rank_k"]] * NKV, [case["rank_v"]] * NKV, NKV
        L, B, per = sum(_lengths(case)), case["batch"], NKV // G
        width = HD if kind == "grouped" else case["rank_v"]
        nbytes = L * (sum(gk) + sum(gv)) * 2 + B * NQ * (HD * 2 + width * (4 if case.get("out") == "f32" else 2))
        nbytes += per * sum(gk) * HD * 2 + (per * sum(gv) * HD * 2 if kind == "grouped" else 0)
        flops = sum(2 * L * per * rk * HD + 2 * L * per * REP * (HD + rv) for rk, rv in zip(gk, gv))
        if kind == "grouped":
            flops += sum(2 * B * per * REP * rv * HD for rv in gv)
        return {"bytes": nbytes, "flops": flops}
    if kind == "mlp":
        r = case["rows"]
        return {"bytes": 3 * DIM * FFN * 2 + 2 * r * DIM * 2, "flops": 2 * r * 3 * DIM * FFN}
    if kind == "prefill":
        return _attn_work(case["users"], case["seq"], case["rank_k"], case["rank_v"], case["group"])
    if kind == "layer":
        return _layer_work(case)
    n = case["batch"] * (case["ctx"] if case["mode"] == "prefill" else 1)
    a = (_attn_work(case["batch"], case["ctx"], case["rank_k"], case["rank_v"], 1) if case["mode"] == "prefill"
         else _layer_work(case))
    return {"bytes": 2 * (a["bytes"] + 3 * DIM * FFN * 2) + VOCAB * DIM * 2 + case["batch"] * VOCAB * 4 + n * DIM * 2,
            "flops": 2 * (a["flops"] + 2 * n * 3 * DIM * FFN) + 2 * case["batch"] * VOCAB * DIM}


def _attn_work(users, S, rk, rv, group):
    G, n = NKV // group, users * S
    cols = NQ * HD + G * (rk + rv)
    pairs = users * S * (S + 1) // 2
    return {"bytes": (cols + NQ * HD) * DIM * 2 + 2 * n * DIM * 2 + n * G * (rk + rv) * 2 + NKV * (rk + rv) * HD * 2,
            "flops": 2 * n * DIM * (cols + NQ * HD) + 2 * n * NKV * rk * HD + 2 * n * NQ * min(rv, HD) * HD +
            2 * pairs * NQ * (HD + min(rv, HD))}


def _layer_work(case):
    B, rk, rv = case["batch"], case["rank_k"], case["rank_v"]
    L = int((_decode_pos_list(case)))
    cols = NQ * HD + NKV * (rk + rv)
    return {"bytes": (cols + NQ * rv) * DIM * 2 + L * NKV * (rk + rv) * 2 + 2 * B * DIM * 2,
            "flops": 2 * B * DIM * (cols + NQ * rv) + 2 * L * NKV * rk * HD + 2 * L * NQ * (HD + rv)}


def _decode_pos_list(case):
    r = random.Random(7919 * case["batch"] + case["ctx"])
    S = case["ctx"]
    return sum((S if b == 0 else r.randint(3 * S // 4, S - 1) + 1) for b in range(case["batch"]))


def tolerance(case):
    # About four times the distance measured between the path and the 64-bit result (op 0.0030, prefill 0.0047,
    # layer 0.0055 on the naive path, mlp 0.0033, model 0.0081; two runs of one path whose blocks are summed in
    # another order stand up to 0.0036 apart, and no element further than 0.022).
    return {"op": {"rel": 0.012, "max": 0.1}, "grouped": {"rel": 0.012, "max": 0.1}, "prefill": {"rel": 0.019, "max": 0.15},
            "layer": {"rel": 0.022, "max": 0.15}, "mlp": {"rel": 0.014, "max": 0.1},
            "model": {"rel": 0.03, "max": 0.25}}[case["kind"]]


# ------------------------------------------------------------------------------------------------
# exact: the same paths in 64-bit torch

def _tile_index(R, role):
    """Offset of (position p, column k), p < 32, k < R, inside a 32-position block of a tiled cache."""
    p, k = torch.arange(32, device=DEV)[:, None], torch.arange(R, device=DEV)[None, :]
    if role == "v":
        return ((k // 16) * 64 + 16 * (p // 8) + k % 16) * 8 + p % 8
    c, nn, full = (p // 4) % 2, 4 * (p // 8) + p % 4, R // 32
    whole = ((k // 32) * 64 + 16 * ((k // 8) % 4) + nn) * 8 + k % 8
    half = full * 512 + (16 * ((k % 16) // 4) + nn) * 4 + k % 4
    return c * 16 * R + torch.where(k // 32 < full, whole, half)


def _store(rows, layout, role):
    """Cache rows [B, G, cap, r] as the cache's storage tensor."""
    if layout == "rows":
        return rows
    B, G, cap, r = rows.shape
    out = torch.empty(B, G, cap // 32, 32 * r, dtype=rows.dtype, device=DEV)
    out[..., _tile_index(r, role).reshape(-1)] = rows.reshape(B, G, cap // 32, 32 * r)
    return out.reshape(B, G, cap // 32, r // 16, 64, 8)


def _attend(q, k, v, u_k, u_v, cos, sin, pos, group):
    """Decode attention of one layer, row by row: q [B, NQ, HD] rotated; latent rows k, v [B, G, S, r]."""
    outs = []
    for b in range(q.shape[0]):
        n = int(pos[b]) + 1
        kb, vb = k[b, :, :n].double(), v[b, :, :n].double()
        heads = []
        for h in range(NKV):
            K = kb[h // group] if u_k is None else _rope(kb[h // group] @ u_k[h].double(), cos[:n], sin[:n])
            p = torch.softmax(q[b, h * REP:(h + 1) * REP] @ K.T * SCALE, -1) @ vb[h // group]
            heads.append(p if u_v is None else p @ u_v[h].double())
        outs.append(torch.cat(heads))
    return torch.stack(outs)


def _exact_layer_decode(w, x, rows, pos, cos, sin, rk, rv, layout):
    """(layer output, K store, V store) of a decode step over x [B, DIM] in 64 bits."""
    k, v = (t.double() for t in rows)
    B, at = x.shape[0], torch.arange(x.shape[0], device=DEV)
    lat = lambda name, r: (x @ w[name].reshape(NKV, HD, DIM)[:, :r].reshape(-1, DIM).double().T).reshape(B, NKV, r)
    c, s = cos[pos.long()][:, None], sin[pos.long()][:, None]
    q = _rope((x @ w["wq"].double().T).reshape(B, NQ, HD), c, s)
    kn = lat("wk_lat_pad", rk)
    k[at, :, pos.long()] = _rope(kn, c, s) if rk == HD else kn
    v[at, :, pos.long()] = lat("wv_lat_pad", rv)
    o = _attend(q, k, v, None if rk == HD else w["u_k"], None, cos, sin, pos, 1)            # [B, NQ, rv]
    wo = (w["wo"] if rv == HD else w["wo_fused"]).reshape(DIM, NQ, HD)[:, :, :rv].reshape(DIM, -1).double()
    return o.reshape(B, -1) @ wo.T, _store(k, layout, "k"), _store(v, layout, "v")


def _exact_prefill(w, x, cap, group, rk, rv, layout):
    """(layer output, K store, V store) of a prefill of x [U, S, DIM] in 64 bits."""
    U, S, _ = x.shape
    G = NKV // group
    cos, sin = (t[:S].double() for t in _tables(S, torch.float64))
    full_k, full_v = group == 1 and rk == HD, group == 1 and rv == HD
    lat = lambda xu, name, r: (xu @ w[name].reshape(G, group * HD, DIM)[:, :r].reshape(-1, DIM).double().T
                               ).reshape(S, G, r).transpose(0, 1)
    ks, vs = (torch.zeros(U, G, cap, r, dtype=torch.float64, device=DEV) for r in (rk, rv))
    mask = torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1)
    outs = []
    for u in range(U):
        kl, vl = lat(x[u], "wk_lat_pad", rk), lat(x[u], "wv_lat_pad", rv)
        q = _rope((x[u] @ w["wq"].double().T).reshape(S, NQ, HD).transpose(0, 1), cos, sin)
        ks[u, :, :S], vs[u, :, :S] = (_rope(kl, cos, sin) if full_k else kl), vl
        heads = []
        for h in range(NQ):
            kv = h // REP
            K = _rope(kl[kv // group] if full_k else kl[kv // group] @ w["u_k"][kv].double(), cos, sin)
            V = vl[kv // group] if full_v else vl[kv // group] @ w["u_v"][kv].double()
            heads.append(torch.softmax((q[h] @ K.T * SCALE).masked_fill_(mask, float("-inf")), -1) @ V)
        outs.append(torch.stack(heads, 1).reshape(S, NQ * HD) @ w["wo"].double().T)
    return torch.stack(outs), _store(ks, layout, "k"), _store(vs, layout, "v")


def _mlp_weights(g):
    return {"w1": _randn(g, FFN, DIM, std=0.02), "w3": _randn(g, FFN, DIM, std=0.02), "w2": _randn(g, DIM, FFN, std=0.02),
            "norm": (1 + 0.1 * torch.randn(DIM, device=DEV, generator=g)).to(BF)}


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _exact_mlp(x, norm, w):
    y = _norm(x, norm)
    g = y @ w["w1"].double().T
    return (torch.nn.functional.silu(g) * (y @ w["w3"].double().T)) @ w["w2"].double().T


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind in ("op", "grouped"):
        x = _op_inputs(case, seed)
        cos, sin = x["cs"][:, :HD].double(), x["cs"][:, HD:].double()
        return _attend(x["q"][0].double(), x["k"], x["v"], x["u_k"], x["u_v"], cos, sin, x["pos"],
                       NKV // x["k"].shape[1])[None]
    if kind == "mlp":
        g = _gen(seed)
        w = _mlp_weights(g)
        return _exact_mlp(_randn(g, case["rows"], DIM).double(), w["norm"], w)
    if kind == "prefill":
        w = _attn_weights(_gen(seed), case["rank_k"], case["rank_v"], case["group"])
        x = _randn(_gen(seed, 2), case["users"], case["seq"], DIM).double()
        return list(_exact_prefill(w, x, _up(case["seq"], 32), case["group"], case["rank_k"], case["rank_v"], case["layout"]))
    pos = None if case.get("mode") == "prefill" else _decode_pos(case)
    cos, sin = (t.double() for t in _tables(_up(case["ctx"], 32), torch.float64))
    if kind == "layer":
        w = _attn_weights(_gen(seed), case["rank_k"], case["rank_v"], 1)
        x = _randn(_gen(seed, 2), case["batch"], DIM).double()
        return list(_exact_layer_decode(w, x, _cache_rows(case, seed), pos, cos, sin, case["rank_k"], case["rank_v"],
                                        case["layout"]))
    m = _model_weights(case, seed)
    shape = (case["batch"], case["ctx"]) if case["mode"] == "prefill" else (case["batch"],)
    h = m["tok"][_tokens(case, seed, *shape)].double()
    stores = []
    for i, L in enumerate(m["layers"]):
        y = _norm(h, L["attention_norm"])
        if case["mode"] == "prefill":
            o, ks, vs = _exact_prefill(L["attn"], y, _up(case["ctx"], 32), 1, case["rank_k"], case["rank_v"], "tiled")
        else:
            o, ks, vs = _exact_layer_decode(L["attn"], y, _cache_rows(case, seed, i), pos, cos, sin, case["rank_k"],
                                            case["rank_v"], "tiled")
        h = h + o
        h = h + _exact_mlp(h, L["ffn_norm"], L)
        stores += [ks, vs]
    last = h[:, -1] if case["mode"] == "prefill" else h
    return [_norm(last, m["norm"]) @ m["out"].double().T] + stores

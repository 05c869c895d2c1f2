"""The prefill attention and cache-fill kernels (palu_prefill_attention, palu_latent_fill).

The attention is compared with 64-bit torch on the same bf16 rows and fp32 tables. The kernel keeps fp32 sums, takes
score operands with 22 bits and rounds its result to bf16 once, so an output may be off by half a bf16 step at its value
plus the computation's own error, which for these sizes stays below 4e-6 of the largest value of its row (fp32 attention
through torch measures 2e-5 of the rms at worst over 2048 positions)."""
import numpy as np
import pytest
import torch

from palu_tt import convert, decoder_ops, fused
from palu_tt.attention import PaluAttention
from palu_tt.cache import GroupedLatentCache, LatentCache

pytestmark = pytest.mark.gpu

HD = 128


def _inputs(users, S, nh, nkv, G, rk, rv, seed, full_k=False, full_v=False):
    g = torch.Generator().manual_seed(seed)
    k0, v0 = nh * HD, nh * HD + G * rk
    cols = v0 + G * rv
    x = torch.randn(users * S, cols + 24, generator=g)[:, :cols + 24].to(torch.bfloat16).cuda()[:, :cols + 16]
    u_k = None if full_k else (torch.randn(nkv, rk, HD, generator=g) / rk ** 0.5).to(torch.bfloat16).cuda()
    u_v = None if full_v else (torch.randn(nkv, rv, HD, generator=g) / rv ** 0.5).to(torch.bfloat16).cuda()
    cos, sin = (t.cuda() for t in fused.cos_sin_tables(HD, S, 500000.0, None))
    return x, k0, v0, u_k, u_v, cos, sin


def _half_step(e):
    """Half the spacing of bf16 values (8 significant bits) at e."""
    return torch.ldexp(torch.ones_like(e), torch.frexp(e).exponent - 9)


def _exact(x, users, nh, nkv, G, k0, rk, u_k, v0, rv, u_v, cos, sin, scale):
    S = x.shape[0] // users
    xd = x.double().view(users, S, -1)
    c, s = cos[:S].double(), sin[:S].double()

    def rope(t):
        p = t.unflatten(-1, (-1, 2))
        return t * c + torch.stack((-p[..., 1], p[..., 0]), -1).flatten(-2) * s
    out = torch.empty(users, S, nh, HD, dtype=torch.float64, device=x.device)
    mask = torch.ones(S, S, dtype=torch.bool, device=x.device).triu(1)
    for u in range(users):
        for h in range(nh):
            kv = h // (nh // nkv)
            gi = kv // (nkv // G)
            kl, vl = xd[u, :, k0 + gi * rk:k0 + (gi + 1) * rk], xd[u, :, v0 + gi * rv:v0 + (gi + 1) * rv]
            K = rope(kl if u_k is None else kl @ u_k[kv].double())
            V = vl if u_v is None else vl @ u_v[kv].double()
            sc = (rope(xd[u, :, h * HD:(h + 1) * HD]) @ K.T * scale).masked_fill(mask, float("-inf"))
            out[u, :, h] = torch.softmax(sc, -1) @ V
    return out.view(users * S, nh * HD)


@pytest.mark.parametrize("users,S,nh,nkv,G,rk,rv,full_k,full_v", [
    (1, 1, 4, 4, 4, 64, 64, False, False), (2, 31, 8, 2, 2, 32, 16, False, False), (1, 33, 4, 1, 1, 48, 48, False, False),
    (1, 64, 6, 2, 2, 16, 80, False, False), (3, 65, 8, 8, 8, 112, 112, False, False), (1, 257, 32, 8, 8, 64, 96, False, False),
    (1, 300, 8, 2, 2, 128, 128, True, True), (2, 129, 8, 2, 2, 128, 32, True, False), (1, 200, 4, 2, 2, 80, 128, False, True),
    (1, 130, 4, 2, 2, 128, 128, False, False), (1, 96, 16, 1, 1, 64, 64, False, False),
    (2, 100, 8, 4, 2, 192, 256, False, False), (1, 515, 32, 8, 2, 512, 384, False, False), (1, 40, 8, 4, 1, 48, 176, False, False)])
def test_prefill_attention(gpu, users, S, nh, nkv, G, rk, rv, full_k, full_v):
    x, k0, v0, u_k, u_v, cos, sin = _inputs(users, S, nh, nkv, G, rk, rv, S + rk + rv, full_k, full_v)
    scale = HD ** -0.5
    out = decoder_ops.prefill_attention(x, users, nh, nkv, G, k0, rk, u_k, v0, rv, u_v, cos, sin, scale).double()
    exp = _exact(x, users, nh, nkv, G, k0, rk, u_k, v0, rv, u_v, cos, sin, scale)
    bound = _half_step(exp) * 1.001 + 4e-6 * exp.abs().amax(-1, keepdim=True)
    worst = ((out - exp).abs() / bound).max().item()
    assert worst <= 1.0, f"{worst:.3f} of the bound"


def test_prefill_attention_wide_range(gpu):
    """Scores in the hundreds (one key dominates, the running maximum is refreshed often), keys beyond the fp16 range,
    and probabilities that underflow: finite results at the same bound plus the score's own fp32 rounding."""
    x, k0, v0, u_k, u_v, cos, sin = _inputs(1, 160, 8, 2, 2, 64, 64, 5)
    x = x.clone()
    x[:, k0:v0] *= 3e5
    x[:, :k0] *= 1e-4
    out = decoder_ops.prefill_attention(x, 1, 8, 2, 2, k0, 64, u_k, v0, 64, u_v, cos, sin, HD ** -0.5).double()
    exp = _exact(x, 1, 8, 2, 2, k0, 64, u_k, v0, 64, u_v, cos, sin, HD ** -0.5)
    # scores reach about 1e3, so their fp32 rounding (1e3 x 2^-24 x a few) moves probabilities by up to about 4e-4
    bound = _half_step(exp) * 1.001 + 4e-4 * exp.abs().amax(-1, keepdim=True)
    assert bool(torch.isfinite(out).all()) and ((out - exp).abs() / bound).max().item() <= 1.0


@pytest.mark.parametrize("kf,qf,spike", [(0.0, 1.0, 1.0), (1e-25, 1e25, 1.0), (1e-12, 1e12, 1.0), (1.0, 1.0, 4096.0)])
def test_prefill_attention_plane_scales(gpu, kf, qf, spike):
    """The power-of-two scales of the score planes: keys that are all zero, keys and queries far apart in magnitude, and
    records whose keys differ by 2^12 (position 40's latent large, its products with the query kept small by it)."""
    x, k0, v0, u_k, u_v, cos, sin = _inputs(1, 96, 8, 2, 2, 64, 64, 9)
    x = x.clone()
    x[:, k0:v0] *= kf
    x[:, :k0] *= qf
    x[40, k0:v0] *= spike
    x[:, :k0] /= spike
    out = decoder_ops.prefill_attention(x, 1, 8, 2, 2, k0, 64, u_k, v0, 64, u_v, cos, sin, HD ** -0.5).double()
    exp = _exact(x, 1, 8, 2, 2, k0, 64, u_k, v0, 64, u_v, cos, sin, HD ** -0.5)
    bound = _half_step(exp) * 1.001 + 4e-6 * exp.abs().amax(-1, keepdim=True)
    assert ((out - exp).abs() / bound).max().item() <= 1.0


@pytest.mark.parametrize("nkv,G,rv", [(2, 2, 64), (4, 2, 96)])
@pytest.mark.parametrize("spike", [2.0 ** 20, 2.0 ** 28, float("inf"), float("-inf")])
def test_prefill_attention_one_key_out_of_line(gpu, nkv, G, rv, spike):
    """One key far above the others of its 32 (or infinite): the rows before it, which don't see it, keep their results bit
    for bit, and the rows after it stay at the bound of test_prefill_attention where its score is that of one key among
    others or rules it out (its products with these queries are above 1e3 in size)."""
    x, k0, v0, u_k, u_v, cos, sin = _inputs(1, 96, 8, nkv, G, 64, rv, 9)
    run = lambda t: decoder_ops.prefill_attention(t, 1, 8, nkv, G, k0, 64, u_k, v0, rv, u_v, cos, sin, HD ** -0.5)
    y = x.clone()
    y[40, k0:v0] *= spike
    out = run(y)
    assert torch.equal(out[:40], run(x)[:40])
    if abs(spike) != float("inf"):
        exp = _exact(y, 1, 8, nkv, G, k0, 64, u_k, v0, rv, u_v, cos, sin, HD ** -0.5)
        bound = _half_step(exp) * 1.001 + 4e-6 * exp.abs().amax(-1, keepdim=True)
        assert ((out.double() - exp).abs() / bound).max().item() <= 1.0


@pytest.mark.parametrize("value", [3e38, -3e38, float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("full_k", [True, False])
def test_prefill_attention_key_at_the_end_of_the_range(gpu, full_k, value):
    """One element of one key (or of its latent) at the end of bf16's range or not finite: results are finite where the
    64-bit ones are (rows before it, and those where its score is -inf), at the bound, and NaN where they are."""
    rk = HD if full_k else 64
    x, k0, v0, u_k, u_v, cos, sin = _inputs(1, 96, 8, 2, 2, rk, 64, 12, full_k=full_k)
    x = x.clone()
    x[40, [k0 + 6, k0 + rk + 9]] = value
    out = decoder_ops.prefill_attention(x, 1, 8, 2, 2, k0, rk, u_k, v0, 64, u_v, cos, sin, HD ** -0.5).double()
    exp = _exact(x, 1, 8, 2, 2, k0, rk, u_k, v0, 64, u_v, cos, sin, HD ** -0.5)
    exp, out = exp.view(96, 8, HD), out.view(96, 8, HD)
    fin = torch.isfinite(exp)
    assert torch.equal(torch.isfinite(out), fin) and bool(fin[:40].all())
    exp, out = exp.nan_to_num(0.0), out.nan_to_num(0.0)
    bound = _half_step(exp) * 1.001 + 4e-6 * exp.abs().amax(-1, keepdim=True) + 1e-30
    assert ((out - exp).abs() / bound).max().item() <= 1.0


def test_prefill_whole_v_heads_keep_a_nonfinite_value_in_its_column(gpu):
    x, k0, v0, u_k, _, cos, sin = _inputs(1, 64, 4, 1, 1, 64, HD, 3, full_v=True)
    x = x.clone()
    x[50, v0 + 21] = float("inf")
    out = decoder_ops.prefill_attention(x, 1, 4, 1, 1, k0, 64, u_k, v0, HD, None, cos, sin, HD ** -0.5)
    other = torch.arange(4 * HD, device="cuda") % HD != 21
    assert bool(torch.isfinite(out[:, other]).all()) and not bool(torch.isfinite(out[50:, ~other]).any())


@pytest.mark.parametrize("kind,w", [("rows", 40), ("rows", 64), ("k", 48), ("k", 64), ("k", 112), ("v", 16), ("v", 80)])
@pytest.mark.parametrize("n_pos", [1, 8, 37, 64])
def test_fill_matches_write_rows(gpu, kind, w, n_pos):
    B, G, S, users, user = 4, 3, 64, 2, 1
    g = torch.Generator().manual_seed(n_pos + w)
    src = torch.randn(users * n_pos, 8 + G * w + 8, generator=g).to(torch.bfloat16).cuda()
    rows = torch.randn(B, G, S, w, generator=g).to(torch.bfloat16).cuda()
    cache = rows.clone() if kind == "rows" else LatentCache.from_rows(rows, kind)
    decoder_ops.fill_from(cache, user, src, users, n_pos, 8, w)
    rows[user:user + users, :, :n_pos] = src[:, 8:8 + G * w].view(users, n_pos, G, w).transpose(1, 2)
    assert torch.equal(cache if kind == "rows" else cache.to_rows(), rows)


def _layer(rk, rv, gs, layout, users, cap, group_ranks=None):
    dim, nh, nkv = 256, 8, 4
    g = torch.Generator().manual_seed(rk + rv)
    W = {"q": torch.randn(nh * HD, dim, generator=g) * 0.05, "o": torch.randn(dim, nh * HD, generator=g) * 0.05}
    n_groups = nkv // gs
    vt = lambda r: (torch.randn(n_groups, r, dim, generator=g) * 0.05).repeat_interleave(gs, 0)
    lr = convert.LowRank(vt(rk), torch.randn(nkv, HD, rk, generator=g) / rk ** 0.5, vt(rv),
                         torch.randn(nkv, HD, rv, generator=g) / rv ** 0.5, group_size=gs)
    sd = {"layers.0.attention.wq.weight": W["q"], "layers.0.attention.wo.weight": W["o"]}
    sd.update({f"layers.0.attention.palu.{k}": t for k, t in convert.palu_layer_tensors(W, lr, nh, nkv, HD).items()})

    class Args:
        pass
    a = Args()
    a.dim, a.n_heads, a.n_kv_heads, a.head_dim, a.max_seq_len, a.max_batch_size = dim, nh, nkv, HD, cap, users + 1
    a.rope_theta, a.rope_scaling = 500000.0, None
    a.palu = convert.PaluConfig(rank_k=[rk], rank_v=[rv], cache_id="t", group_size=gs,
                                group_ranks=[group_ranks] if group_ranks else None)
    return PaluAttention("cuda:0", None, a, sd, None, 0, cache_layout=layout), g


@pytest.mark.parametrize("rk,rv,gs,layout,group_ranks", [
    (64, 48, 1, "tiled", None), (64, 96, 1, "rows", None), (HD, HD, 1, "tiled", None), (HD, 32, 1, "rows", None),
    (96, 128, 2, "tiled", None), (96, 128, 2, "rows", None), (96, 128, 2, "tiled", ([96, 64], [32, 128]))])
def test_layer_prefill_matches_the_torch_path(gpu, rk, rv, gs, layout, group_ranks):
    """The kernels' prefill against the torch path (which a layer takes under autograd): outputs to bf16 rounding, caches
    bit for bit except rotated keys, whose rounding may fall to the neighbouring bf16 value."""
    users, S = 2, 45
    att, g = _layer(rk, rv, gs, layout, users, 64, group_ranks)
    x = torch.randn(users, S + 3, 256, generator=g).to(torch.bfloat16).cuda()[:, :S]          # rows of a wider tensor
    out = att.forward(x, mode="prefill", user_id=1)
    got = [att._store(c).clone() for c in att.layer_past]
    for c in att.layer_past:
        att._store(c).zero_()
    exp = torch.stack([att._prefill_one(x[u], 1 + u) for u in range(users)])
    # one bf16 rounding of each attention value, then fp32-accumulated products rounded to bf16: both paths within
    # 2^-8 of the result's scale
    assert ((out - exp).double().norm() / exp.double().norm()).item() < 2.0 ** -8
    for i, c in enumerate(att.layer_past):
        store = att._store(c)
        if i == 0 and not att.recon_k:
            assert ((got[0].double() - store.double()).abs() <= store.double().abs() * 2.0 ** -7).all()
        else:
            assert torch.equal(got[i], store)


def test_layer_prefill_takes_unaligned_prompts(gpu):
    """A prompt that starts off a 16-byte boundary (a view into a larger buffer) gives what an aligned copy gives."""
    att, g = _layer(64, 64, 1, "tiled", 1, 64)
    buf = torch.randn(1 + 20 * 256, generator=g).to(torch.bfloat16).cuda()
    x = buf[1:].view(1, 20, 256)
    assert x.data_ptr() % 16
    assert torch.equal(att.forward(x, mode="prefill"), att.forward(x.clone(), mode="prefill"))


@pytest.mark.parametrize("as_type", [np.int64, torch.tensor])
def test_layer_prefill_takes_integer_types_as_user_id(gpu, as_type):
    att, g = _layer(64, 64, 1, "tiled", 1, 64)
    x = torch.randn(1, 20, 256, generator=g).to(torch.bfloat16).cuda()
    out = att.forward(x, mode="prefill", user_id=1)
    exp = [c.data.clone() for c in att.layer_past]
    for c in att.layer_past:
        c.data.zero_()
    assert torch.equal(att.forward(x, mode="prefill", user_id=as_type(1)), out)
    assert all(torch.equal(c.data, e) for c, e in zip(att.layer_past, exp))


@pytest.mark.parametrize("kind", ["wider rows", "every other position", "fp32", "unaligned"])
def test_layer_prefill_fills_caches_of_the_callers(gpu, kind):
    """Row-major caches that a caller put into layer_past as views or in another type are filled as torch fills them."""
    att, g = _layer(64, 32, 1, "rows", 1, 64)
    x = torch.randn(1, 20, 256, generator=g).to(torch.bfloat16).cuda()
    out = att._prefill_one(x[0], 1)
    exp = [c.clone() for c in att.layer_past]

    def other(c):
        B, G, S, w = c.shape
        if kind == "wider rows":
            return torch.zeros(B, G, S, w + 16, dtype=c.dtype, device=c.device)[..., :w]
        if kind == "every other position":
            return torch.zeros(B, G, 2 * S, w, dtype=c.dtype, device=c.device)[:, :, ::2]
        if kind == "fp32":
            return torch.zeros_like(c, dtype=torch.float32)
        return torch.zeros(1 + c.numel(), dtype=c.dtype, device=c.device)[1:].view(c.shape)
    att.layer_past = [other(c) for c in att.layer_past]
    assert torch.equal(att.forward(x, mode="prefill", user_id=1)[0], out)
    assert all(torch.equal(c.to(torch.bfloat16), e) for c, e in zip(att.layer_past, exp))


def test_layer_prefill_keeps_autograd(gpu):
    att, g = _layer(64, 64, 1, "rows", 1, 64)
    x = torch.randn(1, 20, 256, generator=g).cuda().requires_grad_()
    att.layer_past = [c.clone() for c in att.layer_past]
    out = att.forward(x, mode="prefill")
    assert out.requires_grad
    out.float().sum().backward()
    assert x.grad is not None and bool(x.grad.abs().sum() > 0)

"""The naive decode (palu_naive_decode) against 64-bit torch on the same bf16 latents and factors.

Bound: a key's dims are rounded to bf16 once (2^-9 relative), so a score is off by at most 2^-9 |q| . |K| scale (plus the
query's own scaled bf16 rounding, as much again), which moves a probability by that times itself; the probabilities
are rounded to bf16 (2^-9) and so is the result."""
import pytest
import torch

from palu_tt import fused
from palu_tt.cache import LatentCache

pytestmark = pytest.mark.gpu

HD = 128


def _case(B, S, nkv, rep, rk, rv, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    return (r(1, B, nkv * rep, HD).cuda(), r(B, nkv, S, rk).cuda(), r(B, nkv, S, rv).cuda(),
            (r(nkv, rk, HD).float() / rk ** 0.5).to(torch.bfloat16).cuda(), *(t.cuda() for t in fused.cos_sin_tables(HD, S, 5e5, None)))


def _check(out, q, k, v, u_k, cos, sin, lens, scale):
    B, nkv = k.shape[:2]
    rep = q.shape[2] // nkv
    for b, n in enumerate(lens):
        if n == 0:
            assert not out[0, b].any()
            continue
        for h in range(nkv):
            K = k[b, h, :n].double() @ u_k[h].double()
            p = K.unflatten(-1, (-1, 2))
            K = K * cos[:n].double() + torch.stack((-p[..., 1], p[..., 0]), -1).flatten(-2) * sin[:n].double()
            qh, V = q[0, b, h * rep:(h + 1) * rep].double(), v[b, h, :n].double()
            w = torch.softmax(qh @ K.T * scale, -1)
            err = 2.0 ** -8 * (qh.abs() @ K.abs().T).amax(-1, keepdim=True) * scale
            # a score error e scales a probability by at most exp(2 e) against the others
            bound = ((torch.exp(2 * err) - 1 + 2.0 ** -7) * w) @ V.abs() + 2.0 ** -8 * (w @ V).abs() + 1e-6
            d = (out[0, b, h * rep:(h + 1) * rep].double() - w @ V).abs()
            assert (d <= bound).all(), f"row {b} head {h}: {(d / bound).max().item():.3f} of the bound"
            # and, as a whole, far closer than the worst case: rounding errors are independent
            assert d.norm() <= 2.0 ** -6 * (w @ V).norm() + 1e-6


# every K width (half tiles among them), lengths around the 32-position blocks and 4-block workgroups, empty rows,
# positions past recon_len (clamped), several blocks a wave (the last)
@pytest.mark.parametrize("B,S,recon,nkv,rep,rk,rv,pos", [
    (1, 32, 32, 1, 1, 16, 32, [0]), (2, 64, 64, 2, 4, 48, 48, [31, 32]), (3, 160, 128, 2, 4, 64, 80, [127, 159, 3]),
    (2, 320, 320, 3, 2, 96, 32, [319, 128]), (2, 288, 288, 8, 4, 112, 112, [-1, 287]), (4, 256, 64, 2, 4, 80, 64, [63, 12, 200, 0]),
    (3, 8192, 8192, 8, 4, 64, 64, [8191, 5000, 100])])
def test_naive_tiled(gpu, B, S, recon, nkv, rep, rk, rv, pos):
    q, k, v, u_k, cos, sin = _case(B, S, nkv, rep, rk, rv, S + rk)
    cp = torch.tensor(pos, dtype=torch.int32, device="cuda")
    out = fused.naive_decode(q, LatentCache.from_rows(k, "k"), u_k, cos, sin, LatentCache.from_rows(v, "v"), cp, recon)
    _check(out, q, k, v, u_k, cos, sin, [min(p + 1, recon) for p in pos], HD ** -0.5)


@pytest.mark.parametrize("B,S,recon,nkv,rep,rk,rv,pos", [
    (1, 1, 1, 1, 4, 32, 32, [0]), (2, 100, 64, 2, 4, 64, 96, [99, 40]), (2, 333, 333, 2, 3, 96, 128, [332, 256]),
    (1, 130, 130, 4, 1, 32, 64, [128])])
def test_naive_rows(gpu, B, S, recon, nkv, rep, rk, rv, pos):
    q, k, v, u_k, cos, sin = _case(B, S, nkv, rep, rk, rv, S + rk)
    cp = torch.tensor(pos, dtype=torch.int32, device="cuda")
    out = fused.naive_decode(q, k, u_k, cos, sin, v, cp, recon)
    _check(out, q, k, v, u_k, cos, sin, [min(p + 1, recon) for p in pos], HD ** -0.5)

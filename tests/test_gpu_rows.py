"""The prefill projection kernel (palu_linear_rows) against 64-bit torch.

Bound: half a bf16 step at the result plus the fp32 sum's rounding. A dot product of k terms is k / 32 MFMAs accumulated
one after another (and up to 16 slices added), each addition rounding by at most 2^-24 of the running sum, which the sum
of the terms' magnitudes bounds."""
import pytest
import torch

from palu_tt import decoder_ops as ops

pytestmark = pytest.mark.gpu


def _half_step(e):
    return torch.ldexp(torch.ones_like(e), torch.frexp(e).exponent - 9)


def _case(m, n, k, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(m, k + 8, generator=g).to(torch.bfloat16).cuda()[:, :k]
    w = (torch.randn(n, k, generator=g) * 0.05).to(torch.bfloat16).cuda()
    return x, w


# rows around the 128-row blocks; columns that are no whole workgroup, and last groups of fewer row tiles; k of one
# tile, an odd number of tiles, every remainder of the four-stage round, and lengths that split (odd slices among them)
@pytest.mark.parametrize("m,n,k,rtw", [
    (65, 16, 32, 1), (127, 48, 64, 2), (128, 80, 96, 3), (129, 272, 160, 4), (300, 1040, 224, 7), (70, 528, 288, 8),
    (200, 512, 352, 5), (257, 64, 416, 6), (1, 96, 512, 2), (100, 128, 2080, 1), (66, 256, 4128, 3), (500, 2064, 1056, 7),
    (1030, 4112, 128, 2)])
def test_linear_rows(gpu, m, n, k, rtw):
    x, w = _case(m, n, k, m + n + k)
    y = ops.linear_rows(x, ops.tile_weight(w, rtw), rtw).double()
    exp = x.double() @ w.double().T
    mag = x.double().abs() @ w.double().abs().T
    bound = _half_step(exp) * 1.001 + (k / 32 + 24) * 2.0 ** -24 * mag
    assert ((y - exp).abs() / bound).max().item() <= 1.0


# one row block of two-tile waves (n at most 64 workgroups' columns) and of four-tile waves, with 0 to 3 stages past the
# last whole round of four, odd slices among them: the last stages wait for copies that the main loop's counts don't cover
@pytest.mark.parametrize("k32", [6, 7, 14, 15, 22, 24, 30, 31, 60, 62])
@pytest.mark.parametrize("m,n", [(128, 1024), (96, 512), (300, 16384)])
def test_linear_rows_last_stages(gpu, m, n, k32):
    test_linear_rows(gpu, m, n, 32 * k32, 2)


@pytest.mark.parametrize("m,f,k,rtw", [(65, 32, 32, 1), (130, 96, 224, 7), (257, 544, 96, 3), (128, 1024, 512, 4), (33, 64, 64, 8)])
def test_linear_rows_swiglu(gpu, m, f, k, rtw):
    x, g = _case(m, f, k, f + k)
    u = _case(1, f, k, f + k + 1)[1]
    y = ops.linear_rows(x, ops.tile_weight(ops.interleave_gate_up(g, u), rtw), rtw, swiglu=True).double()
    xd, gd, ud = x.double(), g.double(), u.double()
    gv, uv = xd @ gd.T, xd @ ud.T
    exp = torch.nn.functional.silu(gv) * uv
    # the fp32 sums of gate and up (|d silu| <= 1.1), and the fp32 exponential and division: a few 2^-22 of the result
    eps = (k / 32 + 24) * 2.0 ** -24
    bound = _half_step(exp) * 1.001 + 1.1 * eps * (xd.abs() @ gd.abs().T) * uv.abs() + eps * gv.abs() * (xd.abs() @ ud.abs().T) \
        + 2.0 ** -20 * exp.abs()
    assert ((y - exp).abs() / bound).max().item() <= 1.0


def test_few_rows_on_two_streams(gpu):
    """A prefill's products of at most 64 rows over one split weight, on two streams at once: each equals its result
    alone bit for bit (the split partials belong to the call, not to the weight)."""
    g = torch.Generator().manual_seed(3)
    lin = ops.DecodeLinear((torch.randn(512, 8192, generator=g) * 0.05).to(torch.bfloat16).cuda(), 64)
    assert lin.ks > 1, "the plan must split for this test"
    xs = [torch.randn(m, 8192, generator=g).to(torch.bfloat16).cuda() for m in (37, 60)]
    alone = [lin.rows(x).clone() for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]
    outs = [[], []]
    for _ in range(40):
        for s, x, o in zip(streams, xs, outs):
            with torch.cuda.stream(s):
                o.append(lin.rows(x))
    torch.cuda.synchronize()
    assert all(torch.equal(y, a) for a, o in zip(alone, outs) for y in o)

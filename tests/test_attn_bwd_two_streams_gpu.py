"""dk and dv at 64 / 64 with two streams of tiles a workgroup, where that can go wrong: a stream without a tile, odd and even
numbers of them, more tiles than stages, several query heads, several runs beside the streams, a block mask that leaves one stream
many tiles and the other few, and the largest call of this form beside the next (which takes one stream)."""
import math

import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _run(family, q, k, v, dout, causal, scale, bias, **masks):
    from metaattention_amd import hip_backend as hb
    fam = {"softmax": hb.MA_ATTN_SOFTMAX, "sigmoid": hb.MA_ATTN_SIGMOID, "relu": hb.MA_ATTN_RELU}[family]
    B, Sq, H, _ = q.shape
    lse = torch.empty(B, H, Sq, device="cuda") if family == "softmax" else None
    o = hb.attn_fwd(q, k, v, family=fam, causal=causal, scale=scale, bias=bias, row_scale=lse, elem_mask=masks.get("elem_mask"))
    return hb.attn_bwd(q, k, v, o, dout, lse, family=fam, causal=causal, scale=scale, bias=bias, **masks)


def _reference(family, q, k, v, dout, allow, scale, bias):
    """Gradients in float64 (allow: which scores are kept)."""
    rep = q.shape[2] // k.shape[2]
    qd, kd, vd = (t.double().requires_grad_() for t in (q, k, v))
    ke, ve = kd.repeat_interleave(rep, 2), vd.repeat_interleave(rep, 2)
    x = torch.matmul(qd.transpose(1, 2), ke.permute(0, 2, 3, 1)) * scale + bias
    if family == "softmax":
        p = torch.softmax(x.masked_fill(~allow, -1e300), -1) * allow
    else:
        p = (torch.sigmoid(x) if family == "sigmoid" else torch.relu(x)) * allow
    return torch.autograd.grad(torch.matmul(p, ve.transpose(1, 2)).transpose(1, 2), (qd, kd, vd), dout.double())


@pytest.mark.parametrize("B,H,Hkv,Sq,Skv,causal", [
    (1, 2, 2, 20, 20, True),          # one tile
    (1, 3, 1, 31, 200, False),        # one tile for each of three heads
    (1, 4, 2, 290, 290, True),        # 10, 6 and 2 tiles of two heads
    (2, 3, 3, 700, 450, False),       # 22 tiles
    (1, 6, 2, 1000, 100, False),      # several runs beside the streams, 96 tiles
    (2, 8, 8, 1025, 1025, True)])
@pytest.mark.parametrize("family,dtype", [("softmax", torch.bfloat16), ("sigmoid", torch.float16), ("relu", torch.bfloat16)])
def test_two_streams(B, H, Hkv, Sq, Skv, causal, family, dtype):
    g = torch.Generator().manual_seed(Sq + Skv)
    q, k, v, dout = (torch.randn(B, s, h, 64, generator=g).to(dtype) for s, h in ((Sq, H), (Skv, Hkv), (Skv, Hkv), (Sq, H)))
    scale, bias = (0.125, 0.0) if family == "softmax" else (0.125, -2.0) if family == "sigmoid" else (0.02, 0.0)
    got = _run(family, *(t.cuda() for t in (q, k, v, dout)), causal, scale, bias)
    allow = torch.arange(Sq).view(Sq, 1) >= torch.arange(Skv).view(1, Skv) if causal else torch.ones(Sq, Skv, dtype=torch.bool)
    for name, a, b in zip(("dq", "dk", "dv"), got, _reference(family, q, k, v, dout, allow, scale, bias)):
        # p and ds are rounded to the tensor type (2^-9 of each, at random): of the 2-norm of a gradient that is well below 1e-2
        assert (a.double().cpu() - b).norm() <= 1e-2 * b.norm(), f"{name} {family} {(B, H, Hkv, Sq, Skv, causal)}"


@pytest.mark.parametrize("every,S", [(2, 1000), (3, 1024)])      # (rows of 1024 bytes come with the tile, others element by element)
def test_block_mask_that_favours_a_stream(every, S):
    """Tiles 0, every, 2 * every, ... of the queries: with two all of them are one stream's (of even heads)."""
    B, H = 1, 2
    g = torch.Generator().manual_seed(every)
    q, k, v, dout = (torch.randn(B, S, H, 64, generator=g).bfloat16() for _ in range(4))
    rows = (torch.arange(S) // 32) % every == 0
    keep = (torch.rand(1, 1, S, S, generator=g) < 0.7) & rows.view(S, 1)
    keep[..., :130] = False                    # (a key block and two keys without any query)
    pad = lambda m: torch.nn.functional.pad(m, (0, 1024 - S, 0, 1024 - S))
    kp = pad(keep[0, 0]).to(torch.uint8)
    kbm, qbm = (m.view(8, 128, 32, 32).amax(dim=(1, 3)).view(1, 1, 8, 32).cuda() for m in (kp, kp.t().contiguous()))
    em, emt = kp[:S, :S].contiguous().view(1, 1, S, S).cuda(), kp.t()[:S, :S].contiguous().view(1, 1, S, S).cuda()
    got = _run("softmax", *(t.cuda() for t in (q, k, v, dout)), False, 0.125, 0.0, elem_mask=em, elem_mask_t=emt, kv_block_mask=kbm, q_block_mask=qbm)
    for name, a, b in zip(("dq", "dk", "dv"), got, _reference("softmax", q, k, v, dout, keep, 0.125, 0.0)):
        assert (a.double().cpu() - b).norm() <= 1e-2 * b.norm(), name       # (as above)
    assert torch.count_nonzero(got[1][:, :130]) == 0 and torch.count_nonzero(got[2][:, :130]) == 0


@pytest.mark.parametrize("tiles", [[3], [3, 5], [2, 4], [2, 3, 5], [1, 3, 5, 7, 9], [2, 5, 6, 7, 8, 9, 11]])     # (none to four and more of a stream)
@pytest.mark.parametrize("H,Hkv", [(2, 2), (2, 1)])
@pytest.mark.parametrize("family", ["softmax", "sigmoid", "relu"])
def test_hidden_queries_stay_hidden(tiles, H, Hkv, family):
    """A gradient of the output that is not finite, in rows that the mask hides from every key: dk and dv have the bits that they
    have without it."""
    S = 384
    g = torch.Generator().manual_seed(len(tiles))
    q, k, v, dout = (torch.randn(1, S, h, 64, generator=g).bfloat16().cuda() for h in (H, Hkv, Hkv, H))
    keep = torch.zeros(S, dtype=torch.bool)
    for t in tiles:
        keep[32 * t:32 * t + 32] = True
    em = keep.view(S, 1).expand(S, S).to(torch.uint8).contiguous().view(1, 1, S, S).cuda()
    emt = em.transpose(2, 3).contiguous()
    kbm, qbm = (m.view(3, 128, 12, 32).amax(dim=(1, 3)).view(1, 1, 3, 12).contiguous() for m in (em, emt))
    scale, bias = (0.125, 0.0) if family != "sigmoid" else (0.125, -2.0)
    run = lambda grad: _run(family, q, k, v, grad, False, scale, bias, elem_mask=em, elem_mask_t=emt, kv_block_mask=kbm, q_block_mask=qbm)
    want = run(dout)
    assert all(torch.isfinite(t).all() and torch.count_nonzero(t) > 0 for t in want[1:])
    for bad in (float("nan"), float("inf")):
        for head in range(H):
            grad = dout.clone()
            grad[0, :, head] = torch.where(keep.view(S, 1).cuda(), grad[0, :, head], bad)
            got = run(grad)
            assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2]), f"{bad} in head {head}"


def test_both_sides_of_the_rule():
    """512 and 516 key blocks: the same sequences' gradients from two streams and from one."""
    g = torch.Generator().manual_seed(1)
    q, k, v, dout = (torch.randn(1, 512, 129, 64, generator=g).bfloat16().cuda() for _ in range(4))
    two = _run("softmax", *(t[:, :, :128].contiguous() for t in (q, k, v, dout)), True, 0.125, 0.0)
    one = _run("softmax", q, k, v, dout, True, 0.125, 0.0)
    for name, a, b in zip(("dq", "dk", "dv"), two, one):
        # the sums are formed in another order in fp32 (512 products below 32: 512 * 32 * 2^-24 apart at most) and rounded to
        # bf16 once: a unit of the last place
        b = b[:, :, :128].float()
        assert ((a.float() - b).abs() <= 2 ** -7 * b.abs() + 1e-3).all(), name

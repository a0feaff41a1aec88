"""dk and dv by pairs of waves (128 / 128, 192 / 128, 128 / 256, 256 / 256), where that can go wrong: one tile, as many tiles as stages and one
more or fewer, several query heads, runs of steps, and masks that leave a key block nothing."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(family, q, k, v, dout, causal, scale, bias, **masks):
    from metaattention_amd import hip_backend as hb
    fam = {"softmax": hb.MA_ATTN_SOFTMAX, "sigmoid": hb.MA_ATTN_SIGMOID, "relu": hb.MA_ATTN_RELU}[family]
    B, Sq, H, _ = q.shape
    lse = torch.empty(B, H, Sq, device="cuda") if family == "softmax" else None
    o = hb.attn_fwd(q, k, v, family=fam, causal=causal, scale=scale, bias=bias, row_scale=lse, elem_mask=masks.get("elem_mask"))
    return hb.attn_bwd(q, k, v, o, dout, lse, family=fam, causal=causal, scale=scale, bias=bias, **masks)


def _check(family, q, k, v, dout, allow, scale, bias, got, what):
    rep = q.shape[2] // k.shape[2]
    qd, kd, vd = (t.double().requires_grad_() for t in (q, k, v))
    ke, ve = kd.repeat_interleave(rep, 2), vd.repeat_interleave(rep, 2)
    x = torch.matmul(qd.transpose(1, 2), ke.permute(0, 2, 3, 1)) * scale + bias
    if family == "softmax":
        p = torch.softmax(x.masked_fill(~allow, -1e300), -1) * allow
    else:
        p = (torch.sigmoid(x) if family == "sigmoid" else torch.relu(x)) * allow
    ref = torch.autograd.grad(torch.matmul(p, ve.transpose(1, 2)).transpose(1, 2), (qd, kd, vd), dout.double())
    for name, a, b in zip(("dq", "dk", "dv"), got, ref):
        # p and ds are rounded to the tensor type (2^-9 of each, at random): of the 2-norm of a gradient that is well below 1e-2
        assert (a.double().cpu() - b).norm() <= 1e-2 * b.norm(), f"{name} {what}"


def _case(B, H, Hkv, Sq, Skv, D, DV, dtype):
    g = torch.Generator().manual_seed(Sq + Skv + D)
    return [torch.randn(B, s, h, d, generator=g).to(dtype) for s, h, d in ((Sq, H, D), (Skv, Hkv, D), (Skv, Hkv, DV), (Sq, H, DV))]


@pytest.mark.parametrize("D,DV", [(128, 128), (192, 128), (128, 256), (256, 256)])
@pytest.mark.parametrize("B,H,Hkv,Sq,Skv,causal", [
    (1, 2, 2, 20, 20, True),           # one tile of one block of keys
    (1, 3, 1, 31, 200, False),         # one tile for each of three heads
    (2, 3, 3, 97, 300, False),         # an odd number of heads, less tiles than stages
    (1, 2, 2, 160, 129, False),        # as many tiles as stages, less one, and a second block of one key
    (1, 2, 2, 193, 100, False),        # more tiles than stages, the last of one row
    (1, 4, 2, 420, 420, True),         # pairs of key blocks, in runs
    (16, 16, 16, 290, 290, True)])     # more items than workgroups
@pytest.mark.parametrize("family,dtype", [("softmax", torch.bfloat16), ("sigmoid", torch.float16), ("relu", torch.bfloat16)])
def test_pairs(B, H, Hkv, Sq, Skv, causal, D, DV, family, dtype):
    q, k, v, dout = _case(B, H, Hkv, Sq, Skv, D, DV, dtype)
    scale, bias = (D ** -0.5, 0.0) if family == "softmax" else (D ** -0.5, -2.0) if family == "sigmoid" else (0.02, 0.0)
    what = f"{family} B{B} H{H}/{Hkv} {Sq} x {Skv} {D}/{DV} causal={causal}"
    print(what, flush=True)
    got = _run(family, *(t.cuda() for t in (q, k, v, dout)), causal, scale, bias)
    allow = torch.arange(Sq).view(Sq, 1) >= torch.arange(Skv).view(1, Skv) if causal else torch.ones(Sq, Skv, dtype=torch.bool)
    _check(family, q, k, v, dout, allow, scale, bias, got, what)


@pytest.mark.parametrize("D,DV", [(128, 128), (192, 128), (128, 256), (256, 256)])
@pytest.mark.parametrize("S,first", [(320, 100), (300, 0), (416, 200)])      # (rows of a multiple of 16 bytes come with the tile, others element by element)
def test_pairs_with_masks(S, first, D, DV):
    """A window of 70 keys over the rows from `first` on: rows and whole key blocks without a score, tiles kept in part and in full."""
    B, H, Hkv = 1, 4, 2
    q, k, v, dout = _case(B, H, Hkv, S, S, D, DV, torch.bfloat16)
    i, j = torch.arange(S).view(S, 1), torch.arange(S).view(1, S)
    allow = (i >= first) & (j <= i) & (i - j < 70)
    n = (S + 127) // 128 * 128
    full = torch.zeros(n, n, dtype=torch.bool)
    full[:S, :S] = allow
    inside = torch.ones(n, n, dtype=torch.bool)
    inside[:S, :S] = allow
    pool = lambda a, b: (full.view(n // a, a, n // b, b).any(3).any(1).to(torch.uint8) + (inside.view(n // a, a, n // b, b).all(3).all(1)).to(torch.uint8))
    up = lambda x: ((x + 31) // 32)
    masks = dict(elem_mask=allow.to(torch.uint8).view(1, 1, S, S).cuda(), elem_mask_t=allow.t().contiguous().to(torch.uint8).view(1, 1, S, S).cuda(),
                 kv_block_mask=pool(128, 32)[:, :up(S)].contiguous().view(1, 1, -1, up(S)).cuda(),
                 q_block_mask=pool(32, 128)[:up(S)].t().contiguous().view(1, 1, -1, up(S)).cuda())
    print(f"masks S{S} {first} {D}/{DV}", flush=True)
    got = _run("softmax", *(t.cuda() for t in (q, k, v, dout)), False, D ** -0.5, 0.0, **masks)
    _check("softmax", q, k, v, dout, allow, D ** -0.5, 0.0, got, f"S{S} {first} {D}/{DV}")

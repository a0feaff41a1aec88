"""The forward kernel's walk over a block mask, 64 tiles of 32 keys at a time, and its forms with and without score terms: more
tiles than one or two such groups, groups of which nothing is kept, a query block without a key, streams with very different
numbers of tiles, blocks that need no element-wise mask, blocks of more than a tile, causal rows that share a workgroup with later
ones (256 / 256: their tiles above the diagonal are multiplied by zeros)."""
import math

import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,DV", [(64, 64), (128, 128), (192, 128), (256, 256)])
@pytest.mark.parametrize("S,Skv,block,causal", [(40, 2047, 32, False), (300, 4200, 32, False), (130, 2111, 64, False), (2100, 2100, 32, True)])
@pytest.mark.parametrize("terms", [False, True])
def test_block_mask(D, DV, S, Skv, block, causal, terms):
    from metaattention_amd import hip_backend as hb
    B, H, scale = 1, 3, 1 / math.sqrt(D)
    g = torch.Generator().manual_seed(S + Skv + D)
    q, k, v = (torch.randn(B, s, H, d, generator=g).bfloat16() for s, d in ((S, D), (Skv, D), (Skv, DV)))
    nq, nb = (S + 127) // 128, (Skv + block - 1) // block
    blocks = (torch.rand(1, H, nq, nb, generator=g) < 0.3).to(torch.uint8)
    blocks[0, 0] = 0                                  # head 0: a few tiles of the last group, all in one stream of four
    blocks[0, 0, :, nb // 8 * 4::4] = 1
    blocks[0, 1, nq - 1] = 0                          # head 1: its last query block has no key
    elem = torch.rand(1, H, S, Skv, generator=g) < 0.5
    keep = blocks.repeat_interleave(128, 2)[:, :, :S].repeat_interleave(block, 3)[..., :Skv]
    whole = blocks.clone()
    whole[0, 2][blocks[0, 2] > 0] = 2                 # head 2: no block of it needs the element-wise mask
    elem[0, 2] = True
    for what, mask, em in (("blocks", blocks, None), ("blocks and elements", whole, elem))[:1 if causal else 2]:
        allow = keep.bool() if em is None else keep.bool() & em
        if causal:
            allow = allow & (torch.arange(S).view(S, 1) >= torch.arange(Skv).view(1, Skv))
        # head 2's mask is not read where its blocks say so: whatever it holds there gives the same
        given = None if em is None else torch.nn.functional.pad(em.index_fill(1, torch.tensor([2]), False), (0, -Skv % 4)).cuda()[..., :Skv]
        s = (torch.matmul(q.double().transpose(1, 2), k.double().permute(0, 2, 3, 1)) * scale).masked_fill(~allow, float("-inf"))
        ref = torch.matmul(torch.nan_to_num(torch.softmax(s, -1)), v.double().transpose(1, 2)).transpose(1, 2)
        lse = torch.full((B, H, S), float("nan"), device="cuda")
        # a term of zeros for every score: the kernel with score terms, the same numbers
        add = torch.zeros(1, 1, 1, 1, device="cuda") if terms else None
        print(f"D{D} DV{DV} S{S} Skv{Skv} block{block} causal={causal} terms={terms}: {what}", flush=True)
        o = hb.attn_fwd(q.cuda(), k.cuda(), v.cuda(), family=hb.MA_ATTN_SOFTMAX, causal=causal, scale=scale, kv_block_mask=mask.cuda(), kv_block_size=block,
                        elem_mask=given, row_scale=lse, score_add=add)
        oracle.assert_close(o.float().cpu(), ref, rtol=1e-2, atol=2e-2)
        torch.testing.assert_close(lse.cpu().double(), torch.logsumexp(s, -1), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("family", ["softmax", "sigmoid", "relu"])
@pytest.mark.parametrize("D,DV", [(256, 256), (256, 512)])
@pytest.mark.parametrize("S", [33, 300])
def test_infinities_above_the_diagonal(family, D, DV, S):
    """The values above the diagonal of a 32-row group are not looked at, infinite ones included."""
    from metaattention_amd import hip_backend as hb
    fam = {"softmax": hb.MA_ATTN_SOFTMAX, "sigmoid": hb.MA_ATTN_SIGMOID, "relu": hb.MA_ATTN_RELU}[family]
    g = torch.Generator().manual_seed(S + DV)
    q, k, v = (torch.randn(1, S, 2, d, generator=g).bfloat16().cuda() for d in (D, D, DV))
    run = lambda v: hb.attn_fwd(q, k, v, family=fam, causal=True, scale=0.1, bias=0.0)
    print(f"{family} D{D} DV{DV} S{S}", flush=True)
    want = run(v)
    for first in range(32, S, 96):
        bad = v.clone()
        bad[:, first:] = float("inf")
        assert torch.equal(run(bad)[:, :first], want[:, :first])

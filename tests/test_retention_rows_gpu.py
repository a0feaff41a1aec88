"""The wide retention forward with a generated multiplier: whole tiles by offsets from their first row, a last tile that ends inside
row by row, as are rows that are too far apart for 32-bit offsets (the same numbers, so the same bits)."""
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 31, 32, 33, 95, 96, 97, 300])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows(S, dtype):
    from metaattention_amd import hip_backend as hb
    g = torch.Generator().manual_seed(S)
    H = 2
    q, k = (torch.randn(1, S, H, 256, generator=g).mul(1 / 16).to(dtype).cuda() for _ in range(2))
    v = torch.randn(1, S, H, 512, generator=g).to(dtype).cuda()
    gamma = torch.tensor([1 - 2.0 ** -5, 1 - 2.0 ** -8]).cuda()
    run = lambda k, v: hb.attn_fwd(q, k, v, family=hb.MA_ATTN_RETENTION, causal=True, scale=1.0, decay_gamma=gamma)
    out = run(k, v)
    i = torch.arange(S, dtype=torch.float64)
    d = i.view(S, 1) - i
    m = torch.where(d >= 0, gamma.double().cpu().view(H, 1, 1) ** d.clamp(min=0), 0.0)
    p = torch.matmul(q.double().cpu().transpose(1, 2), k.double().cpu().permute(0, 2, 3, 1)) * m
    want = torch.matmul(p / p.abs().sum(-1, keepdim=True).clamp(min=1), v.double().cpu().transpose(1, 2)).transpose(1, 2)
    oracle.assert_close(out.float().cpu(), want, rtol=1e-2, atol=2e-2)
    if S <= 33:      # rows of 64 MB: beyond the offsets
        far = torch.empty(S * (1 << 25), dtype=dtype, device="cuda")
        strided = lambda t: far.as_strided(t.shape, (0, 1 << 25, t.shape[3], 1)).copy_(t)
        assert torch.equal(run(strided(k), v), out) and torch.equal(run(k, strided(v)), out)

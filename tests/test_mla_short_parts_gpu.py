"""Ragged latent-cache decode from a plan, about the sizes where the parts of few batch entries get shorter: as many units (3 + the
32-row sub-tiles of an entry) as a quarter of the parts and as the parts, one more, and beyond 64 entries, whose lengths are looked up
another way."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,lens", [
    (16, [1]), (32, [100]), (32, [416] * 8), (32, [416] * 7 + [417]), (32, [416] * 31 + [417, 1]), (16, [416] * 32), (32, [416] * 32 + [0]),
    (64, [416] * 4), (64, [416] * 4 + [5]), (128, [300, 20]), (128, [416] * 16), (16, [33] * 64), (16, [33] * 65), (32, [7, 900] * 40)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_short_parts(H, lens, dtype):
    from metaattention_amd import hip_backend as hb
    B, page, most = len(lens), 64, max(lens)
    per = max(1, -(-most // page))
    g = torch.Generator().manual_seed(B * 1000 + most + H)
    q = torch.randn(B, 1, H, 576, generator=g).to(dtype).cuda()
    pool = torch.randn(B * per, page, 1, 576, generator=g).to(dtype).cuda()
    table = torch.randperm(B * per, generator=g).to(torch.int32).view(B, per).cuda()
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    print(f"H{H} B{B} {lens[:3]}", flush=True)
    out, lse = hb.flash_mla_with_kvcache(q, pool, table, sl, 512, *hb.get_mla_metadata(sl, H, 1))
    # the output (2^-9 or 2^-12), the partial results and the probabilities are rounded to the tensor type, at random: of the 2-norm
    # less than 3 such roundings
    bound = 3 * 2 ** (-9 if dtype == torch.bfloat16 else -12)
    for b, n in enumerate(lens):
        kv = pool[table[b].long()].reshape(-1, 576)[:n].double()
        if n == 0:
            assert torch.count_nonzero(out[b]) == 0 and torch.isneginf(lse[b]).all()
            continue
        s = (q[b, 0].double() @ kv.t()) * 576 ** -0.5
        ref = torch.softmax(s, -1) @ kv[:, :512]
        assert (out[b, 0].double() - ref).norm() <= bound * ref.norm(), b
        assert (lse[b, :, 0].double() - torch.logsumexp(s, -1)).abs().max() <= 1e-4, b

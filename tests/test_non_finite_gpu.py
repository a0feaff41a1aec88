"""NaN in an input: the outputs that depend on it are NaN, whichever way the call is cut, and the others have the bits they
have without it."""
import pytest
import torch

import specs

pytestmark = pytest.mark.gpu
NAN = float("nan")


def _rand(*shape, dtype):
    return torch.randn(*shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(sum(shape))).to(dtype)


@pytest.mark.parametrize("KV", [20, 200, 470, 1200])       # unsplit, and 2 splits and more
@pytest.mark.parametrize("H,Hkv,D,DV,dtype", [(4, 4, 128, 128, torch.bfloat16), (8, 2, 64, 64, torch.float16), (4, 1, 192, 128, torch.bfloat16)])
def test_decode(KV, H, Hkv, D, DV, dtype):
    mod = specs.softmax_attention_decode(2, H, 1, KV, D, DV, dtype=dtype, HKV=Hkv)
    q, k, v = _rand(2, 1, H, D, dtype=dtype), _rand(2, KV, Hkv, D, dtype=dtype), _rand(2, KV, Hkv, DV, dtype=dtype)
    out, scale = mod(q, k, v), mod.final_rowscales.view(2, H)
    grp = H // Hkv

    def check(rows, got, got_scale):
        assert got[:, 0][rows].isnan().all() and got_scale[rows].isnan().all()
        assert torch.equal(got[:, 0][~rows], out[:, 0][~rows]) and torch.equal(got_scale[~rows], scale[~rows])

    rows = torch.zeros(2, H, dtype=torch.bool, device="cuda")
    rows[1, 2] = True
    bad = q.clone()
    bad[1, 0, 2, 5] = NAN
    check(rows, mod(bad, k, v), mod.final_rowscales.view(2, H))
    for key in (0, KV - 1):                                # a key in the first split, one in the last
        rows = torch.zeros(2, H, dtype=torch.bool, device="cuda")
        rows[0, :grp] = True
        bad = k.clone()
        bad[0, key, 0, D - 1] = NAN
        check(rows, mod(q, bad, v), mod.final_rowscales.view(2, H))
        bad = v.clone()
        bad[0, key, 0, 7] = NAN
        got, want = mod(q, k, bad), out.clone()
        assert got[0, 0, :grp, 7].isnan().all()
        want[0, 0, :grp, 7] = got[0, 0, :grp, 7] = 0
        assert torch.equal(got, want) and torch.equal(mod.final_rowscales.view(2, H), scale)


@pytest.mark.parametrize("Hq,KV", [(16, 500), (128, 300)])
def test_latent_cache_decode(Hq, KV):
    from metaattention_amd import hip_backend as hb
    B = 3
    q, k = _rand(B, 1, Hq, 576, dtype=torch.bfloat16), _rand(B * 8, 64, 1, 576, dtype=torch.bfloat16)
    table = torch.arange(B * 8, dtype=torch.int32, device="cuda").view(B, 8)
    lens = torch.tensor([KV, 1, KV - 70], dtype=torch.int32, device="cuda")
    bad = q.clone()
    bad[2, 0, 4, 575] = NAN
    rows = torch.zeros(B, Hq, dtype=torch.bool, device="cuda")
    rows[2, 4] = True
    for plan in ((), hb.get_mla_metadata(lens, Hq, 1)):
        out, lse = hb.flash_mla_with_kvcache(q, k, table, lens, 512, *plan)
        got, got_lse = hb.flash_mla_with_kvcache(bad, k, table, lens, 512, *plan)
        assert got[:, 0][rows].isnan().all() and got_lse[..., 0][rows].isnan().all()
        assert torch.equal(got[:, 0][~rows], out[:, 0][~rows]) and torch.equal(got_lse[..., 0][~rows], lse[..., 0][~rows])


@pytest.mark.parametrize("B,H,S,D,DV", [(1, 4, 70, 128, 128), (1, 8, 300, 128, 128), (2, 4, 300, 128, 256), (1, 4, 200, 64, 64), (2, 16, 257, 192, 128), (1, 4, 300, 256, 256)])
@pytest.mark.parametrize("family", ["softmax", "sigmoid"])
def test_rows_before_a_value_under_a_causal_mask(B, H, S, D, DV, family):
    """The rows of the 32-row groups before that of a NaN value do not see it, however many rows a workgroup has."""
    mod = specs.softmax_attention(B, H, S, D, DV) if family == "softmax" else specs.sigmoid_attention(B, H, S, D, DV, const_bias=-4.0)
    q, k, v = (_rand(B, S, H, d, dtype=torch.bfloat16) for d in (D, D, DV))
    out = mod(q, k, v)
    for key in (S - 1, 63):
        bad = v.clone()
        bad[0, key, 1, 3] = NAN
        got, want, first = mod(q, k, bad), out.clone(), key // 32 * 32
        assert got[0, key:, 1, 3].isnan().all()
        got[0, first:, 1, 3] = want[0, first:, 1, 3] = 0
        assert torch.equal(got, want)

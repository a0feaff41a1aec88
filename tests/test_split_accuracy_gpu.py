"""Calls that are cut into kv splits (or pieces) where one workgroup could take them whole: the merge costs no accuracy against
the unsplit launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(*shape, dtype):
    return torch.randn(*shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(sum(shape))).to(dtype)


def _error(got, want):
    return float((got.double() - want).norm() / want.norm())


# Both launches round the probabilities and the output once.  What differs between them is which probabilities are rounded up and
# which down: of n outputs with independent roundings the two errors' ratio has a standard deviation of about (2 n)^-0.5, below
# 1.6 % for the 2048 outputs or more here; rounded partial results would cost 15 % and more.
ROOM = 1.06


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Hkv,KV,D,DV", [(1, 32, 8, 161, 128, 128), (4, 32, 8, 300, 64, 64), (8, 16, 16, 480, 192, 128), (2, 8, 8, 333, 256, 256), (36, 16, 16, 520, 128, 128)])
def test_decode(dtype, B, H, Hkv, KV, D, DV):
    from metaattention_amd import hip_backend as hb
    q, k, v = _rand(B, 1, H, D, dtype=dtype), _rand(B, KV, Hkv, D, dtype=dtype), _rand(B, KV, Hkv, DV, dtype=dtype)
    kr, vr = (t.repeat_interleave(H // Hkv, dim=2).double() for t in (k, v))
    p = torch.softmax((kr * q.double()).sum(-1) * D ** -0.5, dim=1)                   # [B, KV, H]
    ref = (p.unsqueeze(-1) * vr).sum(1)
    whole, cut = (hb.attn_fwd(q, k, v, family=hb.MA_ATTN_SOFTMAX, causal=False, scale=D ** -0.5, split_kv=s)[:, 0] for s in (False, True))
    assert _error(cut, ref) <= ROOM * _error(whole, ref)


@pytest.mark.parametrize("B,Hq,KV", [(129, 16, 300), (160, 128, 200)])
def test_latent_cache_batch(B, Hq, KV):
    from metaattention_amd import hip_backend as hb
    q, q_pe, kv, k_pe = (_rand(*s, dtype=torch.bfloat16) for s in ((B, 1, Hq, 512), (B, 1, Hq, 64), (B, KV, 1, 512), (B, KV, 1, 64)))
    s = torch.matmul(q[:, 0].double(), kv[:, :, 0].double().transpose(1, 2).contiguous()) + torch.matmul(q_pe[:, 0].double(), k_pe[:, :, 0].double().transpose(1, 2).contiguous())
    ref = torch.matmul(torch.softmax(s * 576 ** -0.5, dim=-1), kv[:, :, 0].double())
    whole, cut = (hb.mla_decode(q, q_pe, kv, k_pe, scale=576 ** -0.5, num_split=n)[:, 0] for n in (1, 0))
    assert _error(cut, ref) <= ROOM * _error(whole, ref)

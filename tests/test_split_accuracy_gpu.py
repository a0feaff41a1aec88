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


def _paged(dtype, Hq, lens):
    """A paged batch through the C ABI: (parameters, tensors to keep, output in 64 bits, the plan)."""
    from metaattention_amd import hip_backend as hb
    B, page = len(lens), 64
    per_seq = -(-max(lens) // page)
    q, pool = _rand(B, 1, Hq, 576, dtype=dtype), _rand(B * per_seq, page, 1, 576, dtype=dtype)
    table = torch.randperm(B * per_seq, generator=torch.Generator().manual_seed(B)).to(torch.int32).cuda().view(B, per_seq)
    seqlens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    ref = torch.zeros(B, Hq, 512, dtype=torch.float64, device="cuda")
    for b, n in enumerate(lens):
        kv = pool[table[b].long()].reshape(-1, 576)[:n].double()
        if n:
            ref[b] = torch.softmax(q[b, 0].double() @ kv.T * 576 ** -0.5, dim=-1) @ kv[:, :512]
    p = hb.MlaParams()
    p.dtype, p.batch, p.heads_q, p.seqlen_kv, p.dim, p.dim_pe = hb._dtype_code(dtype), B, Hq, per_seq * page, 512, 64
    p.q, p.q_stride_b, p.q_stride_h = q.data_ptr(), Hq * 576, 576
    p.q_pe, p.qpe_stride_b, p.qpe_stride_h = q.data_ptr() + 1024, Hq * 576, 576
    p.kv, p.kv_stride_s, p.k_pe, p.kpe_stride_s = pool.data_ptr(), 576, pool.data_ptr() + 1024, 576
    p.scale, p.kv_seqlens, p.block_table, p.block_table_stride, p.page_size = 576 ** -0.5, seqlens.data_ptr(), table.data_ptr(), per_seq, page
    p.o_stride_b, p.o_stride_h = Hq * 512, 512
    return p, (q, pool, table, seqlens), ref, hb.get_mla_metadata(seqlens, Hq, 1)


def _run(p, dtype, plan, parts, size):
    """plan None: unsplit.  size: bytes of workspace (None: what is asked for, "array": the built-in one)."""
    import ctypes
    from metaattention_amd import hip_backend as hb
    lib = hb.load_library()
    out, lse = torch.full((p.batch, p.heads_q, 512), float("nan"), dtype=dtype, device="cuda"), torch.full((p.batch, p.heads_q), float("nan"), device="cuda")
    p.o, p.lse, p.num_split = out.data_ptr(), lse.data_ptr(), 0 if plan else 1
    p.tile_scheduler_metadata, p.num_splits, p.num_sm_parts = (plan[0].data_ptr(), plan[1].data_ptr(), parts) if plan else (None, None, 0)
    if size == "array":
        hb._check(lib.ma_mla_decode_noalloc(ctypes.byref(p), None))
        torch.cuda.synchronize()
        return out, lse
    size = lib.ma_mla_workspace_bytes(ctypes.byref(p)) if size is None else size
    ws = torch.full((size + 256,), 255, dtype=torch.uint8, device="cuda")      # (all NaN; what lies behind the workspace stays as it is)
    p.workspace, p.workspace_bytes = ws.data_ptr(), size
    hb._check(lib.ma_mla_decode(ctypes.byref(p), None))
    torch.cuda.synchronize()
    assert (ws[size:] == 255).all()
    return out, lse


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,lens", [(16, [300]), (32, [20 + 20 * i for i in range(16)]), (64, [300 - 4 * i for i in range(64)]), (128, [150] * 40), (40, [320, 1, 0, 200, 33])])
def test_latent_cache_entries_that_the_plan_leaves_whole(dtype, Hq, lens):
    """With a workspace as asked for (fp32 partial results), and with ones that hold the plan's own parts (no cuts, or fewer parts)."""
    B = len(lens)
    p, keep, ref, plan = _paged(dtype, Hq, lens)
    parts, splits = plan[0].shape[0], plan[1]
    assert int((splits[1:] - splits[:-1]).max()) == 1
    one, lse_one = _run(p, dtype, None, 0, 0)
    slot = Hq * (2 * 512 + 4)
    for n, size in ((parts, None), (parts, (B + parts) * slot), (7, (B + 7) * slot), (1, (B + 1) * slot), (parts, "array")):
        out, lse = _run(p, dtype, plan, n, size)
        assert _error(out, ref) <= ROOM * _error(one, ref), (n, size)
        torch.testing.assert_close(lse, lse_one, rtol=1e-5, atol=1e-5)
        empty = [b for b, n in enumerate(lens) if n == 0]
        assert torch.count_nonzero(out[empty]) == 0 and (lse[empty] == float("-inf")).all()


@pytest.mark.parametrize("Hq,lens", [(128, [64 + 250 * i for i in range(16)]), (32, [3000, 5, 0, 700, 64, 2049, 130, 31] * 3), (64, [4000] + [90] * 50), (200, [1500, 100, 900, 320])])
def test_latent_cache_plan_of_mixed_lengths(Hq, lens):
    """Entries that the plan cuts beside entries that it leaves whole, in every kind of workspace: the former may round their partial
    results (at most the square root of two of the unsplit error), the latter not."""
    dtype, B = torch.bfloat16, len(lens)
    p, keep, ref, plan = _paged(dtype, Hq, lens)
    parts, pieces = plan[0].shape[0], plan[1][1:] - plan[1][:-1]
    whole = (pieces == 1).cpu() & torch.tensor([n > 0 for n in lens])
    assert whole.any() and (pieces > 1).any()
    one, lse_one = _run(p, dtype, None, 0, 0)
    slot = Hq * (2 * 512 + 4)
    for n, size in ((parts, None), (parts, (B + parts) * slot), (16, (B + 16) * slot), (min(parts, 256), "array")):
        out, lse = _run(p, dtype, plan, n, size)
        assert _error(out[whole], ref[whole]) <= ROOM * _error(one[whole], ref[whole]), (n, size)
        assert _error(out, ref) <= 2 ** 0.5 * ROOM * _error(one, ref), (n, size)
        torch.testing.assert_close(lse, lse_one, rtol=1e-5, atol=1e-5)

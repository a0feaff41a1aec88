"""The pipelined chunk loop of the linear scan (tiles two or three chunks ahead, P^T one chunk ahead, scalars two): sequence lengths
around its start and its end, with each workgroup layout (eight state waves; four with four helpers; two heads with four helpers)
and each form of operand addressing, and what a chunk must not let through from later tokens.

Outputs are compared chunk by chunk in the 2-norm: P^T, the state as an operand and the output are rounded to bf16 (2^-9 each, at
most), fp32 sums add nothing that shows, so a chunk's relative error stays below 3 * 2^-9 = 5.9e-3 but for what cancels in it; a
wrong tile, chunk or factor is of the order of 1."""
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu
BOUND = 1e-2
# B, Hq, H, Dk, Dv: <256, 8>, <128, 8>, <256, 4>, <128, 4>, two heads of <128, 2>, key widths that are padded
LAYOUTS = [(1, 2, 2, 256, 256), (1, 1, 2, 128, 256), (1, 2, 2, 256, 128), (2, 1, 1, 128, 128), (1, 1, 4, 128, 64), (1, 2, 2, 192, 256), (1, 2, 2, 64, 128)]


def _hb():
    from metaattention_amd import hip_backend as hb
    hb.load_library()
    return hb


def _case(B, Hq, H, T, Dk, Dv, scaled, seed):
    g = torch.Generator().manual_seed(seed)
    q, k = (torch.randn(B, Hq, T, Dk, generator=g).mul(Dk ** -0.25).bfloat16() for _ in range(2))
    v = torch.randn(B, H, T, Dv, generator=g).bfloat16()
    ld = torch.nn.functional.logsigmoid(torch.randn(B, H, T, generator=g) + 2.0)
    vs = torch.rand(B, H, T, generator=g) + 0.1 if scaled else None
    return q, k, v, ld, vs


def _reference(q, k, v, ld, vs, chunk):
    pad = -q.shape[2] % chunk
    p = lambda t: torch.nn.functional.pad(t, (0, 0, 0, pad) if t.dim() == 4 else (0, pad))   # noqa: E731
    o = oracle.linear_attention_chunked(p(q), p(k), p(v), p(ld), chunk=chunk, v_scale=None if vs is None else p(vs), compute_dtype=torch.float64)
    return o[:, :, :q.shape[2]]


@pytest.mark.parametrize("T", [1, 31, 32, 33, 64, 65, 96, 97, 128, 161])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_lengths_around_the_pipeline(layout, T):
    hb = _hb()
    B, Hq, H, Dk, Dv = layout
    q, k, v, ld, vs = _case(B, Hq, H, T, Dk, Dv, T % 2 == 1, T)
    print(f"pipeline {layout} T{T}", flush=True)
    ref = _reference(q, k, v, ld, vs, 32)
    for segments in (1, 3):
        o = hb.linear_fwd(q.cuda(), k.cuda(), v.cuda(), ld.cuda(), v_scale=None if vs is None else vs.cuda(), segments=segments)
        torch.cuda.synchronize()
        err = (o.double().cpu() - ref).pow(2)
        for t in range(0, T, 32):
            rel = (err[:, :, t:t + 32].sum(dim=(2, 3)) / ref[:, :, t:t + 32].pow(2).sum(dim=(2, 3))).sqrt()
            assert rel.max() < BOUND, (segments, t, rel)


@pytest.mark.parametrize("T", [33, 96, 130])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_gradients_around_the_pipeline(layout, T):
    """The scans on reversed operands, column slices and shared heads, fp32 outputs among them."""
    hb = _hb()
    B, Hq, H, Dk, Dv = layout
    q, k, v, ld, vs = _case(B, Hq, H, T, Dk, Dv, Hq != H, T + 1)
    dout = torch.randn(B, H, T, Dv, generator=torch.Generator().manual_seed(T)).bfloat16()
    print(f"pipeline gradients {layout} T{T}", flush=True)
    ref = oracle.linear_attention_grads(q, k, v, ld, dout, v_scale=vs)
    out = hb.linear_bwd(q.cuda(), k.cuda(), v.cuda(), ld.cuda(), dout.cuda(), v_scale=None if vs is None else vs.cuda())
    torch.cuda.synchronize()
    for name, x, r in zip(("dq", "dk", "dv"), out[:3], ref[:3]):
        err = (x.double().cpu() - r).norm() / r.norm()
        assert err < BOUND, (name, float(err))


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_later_keys_and_decays_stay_out(layout, bad):
    """A key, a decay or a value scale that is not finite changes nothing before its own token, inside its chunk too."""
    hb = _hb()
    B, Hq, H, Dk, Dv = layout
    T, at = 96, 45
    q, k, v, ld, vs = _case(B, Hq, H, T, Dk, Dv, True, 7)
    good = hb.linear_fwd(q.cuda(), k.cuda(), v.cuda(), ld.cuda(), v_scale=vs.cuda(), segments=1)
    for which in ("k", "ld", "vs"):
        k2, ld2, vs2 = k.clone(), ld.clone(), vs.clone()
        {"k": k2, "ld": ld2, "vs": vs2}[which][:, :, at] = bad
        print(f"later {which} = {bad} {layout}", flush=True)
        o = hb.linear_fwd(q.cuda(), k2.cuda(), v.cuda(), ld2.cuda(), v_scale=vs2.cuda(), segments=1)
        torch.cuda.synchronize()
        assert torch.equal(o[:, :, :at], good[:, :, :at]), which


@pytest.mark.parametrize("T", [1, 33, 96, 130])
@pytest.mark.parametrize("B,Hq,H,Dk,Dv,scaled", [
    (1, 2, 2, 256, 256, False), (2, 2, 2, 128, 128, False), (1, 2, 2, 64, 64, False), (1, 2, 2, 192, 256, False),   # one piece: the scans write dq and dk
    (8, 16, 16, 256, 512, False), (3, 43, 43, 256, 512, False), (4, 32, 32, 128, 512, False), (8, 16, 16, 256, 768, False),                       # equal pieces in turn
    (1, 2, 2, 256, 512, False), (8, 16, 16, 192, 512, False), (1, 2, 2, 256, 320, False),                           # pieces side by side, unequal pieces
    (2, 1, 4, 128, 64, True), (1, 2, 2, 256, 512, True),                                                            # shared heads, a value scale
])
def test_gradients_without_the_decays(B, Hq, H, Dk, Dv, scaled, T):
    """dq, dk, dv of the call that leaves the decay's gradient out: the same fp32 sums, each rounded to bf16 once, in two arrangements
    (2^-9 each against the other's value where a sum falls on the other side of a rounding edge)."""
    hb = _hb()
    q, k, v, ld, vs = _case(B, Hq, H, T, Dk, Dv, scaled, T + 3)
    dout = torch.randn(B, H, T, Dv, generator=torch.Generator().manual_seed(T)).bfloat16()
    args = [t.cuda() for t in (q, k, v, ld, dout)]
    kw = dict(v_scale=None if vs is None else vs.cuda())
    print(f"gradients without the decay's B{B} H{Hq}/{H} T{T} {Dk}/{Dv}", flush=True)
    full, some = hb.linear_bwd(*args, **kw), hb.linear_bwd(*args, **kw, with_decay=False)
    torch.cuda.synchronize()
    assert some[3] is None and some[4] is None
    for name, x, y in zip(("dq", "dk", "dv"), some[:3], full[:3]):
        x, y = x.double(), y.double()
        assert torch.isfinite(x).all() and (x - y).norm() <= 2 ** -8 * y.norm(), name


@pytest.mark.parametrize("B,Hq,H,T,Dk,Dv", [(1, 1, 4, 300, 128, 64), (2, 2, 2, 200, 256, 512), (8, 1, 64, 256, 128, 64), (1, 2, 2, 100, 64, 128)])
def test_backward_workspace_is_a_matter_of_sizes(B, Hq, H, T, Dk, Dv):
    """What the query says of sizes alone serves a call with a value scale and one without, with the decay's gradient and without."""
    import ctypes
    hb = _hb()
    lib, p = hb.load_library(), hb.LinearBwdParams()
    p.dtype, p.batch, p.heads, p.heads_q, p.heads_k, p.seqlen, p.dim_k, p.dim_v = hb.MA_BF16, B, H, Hq, Hq, T, Dk, Dv
    q, k, v, ld, vs = (t.cuda() for t in _case(B, Hq, H, T, Dk, Dv, True, T))
    for query, with_decay in ((lib.ma_linear_bwd_workspace_bytes, True), (lib.ma_linear_bwd_qkv_workspace_bytes, False)):
        ws = torch.empty(query(ctypes.byref(p)), dtype=torch.uint8, device="cuda")
        for scale in (None, vs):
            got = hb.linear_bwd(q, k, v, ld, torch.ones_like(v), v_scale=scale, workspace=ws, with_decay=with_decay)
            want = hb.linear_bwd(q, k, v, ld, torch.ones_like(v), v_scale=scale, with_decay=with_decay)
            assert all(a is None and b is None or torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("B,Hq,H,T,Dk,Dv", [(1, 1, 4, 300, 128, 64), (8, 16, 16, 256, 256, 512), (1, 2, 2, 100, 64, 128), (2, 4, 4, 200, 128, 128)])
@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("with_decay", [False, True])
def test_backward_call_takes_what_its_query_says(B, Hq, H, T, Dk, Dv, scaled, with_decay):
    """The query for a call as it is: never more than the one that goes by the sizes, enough for the call, and not a byte too much."""
    import ctypes
    hb = _hb()
    lib, p = hb.load_library(), hb.LinearBwdParams()
    p.dtype, p.batch, p.heads, p.heads_q, p.heads_k, p.seqlen, p.dim_k, p.dim_v = hb.MA_BF16, B, H, Hq, Hq, T, Dk, Dv
    by_sizes = (lib.ma_linear_bwd_workspace_bytes if with_decay else lib.ma_linear_bwd_qkv_workspace_bytes)(ctypes.byref(p))
    q, k, v, ld, vs = (t.cuda() for t in _case(B, Hq, H, T, Dk, Dv, True, T))
    vs = vs if scaled else None
    p.v_scale = p.dv_scale = vs.data_ptr() if scaled else None
    need = lib.ma_linear_bwd_call_workspace_bytes(ctypes.byref(p), int(with_decay))
    assert 0 < need <= by_sizes
    run = lambda n: hb.linear_bwd(q, k, v, ld, torch.ones_like(v), v_scale=vs, with_decay=with_decay, workspace=torch.empty(n, dtype=torch.uint8, device="cuda"))
    for a, b in zip(run(need), run(by_sizes)):
        assert a is None and b is None or torch.equal(a, b)
    with pytest.raises(hb.MetaAttentionError, match=str(need)):
        run(need - 1)


def test_backward_without_the_decays_allocates_what_it_uses():
    """An operator's backward pass that nobody asks the decay's gradient of, every head with its own q and k: beside the gradients it
    holds the fp32 sums of dq and dk, and not the copies per half of the value columns and of dv that the decay's gradient would need."""
    from attn_engine import LinearAttentionEngine
    from core import CustomIO, meta_tensor
    B, H, T, Dk, Dv = 8, 16, 512, 256, 512
    meta = [meta_tensor(B, H, T, d, dtype=torch.bfloat16) for d in (Dk, Dk, Dv)]
    mod = LinearAttentionEngine(tuple(meta), decay_mod=lambda decay, io: decay.log(), custom_io=CustomIO({}))
    g = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = (torch.randn(B, H, T, d, device="cuda", generator=g).mul(0.1).bfloat16().requires_grad_() for d in (Dk, Dk, Dv))
    decay = torch.rand(B, H, T, device="cuda", generator=g)
    grad = torch.ones(B, H, T, Dv, device="cuda", dtype=torch.bfloat16)
    torch.autograd.grad(mod(q, k, v, decay), (q, k, v), grad)
    out = mod(q, k, v, decay)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    grads = torch.autograd.grad(out, (q, k, v), grad)
    used = torch.cuda.max_memory_allocated() - before - sum(t.numel() * 2 for t in grads)
    assert used <= 2 * B * H * T * Dk * 4 + 4 * B * H * T * 4 + (4 << 20)      # dq and dk, values a token, what the allocator rounds up

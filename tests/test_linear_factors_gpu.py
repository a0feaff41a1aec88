"""The decay's logarithm, a head's factor of the decay and a bf16 value scale taken by the linear scan itself (ma_linear_fwd_factors)
against the scan of what they amount to: same fp32 factors, so the same output but for a fused product in the running sum of the
decays.  Lengths of a partial chunk and of several, single pass and segments, each workgroup layout."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 33, 200, 2048])
@pytest.mark.parametrize("B,Hq,H,Dk,Dv", [(1, 2, 2, 256, 256), (1, 2, 2, 256, 128), (2, 1, 3, 128, 128), (1, 1, 4, 128, 64)])
@pytest.mark.parametrize("log,head,half", [(True, False, False), (False, True, True), (True, True, False), (False, False, True)])
def test_factors(T, B, Hq, H, Dk, Dv, log, head, half):
    from metaattention_amd import hip_backend as hb
    lib, g = hb.load_library(), torch.Generator().manual_seed(T + Dk)
    q, k = (torch.randn(B, Hq, T, Dk, generator=g).mul(Dk ** -0.5).bfloat16().cuda() for _ in range(2))
    v = torch.randn(B, H, T, Dv, generator=g).bfloat16().cuda()
    decay = torch.rand(B, H, T, generator=g).cuda() * (1.0 if log else -0.3)
    factor = (torch.rand(H, generator=g) + 0.5).cuda()
    vs = (torch.rand(B, H, T, generator=g) + 0.1).cuda()
    vs = vs.bfloat16() if half else vs
    plain = decay.log() if log else decay
    plain = plain * factor.view(1, H, 1) if head else plain
    for segments in (1, 4):
        want = hb.linear_fwd(q, k, v, plain, v_scale=vs.float(), segments=segments, out_fp32=True)
        out = torch.full_like(want, float("nan"))
        p = hb.LinearParams()
        p.dtype, p.out_fp32, p.segments, p.q_scale = hb.MA_BF16, 1, segments, 1.0
        p.batch, p.heads, p.heads_q, p.heads_k, p.seqlen, p.dim_k, p.dim_v = B, H, Hq, Hq, T, Dk, Dv
        p.q, p.k, p.v, p.o, p.log_decay, p.v_scale = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), decay.data_ptr(), vs.data_ptr()
        ws = torch.empty(max(lib.ma_linear_workspace_bytes(ctypes.byref(p)), 1), dtype=torch.uint8, device="cuda")
        p.workspace, p.workspace_bytes = ws.data_ptr(), ws.numel()
        print(f"factors T{T} {(B, Hq, H, Dk, Dv)} log={log} head={head} half={half} segments={segments}", flush=True)
        assert lib.ma_linear_fwd_factors(ctypes.byref(p), int(log), factor.data_ptr() if head else None, hb.MA_BF16 if half else -1,
                                         torch.cuda.current_stream().cuda_stream) == 0, lib.ma_last_error()
        # the running sums differ by 2^-24 of at most 32 decays each (|log| < 20): 4e-5 of a factor; where that moves a rounding to
        # bf16 of an operand (2^-9 of it), some of a sum's terms do
        assert (out - want).norm() <= 1e-3 * want.norm()
    # (refused before any launch)
    assert lib.ma_linear_fwd_factors(ctypes.byref(p), 0, None, hb.MA_FP16, None) < 0
    p.dim_k = 64
    assert lib.ma_linear_fwd_factors(ctypes.byref(p), 1, None, -1, None) < 0


@pytest.mark.parametrize("T,Hq,H,Dk,Dv,segments", [(40, 2, 2, 256, 256, 1), (200, 1, 4, 128, 64, 3), (33, 2, 2, 256, 64, 1), (300, 1, 3, 128, 128, 4)])
@pytest.mark.parametrize("half", [False, True])
def test_no_value_scale(T, Hq, H, Dk, Dv, segments, half):
    """Without a value scale the type that one would have says nothing: the plain call's kernels and numbers, to the bit."""
    from metaattention_amd import hip_backend as hb
    lib, g = hb.load_library(), torch.Generator().manual_seed(T)
    q, k = (torch.randn(1, Hq, T, Dk, generator=g).mul(Dk ** -0.5).bfloat16().cuda() for _ in range(2))
    v = torch.randn(1, H, T, Dv, generator=g).bfloat16().cuda()
    decay = torch.rand(1, H, T, generator=g).cuda() * -0.3
    want = hb.linear_fwd(q, k, v, decay, segments=segments, out_fp32=True)
    out = torch.full_like(want, float("nan"))
    p = hb.LinearParams()
    p.dtype, p.out_fp32, p.segments, p.q_scale = hb.MA_BF16, 1, segments, 1.0
    p.batch, p.heads, p.heads_q, p.heads_k, p.seqlen, p.dim_k, p.dim_v = 1, H, Hq, Hq, T, Dk, Dv
    p.q, p.k, p.v, p.o, p.log_decay = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), decay.data_ptr()
    ws = torch.empty(max(lib.ma_linear_workspace_bytes(ctypes.byref(p)), 1), dtype=torch.uint8, device="cuda")
    p.workspace, p.workspace_bytes = ws.data_ptr(), ws.numel()
    print(f"no value scale T{T} {(Hq, H, Dk, Dv)} half={half} segments={segments}", flush=True)
    assert lib.ma_linear_fwd_factors(ctypes.byref(p), 0, None, hb.MA_BF16 if half else -1, torch.cuda.current_stream().cuda_stream) == 0, lib.ma_last_error()
    assert torch.count_nonzero(want) > 0 and torch.equal(out, want)


@pytest.mark.parametrize("Dk", [128, 64])
def test_engine_with_and_without_gradients(Dk):
    """The same operator through its native call: factors in the kernel, and (with gradients) as tensors in front of it."""
    from attn_engine import LinearAttentionEngine
    from core import CustomIO, meta_tensor
    B, H, T = 2, 4, 300
    g = torch.Generator().manual_seed(1)
    meta = (meta_tensor(B, 1, T, Dk, dtype=torch.bfloat16), meta_tensor(B, 1, T, Dk, dtype=torch.bfloat16), meta_tensor(B, H, T, 64, dtype=torch.bfloat16))
    mod = LinearAttentionEngine(meta, decay_mod=lambda decay, io: decay * io.input_tensors["A"], v_mod=lambda v, io: v * io.input_tensors["dt"],
                                custom_io=CustomIO({"A": (1, "heads"), "dt": ("batch", "heads", "seq_len")}))
    q, k, v = (torch.randn(B, h, T, d, generator=g).mul(0.3).bfloat16().cuda() for h, d in ((1, Dk), (1, Dk), (H, 64)))
    dt = torch.rand(B, H, T, generator=g).cuda()
    A = -torch.rand(1, H, generator=g).cuda()
    for scale in (dt, dt.bfloat16(), dt.half(), dt.bfloat16().transpose(1, 2).contiguous().transpose(1, 2)):
        want = mod(q, k, v, dt, A, scale.detach().requires_grad_()).detach()
        got = mod(q, k, v, dt, A, scale)
        assert not got.requires_grad
        assert (got.float() - want.float()).norm() <= 2e-3 * want.float().norm()       # (a unit of bf16's last place here and there)
    assert torch.equal(mod(q, k, v, dt, A, dt.half()), mod(q, k, v, dt.clone(), A.clone(), dt.half()))


@pytest.mark.parametrize("Dk", [128, 256])
def test_negated_views(Dk):
    """A decay or a value scale whose negation is a bit of the tensor (as the imaginary part of a conjugate has it): its values."""
    from attn_engine import LinearAttentionEngine
    from core import CustomIO, meta_tensor
    B, H, T = 1, 2, 70
    g = torch.Generator().manual_seed(2)
    meta = [meta_tensor(B, H, T, d, dtype=torch.bfloat16) for d in (Dk, Dk, 64)]
    q, k, v = (torch.randn(B, H, T, d, generator=g).mul(0.3).bfloat16().cuda() for d in (Dk, Dk, 64))
    by_log = LinearAttentionEngine(tuple(meta), decay_mod=lambda decay, io: decay.log(), custom_io=CustomIO({}))
    decay = torch.rand(B, H, T, generator=g).cuda()
    assert torch.equal(by_log(q, k, v, torch._neg_view(-decay)), by_log(q, k, v, decay))
    scaled = LinearAttentionEngine(tuple(meta), decay_mod=lambda decay, io: decay * io.input_tensors["A"], v_mod=lambda v, io: v * io.input_tensors["dt"],
                                   custom_io=CustomIO({"A": (1, "heads"), "dt": ("batch", "heads", "seq_len")}))
    A, dt = -torch.rand(1, H, generator=g).cuda(), torch.rand(B, H, T, generator=g).bfloat16().cuda()
    want = scaled(q, k, v, decay, A, dt)
    for args in ((torch._neg_view(-decay), A, dt), (decay, torch._neg_view(-A), dt), (decay, A, torch._neg_view(-dt))):
        assert (scaled(q, k, v, *args).float() - want.float()).norm() <= 2e-3 * want.float().norm()


@pytest.mark.parametrize("Hq,H,Dk,Dv", [(2, 2, 256, 256), (2, 2, 256, 64), (1, 3, 128, 128), (1, 4, 128, 64)])
@pytest.mark.parametrize("segments", [1, 3])
def test_logarithm(Hq, H, Dk, Dv, segments):
    """The decay's logarithm that the kernel takes is the one that torch's log rounds to: the same outputs to the bit, for decays over
    the whole range, close to 1, of 0 and of a subnormal."""
    from metaattention_amd import hip_backend as hb
    lib, g, B, T = hb.load_library(), torch.Generator().manual_seed(Dk + Dv), 2, 333
    q, k = (torch.randn(B, Hq, T, Dk, generator=g).mul(Dk ** -0.5).bfloat16().cuda() for _ in range(2))
    v = torch.randn(B, H, T, Dv, generator=g).bfloat16().cuda()
    u = torch.rand(B, H, T, generator=g)
    some_zero, tiny = u.clone(), u.clone()
    some_zero[:, :, 100] = 0.0
    tiny[:, :, 100::40] = 1e-42
    for decay in (u, 1 - u / 64, 1 + u / 64, some_zero, tiny):
        decay = decay.cuda()
        want = hb.linear_fwd(q, k, v, decay.log(), segments=segments, out_fp32=True)
        out = torch.zeros_like(want)
        p = hb.LinearParams()
        p.dtype, p.out_fp32, p.segments, p.q_scale = hb.MA_BF16, 1, segments, 1.0
        p.batch, p.heads, p.heads_q, p.heads_k, p.seqlen, p.dim_k, p.dim_v = B, H, Hq, Hq, T, Dk, Dv
        p.q, p.k, p.v, p.o, p.log_decay = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), decay.data_ptr()
        ws = torch.empty(max(lib.ma_linear_workspace_bytes(ctypes.byref(p)), 1), dtype=torch.uint8, device="cuda")
        p.workspace, p.workspace_bytes = ws.data_ptr(), ws.numel()
        assert lib.ma_linear_fwd_factors(ctypes.byref(p), 1, None, -1, torch.cuda.current_stream().cuda_stream) == 0, lib.ma_last_error()
        torch.testing.assert_close(out, want, rtol=0, atol=0, equal_nan=True)

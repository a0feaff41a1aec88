"""The operators' native calls (csrc/host_ops.cpp) against the Python binding: the same launches, so the same bits, and the
cases that the native call hands to the binding."""
import pytest
import torch

import specs

pytestmark = pytest.mark.gpu


def _rand(*shape, dtype=torch.bfloat16, gain=1.0):
    return (torch.randn(*shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(sum(shape))) * gain).to(dtype)


def _grads(fn, args):
    leaves = [a.detach().clone().requires_grad_(a.is_floating_point()) for a in args]
    out = fn(*leaves)
    return (out.detach(), *torch.autograd.grad(out, leaves, torch.ones_like(out), allow_unused=True))


def _window(b, h, q, k):
    return (q >= k) & (q - k < 20)


@pytest.mark.parametrize("family,mask,S,Hkv", [("softmax", "causal", 130, 2), ("softmax", "window", 65, 4), ("sigmoid", "causal", 33, 1), ("relu", "none", 1, 4)])
def test_attention_and_its_gradients(family, mask, S, Hkv):
    def make():
        if family == "relu":
            return specs.relu_attention(2, 4, S, 64, 64)
        if family == "sigmoid":
            return specs.sigmoid_attention(2, 4, S, 64, 64, const_bias=-1.0)
        mod = specs.softmax_attention(2, 4, S, 64, 64)
        if mask == "window":
            from attn_engine import AttentionEngine
            from core import CustomIO, meta_tensor
            meta = tuple(meta_tensor(2, 4, S, 64, dtype=torch.bfloat16) for _ in range(3))
            mod = AttentionEngine(meta, CustomIO({}), score_mod=lambda s, io, b, h, q, k: s * 0.125, mask_mod=_window, online_func=specs.OnlineSoftmax())
        return mod
    q, k, v = _rand(2, S, 4, 64), _rand(2, S, Hkv, 64), _rand(2, S, Hkv, 64)
    a, b = make(), make()
    for _ in range(2):        # (a masked operator's first call builds its masks in the binding)
        got, want = _grads(a, (q, k, v)), _grads(b.attention, (q, k, v))
        assert all(torch.equal(x, y) for x, y in zip(got, want))
        assert (a.final_rowscales is None) == (b.final_rowscales is None)
        assert a.final_rowscales is None or torch.equal(a.final_rowscales, b.final_rowscales)
    # a view that the kernels cannot read in place, and another dtype than the operator was declared with: the binding's business
    wide = torch.zeros(2, S, 4, 65, dtype=q.dtype, device="cuda")
    wide[..., :64] = q
    assert torch.equal(a(wide[..., :64], k, v), got[0])
    assert a(q.half(), k.half(), v.half()).dtype == torch.float16
    with pytest.raises(TypeError):
        a(q, k, v, q)


@pytest.mark.parametrize("op,T", [("retnet", 65), ("gated", 1), ("mamba2", 40)])
def test_linear_and_its_gradients(op, T):
    B, H = 2, 4
    Hq = 1 if op == "mamba2" else H
    q, k, v = _rand(B, Hq, T, 128, gain=0.1), _rand(B, Hq, T, 128, gain=0.1), _rand(B, H, T, 64)
    dt = torch.rand(B, H, T, device="cuda") * 0.1 + 0.5
    if op == "mamba2":
        mod, args = specs.mamba2(B, 1, T, 128, 64, HV=H), (q, k, v, dt, -torch.rand(1, H, device="cuda"), dt.bfloat16())
    elif op == "retnet":
        mod, args = specs.retnet_recurrent(B, H, T, 128, 64), (q, k, v, dt)
    else:
        mod, args = specs.gated_retention(B, H, T, 128, 64), (q, k, v, -dt)
    assert torch.equal(mod(*args), mod.attention(*args))
    assert all(torch.equal(x, y) for x, y in zip(_grads(mod, args), _grads(mod.attention, args)))


@pytest.mark.parametrize("Hq,KV", [(128, 300), (5, 33)])
def test_mla_and_decode(Hq, KV):
    from hip_backend import mla_decode
    mod = specs.mla_decode(3, Hq, KV, 576, 512)
    args = (_rand(3, 1, Hq, 512), _rand(3, 1, Hq, 64), _rand(3, KV, 1, 512), _rand(3, KV, 1, 64))
    assert torch.equal(mod(*args), mla_decode(*args, scale=576 ** -0.5))
    dec = specs.softmax_attention_decode(2, 8, 1, KV, 128, 128, HKV=2)
    q, k, v = _rand(2, 1, 8, 128, dtype=torch.float16), _rand(2, KV, 2, 128, dtype=torch.float16), _rand(2, KV, 2, 128, dtype=torch.float16)
    out = dec(q, k, v)
    scales = dec.final_rowscales
    assert torch.equal(out, dec.attention(q, k, v)) and torch.equal(scales, dec.final_rowscales)


def _binding_is_off(monkeypatch):
    import hip_backend

    def refuse(*args, **kwargs):
        raise AssertionError("the binding was called")
    for name in ("attn_fwd", "attn_bwd", "linear_fwd", "linear_bwd", "mla_decode", "_require_gpu"):
        monkeypatch.setattr(hip_backend, name, refuse)


def test_ordinary_calls_are_served_natively(monkeypatch):
    """Forward and, through the native autograd functions, backward of the ordinary calls never reach the Python binding."""
    from hip_backend import flash_mla_with_kvcache, get_mla_metadata
    lens = torch.tensor([100, 64], dtype=torch.int32, device="cuda")
    plan = get_mla_metadata(lens, 16, 1)
    window = specs.softmax_attention(2, 4, 65, 64, 64)
    window.mask_kind, window.mask_mod = "other", _window
    q, k, v = _rand(2, 65, 4, 64), _rand(2, 65, 2, 64), _rand(2, 65, 2, 64)
    want = _grads(window, (q, k, v))                     # (the first call builds the masks, in the binding)
    _binding_is_off(monkeypatch)
    assert all(torch.equal(x, y) for x, y in zip(_grads(window, (q, k, v)), want))
    for mod in (specs.softmax_attention(2, 4, 65, 64, 64), specs.relu_attention(2, 4, 65, 64, 64), specs.sigmoid_attention(2, 4, 65, 64, 64, const_bias=-1.0)):
        _grads(mod, (q, k, v))
    decay = torch.rand(2, 4, 65, device="cuda") * 0.1 + 0.5
    lin = _rand(2, 4, 65, 64, gain=0.1), _rand(2, 4, 65, 64, gain=0.1), _rand(2, 4, 65, 64)
    _grads(specs.retnet_recurrent(2, 4, 65, 64, 64), (*lin, decay))
    _grads(specs.gated_retention(2, 4, 65, 64, 64), (*lin, -decay))
    _grads(specs.mamba2(2, 1, 65, 64, 64, HV=4), (lin[0][:, :1].contiguous(), lin[1][:, :1].contiguous(), lin[2], decay, -torch.rand(1, 4, device="cuda"), decay.bfloat16()))
    specs.softmax_attention_decode(2, 4, 1, 300, 64, 64, dtype=torch.bfloat16, HKV=2)(q[:, :1].contiguous(), _rand(2, 300, 2, 64), _rand(2, 300, 2, 64))
    specs.mla_decode(2, 16, 100, 576, 512)(_rand(2, 1, 16, 512), _rand(2, 1, 16, 64), _rand(2, 100, 1, 512), _rand(2, 100, 1, 64))
    table = torch.arange(4, dtype=torch.int32, device="cuda").view(2, 2)
    for p in ((), plan):
        flash_mla_with_kvcache(_rand(2, 1, 16, 576), _rand(4, 64, 1, 576), table, lens, 512, *p)
    ret = specs.retention_parallel(1, 2, 68, 256, 512)
    ret(_rand(1, 68, 2, 256, gain=0.1), _rand(1, 68, 2, 256, gain=0.1), _rand(1, 68, 2, 512), _rand(1, 2, 68, 68))


def test_what_the_native_call_hands_over_it_does_not_launch():
    """Such calls return None at the checks, before anything is allocated for a launch; the operator then serves them once."""
    mod = specs.softmax_attention(1, 4, 70, 64, 64)
    q, k, v = _rand(1, 70, 4, 64), _rand(1, 70, 4, 64), _rand(1, 70, 4, 64)
    out = mod(q, k, v)
    wide = torch.zeros(1, 70, 4, 65, dtype=q.dtype, device="cuda")[..., :64]
    wide.copy_(q)
    odd = {"unaligned view": (wide, k, v), "another dtype": (q.half(), k.half(), v.half()), "too many": (q, k, v, q), "not on the GPU": (q.cpu(), k, v),
           "a subclass": (torch.Tensor._make_subclass(type("Mine", (torch.Tensor,), {}), q), k, v)}
    for name, args in odd.items():
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        assert mod._native_fn(*args) is None, name
        assert torch.cuda.memory_stats()["allocation.all.allocated"] == before, name
    assert torch.equal(mod(*odd["unaligned view"]), out)

"""Gradients where a mask hides values that are not finite: what a key does not see leaves dk (and, from tiles that none of a wave's
32 keys sees, dv) the bits that it has without them.  In one run of steps and in several, with one item a workgroup and with more."""
import pytest
import torch

pytestmark = pytest.mark.gpu
SIZES = [(128, 128), (192, 128), (128, 256), (256, 256)]
BAD = [float("nan"), float("inf"), float("-inf")]


def _inputs(B, H, Hkv, S, D, DV, dtype=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(S + D + H)
    return [torch.randn(B, S, h, d, device="cuda", generator=g).to(dtype) for h, d in ((H, D), (Hkv, D), (Hkv, DV), (H, DV))]


def backward(family, q, k, v, dout, monkeypatch, one_run, causal=False, seen_v=None, **masks):
    """(dq, dk, dv), with the library's own choice of runs or in one (a call with only the required workspace).  seen_v: V of the forward
    pass, where V holds values in keys that it need not read."""
    from metaattention_amd import hip_backend as hb
    fam = {"softmax": hb.MA_ATTN_SOFTMAX, "sigmoid": hb.MA_ATTN_SIGMOID, "relu": hb.MA_ATTN_RELU}[family]
    B, S, H, D = q.shape
    kw = dict(family=fam, causal=causal, scale=D ** -0.5, bias=-2.0 if family == "sigmoid" else 0.0)
    lse = torch.empty(B, H, S, device="cuda") if family == "softmax" else None
    o = hb.attn_fwd(q, k, v if seen_v is None else seen_v, row_scale=lse, elem_mask=masks.get("elem_mask"), **kw)
    lib = hb.load_library()

    class Lib:
        def __getattr__(self, name):
            return (lambda p: 4 * B * H * S if family == "softmax" else 0) if one_run and name == "ma_attn_bwd_workspace_bytes" else getattr(lib, name)
    with monkeypatch.context() as m:
        m.setattr(hb, "_lib", Lib())
        return hb.attn_bwd(q, k, v, o, dout, lse, **masks, **kw)


def masks_of(allow):
    """The masks of a call in the forms that it takes, from which scores are kept (rows padded to 16 bytes)."""
    S = allow.shape[0]
    n, rows = (S + 127) // 128 * 128, (S + 31) // 32

    def elem(m):
        buf = torch.zeros(S, (S + 15) // 16 * 16, dtype=torch.uint8)
        buf[:, :S] = m
        return buf.cuda().view(1, 1, S, -1)[..., :S]

    def tiles(m):
        kept, whole = torch.zeros(n, n, dtype=torch.bool), torch.ones(n, n, dtype=torch.bool)
        kept[:S, :S], whole[:S, :S] = m, m
        pool = kept.view(n // 128, 128, n // 32, 32).any(3).any(1).to(torch.uint8) * (1 + whole.view(n // 128, 128, n // 32, 32).all(3).all(1).to(torch.uint8))
        return pool[:, :rows].contiguous().cuda().view(1, 1, n // 128, rows)

    return dict(elem_mask=elem(allow), elem_mask_t=elem(allow.t()), kv_block_mask=tiles(allow), q_block_mask=tiles(allow.t()))


@pytest.mark.parametrize("D,DV", SIZES)
@pytest.mark.parametrize("family", ["softmax", "sigmoid", "relu"])
@pytest.mark.parametrize("one_run", [True, False])
def test_later_keys_do_not_see_a_row_under_a_causal_mask(D, DV, family, one_run, monkeypatch):
    """A row of dout: the keys of the 32-key groups behind that of the row."""
    for B, H, Hkv, S, row in ((1, 4, 2, 420, 5), (1, 4, 2, 420, 200), (2, 3, 3, 290, 130), (1, 2, 2, 100, 33)):
        print(f"causal {family} {D}/{DV} B{B} H{H}/{Hkv} S{S} row {row} one_run={one_run}", flush=True)
        q, k, v, dout = _inputs(B, H, Hkv, S, D, DV)
        want = backward(family, q, k, v, dout, monkeypatch, one_run, causal=True)
        for bad in BAD:
            grad = dout.clone()
            grad[0, row, 1] = bad
            got = backward(family, q, k, v, grad, monkeypatch, one_run, causal=True)
            behind = row // 32 * 32 + 32
            for name, a, b in zip(("dk", "dv"), got[1:], want[1:]):
                assert torch.equal(a[:, behind:], b[:, behind:]) and torch.equal(a[1:], b[1:]), f"{name} {bad}"
            assert not got[2][0, :row, 1 * Hkv // H].isfinite().any(), "the keys that see the row have it"


@pytest.mark.parametrize("D,DV", [(64, 64)] + SIZES)
@pytest.mark.parametrize("family", ["softmax", "sigmoid", "relu"])
@pytest.mark.parametrize("one_run", [True, False])
@pytest.mark.parametrize("B,H,Hkv,S", [(1, 4, 2, 320), (2, 3, 3, 300), (8, 16, 16, 384), (3, 43, 43, 300)])     # (the last two: more items than workgroups)
def test_hidden_keys_and_rows_under_a_mask(B, H, Hkv, S, D, DV, family, one_run, monkeypatch):
    """V of 32 padding keys that no row sees, and the gradient of five rows that see no key, in a tile whose other rows do (not at 64 / 64,
    whose one wave has a row's delta only behind the mask)."""
    print(f"mask {family} {D}/{DV} B{B} H{H}/{Hkv} S{S} one_run={one_run}", flush=True)
    q, k, v, dout = _inputs(B, H, Hkv, S, D, DV)
    i, j = torch.arange(S).view(S, 1), torch.arange(S).view(1, S)
    keys, rows = slice(96, 128), slice(40, 45)
    allow = (j <= i + 7) & (i - j < 150)
    allow[:, keys] = False
    allow[rows] = False
    m = masks_of(allow)
    want = backward(family, q, k, v, dout, monkeypatch, one_run, **m)
    assert all(t.isfinite().all() for t in want) and not want[1][:, keys].any() and not want[2][:, keys].any()
    for bad in BAD:
        other = v.clone()
        other[:, keys] = bad
        for name, a, b in zip(("dq", "dk", "dv"), backward(family, q, k, other, dout, monkeypatch, one_run, seen_v=v, **m), want):
            assert torch.equal(a, b), f"{name}, V {bad}"
        if D == 64:
            continue
        grad = dout.clone()
        grad[:, rows] = bad
        got = backward(family, q, k, v, grad, monkeypatch, one_run, **m)
        assert torch.equal(got[1], want[1]), f"dk, dout {bad}"


@pytest.mark.parametrize("D,DV", SIZES)
@pytest.mark.parametrize("one_run", [True, False])
# (but for the last: more key blocks than CUs, in 1.5 to 2 rounds, in 3 and almost 4 full ones and in 2.25)
@pytest.mark.parametrize("B,H,Hkv,S", [(8, 16, 16, 400), (3, 34, 34, 400), (8, 32, 16, 300), (8, 32, 32, 384), (5, 51, 51, 400), (9, 16, 16, 400), (1, 4, 2, 400)])
def test_masked_gradients(B, H, Hkv, S, D, DV, one_run, monkeypatch):
    """A workgroup's key blocks one after the other, a list of steps made for each: a window, and a key block that no row sees."""
    print(f"masked {D}/{DV} B{B} H{H}/{Hkv} S{S} one_run={one_run}", flush=True)
    q, k, v, dout = _inputs(B, H, Hkv, S, D, DV)
    i, j = torch.arange(S).view(S, 1), torch.arange(S).view(1, S)
    allow = (j <= i) & (i - j < 170) & ((j < 128) | (j >= 256)) & (i >= 20)
    got = backward("softmax", q, k, v, dout, monkeypatch, one_run, **masks_of(allow))
    hidden = ~allow.cuda()
    for b in range(B):      # (an entry at a time: double precision)
        qd, kd, vd = (t[b].double().transpose(0, 1).contiguous().requires_grad_() for t in (q, k, v))
        ke, ve = (t.repeat_interleave(H // Hkv, 0) for t in (kd, vd))
        x = torch.matmul(qd, ke.transpose(1, 2)) * D ** -0.5
        p = torch.softmax(x.masked_fill(hidden, -1e300), -1) * ~hidden
        ref = torch.autograd.grad(torch.matmul(p, ve), (qd, kd, vd), dout[b].double().transpose(0, 1))
        for name, a, want in zip(("dq", "dk", "dv"), got, ref):
            # p and ds are rounded to bf16 (2^-9 of each, at random): of the 2-norm of a gradient that is well below 1e-2
            assert (a[b].double().transpose(0, 1) - want).norm() <= 1e-2 * want.norm(), f"{name} {b}"
    assert not got[1][:, 128:256].any() and not got[2][:, 128:256].any()


def test_a_triangular_mask_gives_a_causal_calls_bits_at_256(monkeypatch):
    """Several runs of steps: the same tiles and masked elements by the masked and the causal form of the kernel."""
    B, H, Hkv, S = 1, 4, 2, 257
    q, k, v, dout = _inputs(B, H, Hkv, S, 256, 256)
    want = backward("softmax", q, k, v, dout, monkeypatch, False, causal=True)
    elem = {n: m for n, m in masks_of(torch.ones(S, S, dtype=torch.bool).tril()).items() if n.startswith("elem")}
    for name, a, b in zip(("dq", "dk", "dv"), backward("softmax", q, k, v, dout, monkeypatch, False, **elem), want):
        assert torch.equal(a, b), name

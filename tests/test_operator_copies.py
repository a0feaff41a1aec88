"""Operators can be pickled and copied whether or not they have been called, and a copy has native callables and masks of its own."""
import copy
import pickle

import pytest
import torch

import specs
from attn_engine import AttentionEngine
from core import CustomIO, meta_tensor

DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _window(b, h, q, k):
    return (q >= k) & (q - k < 20)


def _score(s, io, b, h, q, k):
    return s * 0.125


def _make(which):
    if which == "window":
        return AttentionEngine(tuple(meta_tensor(1, 2, 72, 64, dtype=torch.bfloat16) for _ in range(3)), CustomIO({}), score_mod=_score, mask_mod=_window,
                               online_func=specs.OnlineSoftmax())
    return {"softmax": lambda: specs.softmax_attention(1, 2, 72, 64, 64), "gated": lambda: specs.gated_retention(1, 2, 72, 64, 64),
            "mla": lambda: specs.mla_decode(1, 16, 72, 576, 512), "retention": lambda: specs.retention_parallel(1, 2, 72, 256, 512)}[which]()


def _args(which, S=72, seed=0):
    g = torch.Generator().manual_seed(seed)
    shapes = {"gated": [(1, 2, S, 64)] * 3, "mla": [(1, 1, 16, 512), (1, 1, 16, 64), (1, S, 1, 512), (1, S, 1, 64)],
              "retention": [(1, S, 2, 256), (1, S, 2, 256), (1, S, 2, 512), (1, 2, S, S)]}.get(which, [(1, S, 2, 64)] * 3)
    args = [torch.randn(*s, generator=g).bfloat16().to(DEV) for s in shapes]
    return args + [-torch.rand(1, 2, S, generator=g).to(DEV)] if which == "gated" else args


def _call(mod, args):
    from hip_backend import MetaAttentionError
    if DEV == "cuda":
        return mod(*args)
    with pytest.raises(MetaAttentionError):         # (no GPU: as far as the binding's check of the tensors)
        mod(*args)


OPERATORS = ["softmax", "window", "gated", "mla", "retention"]


def _copies(mod):
    made = [copy.copy(mod), copy.deepcopy(mod)]
    try:
        made.append(pickle.loads(pickle.dumps(mod)))
    except (AttributeError, pickle.PicklingError) as e:      # (a spec with functions that pickle cannot name)
        assert "local object" in str(e) or "lambda" in str(e), e
    return made


@pytest.mark.parametrize("which", OPERATORS)
def test_copies_do_not_share_native_callables(which):
    mod, args = _make(which), _args(which)
    _call(mod, args)
    if which in ("window", "softmax"):
        pickle.dumps(mod.__getstate__() | {"mask_mod": None, "custom_fwd_inputs": None})      # (whatever the spec's functions are)
    for c in _copies(mod):
        assert c._native_fn is None and getattr(c, "_native_mla", None) is None
        _call(c, args)


def test_pickle_after_a_call():
    mod, args = _make("window"), _args("window")
    _call(mod, args)
    again = pickle.loads(pickle.dumps(mod))
    _call(again, args)


@pytest.mark.gpu
@pytest.mark.parametrize("which", OPERATORS)
def test_copies_compute_the_same(which):
    mod, args = _make(which), _args(which)
    mod(*args)
    out = mod(*args)
    for c in _copies(mod):
        assert torch.equal(c(*args), out)
        if which != "mla":
            assert c._native_fn(*(args if which != "retention" else args[:4])) is not None      # (served, with the masks it was copied with)
        shorter = _args(which, S=40, seed=1)
        want = mod.attention(*shorter)
        assert torch.equal(c(*shorter), want)
        assert torch.equal(mod(*args), out)

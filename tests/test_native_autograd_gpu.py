"""What goes round or through autograd beside plain reverse mode, at the operators' native calls: forward mode, functorch's
transforms, compiled autograd, saved-tensor hooks, tracing."""
import pytest
import torch

import specs
from attn_engine import AttentionEngine
from core import CustomIO, meta_tensor

pytestmark = pytest.mark.gpu


def _rand(*shape):
    return torch.randn(*shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(sum(shape))).bfloat16()


def _operators():
    """(operator, inputs, which of them get gradients): attention with and without a row scale and a dense mask, a scan."""
    q, k, v = _rand(1, 70, 4, 64), _rand(1, 70, 2, 64), _rand(1, 70, 2, 64)
    scan = (_rand(1, 4, 70, 64), _rand(1, 4, 70, 64), _rand(1, 4, 70, 64), -torch.rand(1, 4, 70, device="cuda"))
    return {"softmax": (specs.softmax_attention(1, 4, 70, 64, 64), (q, k, v)), "relu": (specs.relu_attention(1, 4, 70, 64, 64), (q, k, v)),
            "gated": (specs.gated_retention(1, 4, 70, 64, 64), scan)}


OPERATORS = ["softmax", "relu", "gated"]


@pytest.mark.parametrize("which", OPERATORS)
def test_forward_mode_is_refused(which):
    """There are no tangents: an output without one would say that the derivative is zero."""
    import torch.autograd.forward_ad as fwd
    mod, args = _operators()[which]
    for i in range(len(args)):
        with fwd.dual_level():
            dual = [fwd.make_dual(a.clone().requires_grad_(True), torch.ones_like(a)) if j == i else a for j, a in enumerate(args)]
            with pytest.raises(NotImplementedError, match="jvp"):
                mod(*dual)


@pytest.mark.parametrize("which", OPERATORS)
def test_functorch_transforms_are_refused(which):
    mod, args = _operators()[which]
    mod(*args)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda x: mod(x, *args[1:]))(torch.stack([args[0], args[0]]))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: mod(x, *args[1:]).float().sum())(args[0])
    with pytest.raises((RuntimeError, NotImplementedError)):
        torch.func.jvp(lambda x: mod(x, *args[1:]), (args[0],), (torch.ones_like(args[0]),))


def _leaves(args):
    return [a.detach().clone().requires_grad_(True) for a in args]


def _grads(mod, args):
    leaves = _leaves(args)
    out = mod(*leaves)
    out.backward(torch.ones_like(out))
    return [out.detach()] + [x.grad for x in leaves]


@pytest.mark.parametrize("which", OPERATORS + ["window"])
def test_compiled_autograd(which):
    from torch._dynamo import compiled_autograd
    if which == "window":
        mod = AttentionEngine(tuple(meta_tensor(1, 4, 70, 64, dtype=torch.bfloat16) for _ in range(3)), CustomIO({}),
                              score_mod=lambda s, io, b, h, q, k: s * 0.125, mask_mod=lambda b, h, q, k: (q >= k) & (q - k < 20),
                              online_func=specs.OnlineSoftmax())
        args = tuple(_rand(1, 70, 4, 64) for _ in range(3))
    else:
        mod, args = _operators()[which]
    want = _grads(mod, args)
    want = _grads(mod, args)                    # (a masked operator's first call builds its masks in the binding)
    for _ in range(2):
        with compiled_autograd._enable(lambda gm: gm):
            got = _grads(mod, args)
        assert all(torch.equal(x, y) for x, y in zip(got, want))


@pytest.mark.parametrize("which", OPERATORS)
def test_saved_tensor_hooks(which):
    """What the backward needs goes through the hooks, and through nothing else: the inputs, the output, the row scale."""
    mod, args = _operators()[which]
    want, packed = _grads(mod, args), []

    def pack(t):
        packed.append(t.shape)
        return t.cpu()
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        got = _grads(mod, args)
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    assert len(packed) == {"softmax": 5, "relu": 4, "gated": 4}[which]


@pytest.mark.parametrize("which", OPERATORS)
def test_backward_twice_and_inputs_changed_in_between(which):
    mod, args = _operators()[which]
    leaves = _leaves(args)
    out = mod(*leaves)
    first = torch.autograd.grad(out, leaves, torch.ones_like(out), retain_graph=True)
    again = torch.autograd.grad(out, leaves, torch.ones_like(out))
    assert all(torch.equal(x, y) for x, y in zip(first, again))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, leaves, torch.ones_like(out))
    leaves = _leaves(args)
    scaled = [x * 1 for x in leaves]
    out = mod(*scaled)
    scaled[2].mul_(2)
    with pytest.raises(RuntimeError, match="inplace operation"):
        out.sum().backward()


@pytest.mark.parametrize("which", OPERATORS)
@pytest.mark.filterwarnings("ignore")
def test_trace(which):
    """A trace made with inputs that get gradients runs the operator, on other inputs than those it was made with as well."""
    mod, args = _operators()[which]
    mod(*args)
    traced = torch.jit.trace(lambda *a: mod(*a) + 0, tuple(_leaves(args)), check_trace=False)
    other = _leaves([a.flip(0, 1) for a in args])
    assert torch.equal(traced(*other), mod(*other))
    assert all(torch.equal(x, y) for x, y in zip(_grads(traced, other), _grads(mod, other)))


@pytest.mark.parametrize("which", OPERATORS)
def test_checkpointing_leaves_nothing_behind(which):
    """A recomputation ends in the middle of saving, by an exception: what was computed is freed with the graph all the same."""
    from torch.utils.checkpoint import checkpoint
    mod, args = _operators()[which]
    leaves = _leaves(args)

    def step():
        out = checkpoint(mod, *leaves, use_reentrant=False)
        return torch.autograd.grad(out, leaves, torch.ones_like(out))
    want = torch.autograd.grad(mod(*leaves), leaves, torch.ones_like(args[0]))
    assert all(torch.equal(x, y) for x, y in zip(step(), want))
    before = torch.cuda.memory_allocated()
    for _ in range(3):
        step()
    assert torch.cuda.memory_allocated() == before
    edge = torch.autograd.graph.get_gradient_edge(leaves[0]).node      # (made anew when no graph holds it)
    assert "seen" not in edge.metadata
    edge.metadata["seen"] = True
    del edge
    assert "seen" not in torch.autograd.graph.get_gradient_edge(leaves[0]).node.metadata


@pytest.mark.parametrize("which", OPERATORS)
def test_training_pass_in_a_graph(which):
    mod, args = _operators()[which]
    leaves, dout = _leaves(args), torch.ones_like(args[0])

    def step():
        return torch.autograd.grad(mod(*leaves), leaves, dout)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step()
    for seed in range(3):
        with torch.no_grad():
            for x, a in zip(leaves, args):
                x.copy_(a.roll(seed, 0).flip(1))
        want = step()
        for x in got:
            x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(got, want))

"""What goes round or through autograd beside plain reverse mode, at the operators' native calls: forward mode, functorch's
transforms, compiled autograd, saved-tensor hooks, tracing."""
import pytest
import torch

import specs

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

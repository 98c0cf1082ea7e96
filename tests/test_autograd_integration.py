"""The two layers' autograd nodes inside torch's own machinery: the function transforms are refused by name, and
saved-tensor hooks and activation checkpointing (both of which replace the tensors that a node keeps) give the same
gradients as a plain backward."""
import pytest
import torch
from torch.utils.checkpoint import checkpoint

from mhc import MHCLayer


def _layer(dynamic, device="cpu"):
    torch.manual_seed(3)
    return MHCLayer(128, 4, use_dynamic_h=dynamic).to(device)


@pytest.mark.parametrize("dynamic", [True, False])
@pytest.mark.parametrize("transform", ["grad", "vmap", "jvp"])
def test_function_transforms_are_refused_by_name(transform, dynamic):
    layer, x = _layer(dynamic), torch.randn(2, 4, 128)
    with pytest.raises(RuntimeError, match="(?i)autograd.*function|forward-mode|functorch|transforms"):
        if transform == "grad":
            torch.func.grad(lambda t: layer(t).sum())(x)
        elif transform == "vmap":
            torch.func.vmap(layer)(x.unsqueeze(0))
        else:
            torch.func.jvp(layer, (x,), (x,))


def _grads(layer, x, dy, call):
    layer.zero_grad()
    x = x.clone().requires_grad_(True)
    call(layer, x).backward(dy)
    return [x.grad] + [p.grad.clone() for p in layer.parameters()]


def _hooked(layer, x):
    def pack(t):
        return (t.device, t.cpu())

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda p: p[1].to(p[0])):
        return layer(x)


@pytest.mark.gpu
@pytest.mark.parametrize("dynamic", [True, False])
@pytest.mark.parametrize("call", [
    _hooked,
    lambda layer, x: checkpoint(layer, x, use_reentrant=False),
    lambda layer, x: checkpoint(layer, x, use_reentrant=True),
    lambda layer, x: checkpoint(lambda t: layer(layer(t)), x, use_reentrant=False),
], ids=["hooks to the host", "checkpoint", "reentrant checkpoint", "checkpoint over two calls"])
def test_saved_tensors_may_be_replaced(call, dynamic, request):
    layer = _layer(dynamic, "cuda")
    x, dy = torch.randn(5, 4, 128, device="cuda"), torch.randn(5, 4, 128, device="cuda")
    plain = (lambda l, t: l(l(t))) if "two calls" in request.node.callspec.id else (lambda l, t: l(t))
    for a, b in zip(_grads(layer, x, dy, call), _grads(layer, x, dy, plain)):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dynamic", [True, False])
def test_a_hook_that_changes_the_type_is_refused(dynamic):
    layer, x = _layer(dynamic, "cuda"), torch.randn(5, 4, 128, device="cuda")
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.to(torch.float16), lambda t: t):
        y = layer(x)
    with pytest.raises(RuntimeError, match="saved-tensor hook"):
        y.sum().backward()

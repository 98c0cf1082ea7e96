"""Argument forms of MHCLayer that come from configuration files and from user code: numbers of another type for
sinkhorn_iters and eps, an alpha that was replaced by a plain number."""
import pytest
import torch

from mhc import MHCLayer


def _layer(**kw):
    torch.manual_seed(0)
    return MHCLayer(64, 4, **kw)


def _with_number(**kw):
    layer = _layer(**kw)
    del layer.alpha_pre
    layer.alpha_pre = 0.01
    return layer


FORMS = [
    ("iters as a float", lambda d: _layer(use_dynamic_h=d, sinkhorn_iters=20.0)),
    ("iters and eps as text", lambda d: _layer(use_dynamic_h=d, sinkhorn_iters="20", eps="1e-5")),
    ("alpha as a number", lambda d: _with_number() if d else None),
]


@pytest.mark.parametrize("dynamic", [True, False])
@pytest.mark.parametrize("form,make", FORMS, ids=[f[0] for f in FORMS])
def test_argument_forms_reach_the_operator(form, make, dynamic):
    # the operator is reached: it refuses the CPU tensor, not the argument
    layer = make(dynamic)
    if layer is not None:
        with pytest.raises(RuntimeError, match="must live on a HIP"):
            layer(torch.randn(2, 4, 64))


@pytest.mark.gpu
@pytest.mark.parametrize("dynamic", [True, False])
@pytest.mark.parametrize("form,make", FORMS, ids=[f[0] for f in FORMS])
def test_argument_forms_give_the_same_result(form, make, dynamic):
    layer = make(dynamic)
    if layer is not None:
        x = torch.randn(2, 4, 64, device="cuda")
        with torch.no_grad():
            assert torch.equal(layer.cuda()(x), _layer(use_dynamic_h=dynamic).cuda()(x))

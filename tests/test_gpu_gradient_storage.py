"""What a kept gradient keeps alive: the small parameter gradients of a call (weight, biases, alphas) share no storage
with dphi, which is D * n * C floats and up to some hundred megabytes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 12])
def test_small_gradients_do_not_keep_dphi(n):
    from mhc import MHCLayer
    C = 512
    layer = MHCLayer(C, n).cuda()
    layer.phi_res.requires_grad_(False)
    layer(torch.randn(4, n, C, device="cuda")).sum().backward()
    D = n * n + 2 * n
    small = 4 * (D + 3 + 64 + C)  # floats, the second part at a multiple of 256 bytes
    for k in ("rmsnorm_weight", "alpha_pre", "alpha_post", "alpha_res", "b_pre", "b_post", "b_res"):
        assert getattr(layer, k).grad.untyped_storage().nbytes() <= small, k
    assert layer.phi_pre.grad.untyped_storage().nbytes() == 4 * D * n * C

"""The fp32 tier for n <= 8 at the edges of its kernels' tiles (32 samples and 32-element K chunks of the projection,
16 samples and 32 channels of the slab backward, 128 or 64 columns of dphi, batch splits): forward and every gradient
against the float64 oracle at 1e-5."""
import pytest
import torch

from gpu_util import hip_dynamic
from helpers import rel_err
from oracle import naive_mhc as nm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,n,C,inject", [
    (1, 4, 64, False), (15, 4, 66, True), (17, 4, 1282, False), (65, 3, 172, False), (33, 3, 90, True),
    (31, 2, 130, False), (200, 2, 258, False), (1100, 4, 40, False), (2500, 2, 34, False), (700, 4, 1280, False),
    (5, 8, 36, False), (64, 6, 130, True), (130, 5, 68, False), (600, 8, 100, False), (129, 7, 1284, False),
])
def test_fp32_narrow_products_vs_oracle(B, n, C, inject):
    x, dy, f, p = nm.make_dynamic_inputs(B, n, C, with_f=inject)
    g = torch.Generator().manual_seed(1)
    for k in ("alpha_pre", "alpha_post", "alpha_res"):
        p[k] = torch.full_like(p[k], 0.3)
    for k in ("b_pre", "b_post", "b_res"):
        p[k] = 0.5 * torch.randn(p[k].shape, generator=g)
    p["w"] = 1.0 + 0.3 * torch.randn(C, generator=g)
    y_ref, g_ref = nm.mhc_dynamic_fwd_bwd(x, p, dy, 20, 1e-6, f_inject=f, dtype=torch.float64)
    y, got = hip_dynamic(x, p, dy, 20, 1e-6, f_inject=f)
    assert rel_err(y, y_ref) <= 1e-5
    for k, v in g_ref.items():
        if not k.startswith("alpha"):  # sums of terms of both signs: test_gpu_parity holds them to their terms
            assert rel_err(got[k], v) <= 1e-5, k
        else:
            assert abs(float(got[k]) - float(v)) <= 1e-4 * abs(float(v)) + 1e-3, k

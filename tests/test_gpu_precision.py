"""How far results are from float64, by their 2-norm, where a faster path must not cost bits.

One rounding to bfloat16 is off by at most 2^-9 of every value, and so is a whole tensor's 2-norm; a second rounding
on the way adds to that (2.35e-3 in all).  Gradients in float32 of ragged rows: sums of a few hundred terms with 24 bits
each are off by 2e-7 .. 4e-7; a factor held in a bfloat16 value and remainder (16 bits) makes that 2.4e-6."""
import pytest
import torch

from gpu_util import hip_dynamic, hip_static
from oracle import naive_mhc as nm

pytestmark = pytest.mark.gpu

T, EPS = 20, 1e-5


def rel2(got, ref):
    return float((got.double() - ref.double()).norm() / ref.double().norm())


def _dynamic(B, n, C, bf16_weight=True):
    x, dy, _, p = nm.make_dynamic_inputs(B, n, C)
    g = torch.Generator().manual_seed(5)
    for k in ("alpha_pre", "alpha_post", "alpha_res"):
        p[k] = torch.full_like(p[k], 0.1)
    for k in ("b_pre", "b_post", "b_res"):
        p[k] = 0.5 * torch.randn(p[k].shape, generator=g)
    p["w"] = 1.0 + 0.1 * torch.randn(C, generator=g)
    if bf16_weight:
        p["w"] = p["w"].bfloat16().float()
    for k in ("phi_pre", "phi_post", "phi_res"):
        p[k] = p[k].bfloat16().float()
    return x.bfloat16().float(), dy.bfloat16().float(), p


# ragged rows; rows of more than 2560 channels; n = 5 .. 8 with rows of at most 512, with and without a split batch
@pytest.mark.parametrize("B,n,C", [(65, 4, 203), (40, 8, 77), (33, 3, 2701), (20, 4, 2568), (9, 8, 4096), (300, 2, 2816),
                                   (1100, 5, 264), (1030, 8, 512), (2100, 7, 64), (40, 8, 512)])
def test_dx_is_rounded_once(B, n, C):
    x, dy, p = _dynamic(B, n, C)
    _, ref = nm.mhc_dynamic_fwd_bwd(x, p, dy, T, EPS, dtype=torch.float64)
    _, got = hip_dynamic(x, p, dy, T, EPS, act_dtype=torch.bfloat16, out_dtype=torch.bfloat16, w_dtype=torch.bfloat16)
    assert rel2(got["x"], ref["x"]) <= 2.0 ** -9


@pytest.mark.parametrize("B,n,C", [(333, 3, 410), (130, 8, 213), (200, 6, 643), (1600, 4, 131)])
def test_ragged_rows_keep_float32_gradients(B, n, C):
    x, dy, p = _dynamic(B, n, C, bf16_weight=False)
    y_ref, ref = nm.mhc_dynamic_fwd_bwd(x, p, dy, T, EPS, dtype=torch.float64)
    y, got = hip_dynamic(x, p, dy, T, EPS, act_dtype=torch.bfloat16, w_dtype=torch.float32)  # dy in bfloat16 values
    for k in ("phi_pre", "phi_post", "phi_res", "w"):
        assert rel2(got[k], ref[k]) <= 1e-6, (k, rel2(got[k], ref[k]))
    assert rel2(y, y_ref) <= 5e-7  # float32 result of bfloat16 activations


@pytest.mark.parametrize("B,n,C", [(333, 3, 410), (130, 8, 213), (60, 5, 2575)])
def test_ragged_rows_of_shared_coefficients_keep_float32_results(B, n, C):
    x, dy, _, p = nm.make_static_inputs(B, n, C)
    x, dy = x.bfloat16().float(), dy.bfloat16().float()
    y_ref, ref = nm.mhc_static_fwd_bwd(x, p, dy, T, EPS, dtype=torch.float64)
    y, got = hip_static(x, p, dy, T, EPS, act_dtype=torch.bfloat16)
    assert rel2(y, y_ref) <= 5e-7 and rel2(got["w"], ref["w"]) <= 1e-6

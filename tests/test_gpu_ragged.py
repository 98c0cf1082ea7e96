"""Rows that are no multiple of a 16-byte access (n <= 8): the projection's K tail, the last chunk of a row in the
fused forward and in the two backward launches, and the longest rows of the sample-resident backward, against the
oracle at the tolerances of the two tiers; dynamic and static H."""
import pytest
import torch

from gpu_util import hip_dynamic, hip_static
from helpers import rel_err
from oracle import naive_mhc as nm

pytestmark = pytest.mark.gpu

T, EPS = 20, 1e-6
# (one stream only with an injected f: without it the gradients of Hpre are O(eps))
SHAPES = [(1, 8, 8), (3, 4, 9), (2, 1, 69), (33, 3, 90), (5, 3, 1230), (129, 2, 71), (40, 8, 277), (31, 5, 1037),
          (300, 4, 514), (130, 7, 643), (2, 4, 2561), (3, 8, 2575), (2, 6, 4095), (9, 3, 4096), (900, 4, 131)]


def _close(got, ref, k, bf16):
    e = rel_err(got, ref)
    assert torch.isfinite(got).all() and e <= (2e-2 if bf16 else 1e-5), f"{k}: {e:.3e}"
    if bf16 and k in ("y", "x"):
        bad = (got.double() - ref.double()).abs() > 2e-2 * ref.double().abs() + 1e-2
        assert not bad.any(), f"{k}: {int(bad.sum())} elements outside rtol/atol"


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("B,n,C", SHAPES)
def test_dynamic_rows_of_any_length(B, n, C, bf16):
    inject = C % 3 == 0
    x, dy, f, p = nm.make_dynamic_inputs(B, n, C, with_f=inject)
    g = torch.Generator().manual_seed(2)
    for k in ("alpha_pre", "alpha_post", "alpha_res"):
        p[k] = torch.full_like(p[k], 0.1)
    for k in ("b_pre", "b_post", "b_res"):
        p[k] = 0.5 * torch.randn(p[k].shape, generator=g)
    p["w"] = (1.0 + 0.3 * torch.randn(C, generator=g)).bfloat16().float()
    if bf16:
        x, dy, f = x.bfloat16().float(), dy.bfloat16().float(), None if f is None else f.bfloat16().float()
        for k in ("phi_pre", "phi_post", "phi_res"):
            p[k] = p[k].bfloat16().float()
    act = torch.bfloat16 if bf16 else torch.float32
    y_ref, g_ref = nm.mhc_dynamic_fwd_bwd(x, p, dy, T, EPS, f_inject=f, dtype=torch.float64)
    y, got = hip_dynamic(x, p, dy, T, EPS, f_inject=f, act_dtype=act, out_dtype=act,
                         w_dtype=torch.bfloat16 if C % 2 else torch.float32)
    _close(y, y_ref, "y", bf16)
    for k, v in g_ref.items():
        if k.startswith("alpha"):  # sums of terms of both signs
            assert abs(float(got[k]) - float(v)) <= (2e-2 if bf16 else 1e-4) * abs(float(v)) + (2e-1 if bf16 else 1e-3), k
        else:
            _close(got[k], v, k, bf16 or (k == "w" and C % 2))


@pytest.mark.parametrize("B,n,C", SHAPES)
def test_static_rows_of_any_length(B, n, C):
    x, dy, f, p = nm.make_static_inputs(B, n, C, with_f=C % 3 == 0)
    x, dy, f = x.bfloat16().float(), dy.bfloat16().float(), None if f is None else f.bfloat16().float()
    g = torch.Generator().manual_seed(3)
    for k in ("H_pre", "H_post", "H_res"):
        p[k] = torch.randn(p[k].shape, generator=g)
    y_ref, g_ref = nm.mhc_static_fwd_bwd(x, p, dy, T, EPS, f_inject=f, dtype=torch.float64)
    y, got = hip_static(x, p, dy, T, EPS, f_inject=f, act_dtype=torch.bfloat16, out_dtype=torch.bfloat16)
    _close(y, y_ref, "y", True)
    for k, v in g_ref.items():
        _close(got[k], v, k, True)

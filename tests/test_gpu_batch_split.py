"""The second backward launch with the batch split over workgroups (few column slabs, many samples; its partial sums of
dphi, dw, dbias and dalpha are added up by one more launch): blocks and parts of 128 samples at their edges, one to
three row tiles of phi, whole and ragged rows, and the narrowest tile-wave counts, against the oracle."""
import pytest
import torch

from gpu_util import hip_dynamic
from helpers import rel_err
from oracle import naive_mhc as nm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,n,C", [(1281, 8, 64), (1536, 5, 48), (1921, 4, 37), (2049, 6, 16), (1793, 2, 30), (1600, 7, 33)])
def test_split_batch_against_the_oracle(B, n, C):
    x, dy, _, p = nm.make_dynamic_inputs(B, n, C)
    g = torch.Generator().manual_seed(4)
    for k in ("alpha_pre", "alpha_post", "alpha_res"):
        p[k] = torch.full_like(p[k], 0.1)
    for k in ("b_pre", "b_post", "b_res"):
        p[k] = 0.5 * torch.randn(p[k].shape, generator=g)
    p["w"] = (1.0 + 0.3 * torch.randn(C, generator=g)).bfloat16().float()
    x, dy = x.bfloat16().float(), dy.bfloat16().float()
    for k in ("phi_pre", "phi_post", "phi_res"):
        p[k] = p[k].bfloat16().float()
    y_ref, g_ref = nm.mhc_dynamic_fwd_bwd(x, p, dy, 20, 1e-6, dtype=torch.float64)
    y, got = hip_dynamic(x, p, dy, 20, 1e-6, act_dtype=torch.bfloat16, out_dtype=torch.bfloat16)
    assert rel_err(y, y_ref) <= 2e-2 and rel_err(got["x"], g_ref["x"]) <= 2e-2
    for k, v in g_ref.items():
        if k.startswith("alpha"):  # sums over all samples of terms of both signs
            assert abs(float(got[k]) - float(v)) <= 1e-2 * abs(float(v)) + 1e-1, k
        elif k != "x":
            assert rel_err(got[k], v) <= 1e-3, k

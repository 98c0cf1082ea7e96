"""Sinkhorn of n > 8 streams (one wave per matrix: 16 x 16 tiles up to n = 16, 32 x 32 beyond): M and the saved denominators against
float64, on either side of the tiles' edges, for no, one and many iterations, both tiers.

A half-step rounds a sum of at most 16 products in four chains (9 * 2^-24 with the sums of the chains and halves) and a reciprocal
(2^-23); the entries come with the error of the exponential (2^-22 for logits of a few units).  What a half-step leaves behind in
a scaling the next ones divide out again: four times the sum of these, 4e-6 of the largest value."""
import pytest
import torch

from helpers import rel_err
from test_gpu_sinkhorn_state import _fwd_bwd

pytestmark = pytest.mark.gpu
EPS = 1e-6


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [9, 15, 16, 17, 24, 31, 32])
def test_against_float64(n, dtype):
    for T in (0, 1, 2, 20, 33):
        got = _fwd_bwd(3, n, 64, dtype, T, EPS, seed=n, with_state=True)
        if T == 0:  # M is the matrix of the exponentials, which nothing else returns
            assert torch.isfinite(got["M"]).all() and (got["M"] > 0).all()
            continue
        logits = (got["alpha_res"] * got["P"][:, 2 * n:].double().reshape(3, n, n) + got["b_res"].double())
        E = torch.exp(logits)
        u = torch.ones(3, n, dtype=torch.float64)
        v = torch.ones(3, n, dtype=torch.float64)
        for t in range(T):
            rho = u * (E @ v[..., None])[..., 0] + EPS
            u = u / rho
            s = v * (E.transpose(1, 2) @ u[..., None])[..., 0] + EPS
            v = v / s
            assert rel_err(got["sk"][:, t, 0].double(), rho) <= 4e-6, (T, t)
            assert rel_err(got["sk"][:, t, 1].double(), s) <= 4e-6, (T, t)
        assert rel_err(got["M"].double(), u[..., None] * E * v[:, None, :]) <= 4e-6, T

"""MHCLayer: drop-in for the reference's mhc.MHCLayer (src/python/mhc/layer.py:6-101).

Same constructor, parameter names, shapes, dtypes and initialisers; forward returns float32
[B, n, C] for any floating input unless `output_dtype` is set.
"""
from __future__ import annotations

import torch
import torch.nn as nn

from .ops import _as_tensor, _ext

# in the order of the operators' arguments
_DYNAMIC_PARAMS = ("rmsnorm_weight", "phi_pre", "phi_post", "phi_res", "alpha_pre", "alpha_post", "alpha_res",
                   "b_pre", "b_post", "b_res")
_STATIC_PARAMS = ("rmsnorm_weight", "H_pre", "H_post", "H_res")


class MHCLayer(nn.Module):
    """mHC: Manifold-Constrained Hyper-Connections (DeepSeek-AI, arXiv 2512.24880).

    Args:
        hidden_dim: hidden dimension C (at most 32768; larger values raise MHCError at the first call).
        expansion_rate: number of residual streams n (1..32).
        sinkhorn_iters: Sinkhorn-Knopp iterations (at most 256: the exact backward keeps the
            denominators of every iteration on chip).
        eps: one epsilon shared by both RMSNorms and the Sinkhorn denominators.
        alpha_init: initial value of the alpha gates (dynamic) / scale of H_res (static).
        use_dynamic_h: per-sample coefficients projected from x (True) or shared parameters.
        output_dtype: dtype of the result; None keeps the reference's float32.  Passing
            torch.bfloat16 with bfloat16 inputs keeps the whole layer at 2 bytes per element.
        compute_dtype: None computes in the dtype of the input (float32 inputs take the exact
            float32 kernels).  torch.bfloat16 selects the matrix-core kernels for float32 inputs,
            which is what the reference's fused path does with them (its kernels store activations
            as bfloat16, src/csrc/include/mhc_types.h:10): dynamic H with n <= 8 and a batch the
            two-launch backward serves rounds the activations inside the kernels (no cast pass);
            other shapes and static H cast the input first.
    """

    def __init__(self, hidden_dim: int, expansion_rate: int = 4, sinkhorn_iters: int = 20,
                 eps: float = 1e-5, alpha_init: float = 0.01, use_dynamic_h: bool = True,
                 output_dtype=None, compute_dtype=None):
        super().__init__()
        self.hidden_dim = hidden_dim
        self.expansion_rate = expansion_rate
        self.sinkhorn_iters = sinkhorn_iters
        self.eps = eps
        self.use_dynamic_h = use_dynamic_h
        self.output_dtype = output_dtype
        self.compute_dtype = compute_dtype

        n, C = expansion_rate, hidden_dim
        nC = n * C
        self.rmsnorm_weight = nn.Parameter(torch.ones(C, dtype=torch.bfloat16))
        if use_dynamic_h:
            self.phi_pre = nn.Parameter(torch.randn(n, nC) * 0.02)
            self.phi_post = nn.Parameter(torch.randn(n, nC) * 0.02)
            self.phi_res = nn.Parameter(torch.randn(n * n, nC) * 0.02)
            self.b_pre = nn.Parameter(torch.zeros(n))
            self.b_post = nn.Parameter(torch.zeros(n))
            self.b_res = nn.Parameter(torch.zeros(n, n))
            self.alpha_pre = nn.Parameter(torch.tensor(alpha_init))
            self.alpha_post = nn.Parameter(torch.tensor(alpha_init))
            self.alpha_res = nn.Parameter(torch.tensor(alpha_init))
        else:
            self.H_pre = nn.Parameter(torch.zeros(n, dtype=torch.float32))
            self.H_post = nn.Parameter(torch.zeros(n, dtype=torch.float32))
            self.H_res = nn.Parameter((alpha_init * torch.randn(n, n)).float())

    def _params(self, names):
        # nn.Module.__getattr__ is a Python call per parameter, which adds up at the sizes where the host
        # decides the time of a call; a parameter that was replaced by a property (parametrizations,
        # pruning) is not in the dictionary and goes the ordinary way
        p = self._parameters
        try:
            return [p[k] for k in names]
        except KeyError:
            # (an alpha may also have been replaced by a plain number)
            return [_as_tensor(getattr(self, k), self.phi_pre) if k.startswith("alpha") else getattr(self, k) for k in names]

    def forward(self, x_expanded: torch.Tensor) -> torch.Tensor:
        B, n, C = x_expanded.shape
        assert n == self.expansion_rate
        assert C == self.hidden_dim
        compute = self.compute_dtype
        # (a configuration file hands over 20.0 or "1e-5")
        iters, eps = int(self.sinkhorn_iters), float(self.eps)
        cast = compute is not None and x_expanded.dtype != compute
        if self.use_dynamic_h:
            # float32 activations with compute_dtype=bfloat16: the operator rounds them inside its kernels
            # where it can and casts them itself elsewhere
            in_op = cast and compute == torch.bfloat16 and x_expanded.dtype == torch.float32
            if cast and not in_op:
                x_expanded = x_expanded.to(compute)
            return _ext.mhc_layer_dynamic(x_expanded, *self._params(_DYNAMIC_PARAMS), iters, eps,
                                          self.output_dtype, None, in_op)
        if cast:
            x_expanded = x_expanded.to(compute)
        params = self._params(_STATIC_PARAMS)
        if not self.training and not torch.is_grad_enabled():
            return _ext.mhc_layer_inference(x_expanded, *params, iters, eps, self.output_dtype)
        return _ext.mhc_layer_static(x_expanded, *params, iters, eps, self.output_dtype, None)

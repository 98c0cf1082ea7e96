"""The projection of the forward for n = 5 .. 8 with one row tile of phi per workgroup (few workgroups) and with all of them
(more than 22 MiB of x), around the line between the two and at the edges of the tiles: the saved projection and RMS, with phi
packed and with phi read from the caller's float32 parameters.

Bound: the products are exact (bf16) or rounded once (float32); a sum of K terms in float32 is off by at most K 2^-24 times the sum
of the magnitudes, of which an accumulation over tiles of at least 8 terms leaves K / 8.  Inputs as the kernels see them."""
import ctypes

import pytest
import torch

from test_gpu_param_gather import Params

pytestmark = pytest.mark.gpu

K_GATHER = 10


@pytest.mark.parametrize("B,n,C,kind", [
    (1, 5, 64, "bf16"), (33, 6, 72, "bf16"), (64, 7, 777, "bf16"), (100, 8, 2560, "bf16"), (1126, 8, 1280, "bf16"), (1127, 8, 1280, "bf16"),
    (31, 8, 264, "mixed"), (563, 8, 1280, "mixed"), (564, 8, 1280, "mixed"),
    (5, 5, 52, "fp32"), (65, 8, 1283, "fp32"), (563, 8, 1280, "fp32"), (564, 8, 1280, "fp32"), (751, 6, 1280, "fp32")])
@pytest.mark.parametrize("gather", [1, 2])
def test_projection_in_row_groups(B, n, C, kind, gather):
    from mhc import _lib
    from mhc._lib import check, ptr

    lib = _lib.tuning_lib()
    D, nC, T = n * n + 2 * n, n * C, 20
    g = torch.Generator(device="cuda").manual_seed(B + n + C)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = r(B, n, C).bfloat16() if kind == "bf16" else r(B, n, C)
    w = r(C).bfloat16()
    phi = [r(n, nC) * 0.1, r(n, nC) * 0.1, r(n * n, nC) * 0.1]
    small = [r(n), r(n), r(n * n), r(()), r(()), r(())]
    p = Params(*[t.data_ptr() for t in phi], _lib.MHC_F32, *[t.data_ptr() for t in small])
    cd = torch.float32 if kind == "fp32" else torch.bfloat16
    code = {"bf16": _lib.MHC_BF16, "mixed": _lib.MHC_F32_AS_BF16, "fp32": _lib.MHC_F32}[kind]
    xs, ps = x.to(cd).double().reshape(B, nC), torch.cat(phi).to(cd).double()
    rms = (xs.square().mean(1) + 1e-6).sqrt()
    want, size = xs @ ps.T / rms[:, None], xs.abs() @ ps.abs().T / rms[:, None]
    f = lambda *s: torch.full(s, float("nan"), device="cuda")
    y, Hp, Ho, M, P, rr, q = torch.full_like(x, float("nan")), f(B, n), f(B, n), f(B, n, n), f(B, D), f(B), f(B)
    sk, phi_o, bias, alpha = f(lib.mhc_layer_sinkhorn_state_floats(B, n, T)), f(D, nC).to(cd), f(D), f(3)
    ws = torch.full((lib.mhc_layer_dynamic_workspace_bytes(B, n, C),), 255, dtype=torch.uint8, device="cuda")
    try:
        assert lib.mhc_tuning_set(K_GATHER, gather) == 0
        check("mhc_layer_fwd_dynamic_params", lib.mhc_layer_fwd_dynamic_params(
            ptr(x), code, ptr(w), _lib.MHC_BF16, ctypes.addressof(p), ptr(phi_o), _lib.MHC_F32 if kind == "fp32" else _lib.MHC_BF16,
            ptr(bias), ptr(alpha), None, ptr(y), _lib.dtype_code(y), ptr(Hp), ptr(Ho), ptr(M), ptr(P), ptr(rr),
            ptr(q), ptr(sk), B, n, C, T, 1e-6, ptr(ws), ws.numel(), _lib.stream_ptr(x.device)))
        torch.cuda.synchronize()
    finally:
        lib.mhc_tuning_set(K_GATHER, 0)
    bound = (nC / 8 + 64) * 2.0 ** -24
    assert torch.equal(phi_o, torch.cat(phi).to(cd)) and torch.isfinite(y).all()
    assert ((P.double() - want).abs() <= bound * size).all()
    assert ((rr.double() - rms).abs() <= bound * rms).all()

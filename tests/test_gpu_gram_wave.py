"""Backward of n = 5 .. 8 with a wave per sample for the channel sums and the coefficient backward: against the sample-resident backward
on the same inputs, over rows shorter than, at and beyond a step, batches that end inside a workgroup, both types of the weight, an f
of the caller's, with and without the saved Sinkhorn state.

Both round x, dy and the operands of dP phi alike and compute in float32 behind that: they differ by the order of float32 sums and by
coefficients of 1 ulp, 2e-5 of the largest value at most; dx and df leave in bf16, where neighbours are up to 2^-7 of a value apart."""
import pytest
import torch

from helpers import rel_err

pytestmark = pytest.mark.gpu

T, EPS = 20, 1e-6
K_GRAM, K_RESIDENT = 2, 7


@pytest.fixture(autouse=True)
def _reset_tuning():
    from mhc._lib import tuning_lib

    yield
    for k in (K_GRAM, K_RESIDENT):
        tuning_lib().mhc_tuning_set(k, 0)


def _run(B, n, C, wt, inject, state, wave):
    from mhc import _lib
    from mhc._lib import check, dtype_code, ptr

    lib = _lib.tuning_lib()
    assert lib.mhc_tuning_set(K_RESIDENT, 1 if wave else 2) == 0 and lib.mhc_tuning_set(K_GRAM, 2 if wave else 0) == 0
    g = torch.Generator(device="cuda").manual_seed(B + n + C)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    D, f32, bf = n * n + 2 * n, dict(device="cuda"), torch.bfloat16
    x, dy, w, phi = rn(B, n, C).to(bf), rn(B, n, C).to(bf), (1 + 0.1 * rn(C)).to(wt), (0.02 * rn(D, n * C)).to(bf)
    bias, alpha = 0.5 * rn(D), torch.tensor([0.3, 0.4, 0.5], device="cuda")
    f = rn(B, C).to(bf) if inject else None
    y = torch.empty_like(dy)
    Hp, Ho, M = torch.empty(B, n, **f32), torch.empty(B, n, **f32), torch.empty(B, n, n, **f32)
    P, r, q = torch.empty(B, D, **f32), torch.empty(B, **f32), torch.empty(B, **f32)
    sk = torch.empty(lib.mhc_layer_sinkhorn_state_floats(B, n, T), **f32) if state else None
    ws = torch.full((lib.mhc_layer_dynamic_workspace_bytes(B, n, C),), 0xFF, dtype=torch.uint8, device="cuda")
    st = _lib.stream_ptr(x.device)
    opt = lambda t: None if t is None else ptr(t)
    check("mhc_layer_fwd_dynamic",
          lib.mhc_layer_fwd_dynamic(ptr(x), dtype_code(x), ptr(w), dtype_code(w), ptr(phi), dtype_code(phi), ptr(bias), ptr(alpha), opt(f),
                                    ptr(y), dtype_code(y), ptr(Hp), ptr(Ho), ptr(M), ptr(P), ptr(r), ptr(q), opt(sk), B, n, C, T, EPS,
                                    ptr(ws), ws.numel(), st))
    nan = lambda *s, dt=torch.float32: torch.full(s, float("nan"), device="cuda", dtype=dt)
    dx = nan(B + 1, n, C, dt=bf)  # one sample more: nothing may be written there
    out = dict(dphi=nan(D, n * C), dbias=nan(D), dalpha=nan(3))
    out.update(dict(df=nan(B, C, dt=bf)) if inject else dict(dw=nan(C)))
    check("mhc_layer_bwd_dynamic",
          lib.mhc_layer_bwd_dynamic(ptr(dy), dtype_code(dy), ptr(x), dtype_code(x), ptr(w), dtype_code(w), ptr(phi), dtype_code(phi),
                                    ptr(bias), ptr(alpha), opt(f), ptr(Hp), ptr(Ho), ptr(M), ptr(P), ptr(r), ptr(q), opt(sk), ptr(dx),
                                    opt(out.get("df")), opt(out.get("dw")), ptr(out["dphi"]), ptr(out["dbias"]), ptr(out["dalpha"]),
                                    B, n, C, T, EPS, ptr(ws), ws.numel(), st))
    torch.cuda.synchronize()
    assert torch.isnan(dx[B].float()).all(), "wrote behind the batch"
    return dict(out, dx=dx[:B])


@pytest.mark.parametrize("wt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [5, 6, 7, 8])
def test_same_as_the_resident_backward(n, wt):
    for B, C, inject, state in ((1, 8, False, True), (3, 64, True, True), (4, 128, False, False), (5, 136, False, True), (17, 264, True, False),
                                (66, 512, False, True), (130, 1032, False, True)):
        want, got = (_run(B, n, C, wt, inject, state, wave) for wave in (False, True))
        for k in want:
            assert torch.isfinite(got[k].float()).all(), (B, C, k)
            # the three dalpha: sums over the batch of terms of both signs
            e = rel_err(got[k].cpu(), want[k].cpu())
            assert e <= {"dalpha": 1e-3, "dx": 2.0 ** -7, "df": 2.0 ** -7}.get(k, 2e-5), (B, C, k, e)

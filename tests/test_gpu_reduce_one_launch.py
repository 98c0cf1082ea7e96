"""Channel sums and coefficient backward of the tiled path (n <= 8, everything but whole bf16 rows) in one launch and in two: the same
chains in the same order, so every output is the same bit for bit - rows of one and of two column parts, rows that end inside a chunk,
both widths of the streams' tile, an f of the caller's, with and without the saved Sinkhorn state.  (n > 4 without it: the iterations are
repeated, and there the lanes of a row have one rounding of its sum in common; 20 of 2^-24, 2e-5 of the largest value at most.)

One wave per sample (n <= 4) adds in another order: float32 sums of up to 2048 channels, 2e-5 of the largest value; bf16 results may
become the neighbour, up to 2^-7 of a value."""
import pytest
import torch

from helpers import rel_err

pytestmark = pytest.mark.gpu

T, EPS = 20, 1e-6
K_FUSED, K_RESIDENT = 2, 7


@pytest.fixture(autouse=True)
def _reset_tuning():
    from mhc._lib import tuning_lib

    yield
    for k in (K_FUSED, K_RESIDENT):
        tuning_lib().mhc_tuning_set(k, 0)


def _run(B, n, C, xt, yt, inject, state, one):
    from mhc import _lib
    from mhc._lib import check, dtype_code, ptr

    lib = _lib.tuning_lib()
    assert lib.mhc_tuning_set(K_RESIDENT, 1) == 0 and lib.mhc_tuning_set(K_FUSED, one) == 0
    g = torch.Generator(device="cuda").manual_seed(B + n + C)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    D, f32 = n * n + 2 * n, dict(device="cuda")
    x, dy, w, phi = rn(B, n, C).to(xt), rn(B, n, C).to(yt), 1 + 0.1 * rn(C), (0.02 * rn(D, n * C)).to(xt)
    bias, alpha = 0.5 * rn(D), torch.tensor([0.3, 0.4, 0.5], device="cuda")
    f = rn(B, C).to(xt) if inject else None
    y = torch.empty_like(dy)
    Hp, Ho, M = torch.empty(B, n, **f32), torch.empty(B, n, **f32), torch.empty(B, n, n, **f32)
    P, r, q = torch.empty(B, D, **f32), torch.empty(B, **f32), torch.empty(B, **f32)
    sk = torch.empty(lib.mhc_layer_sinkhorn_state_floats(B, n, T), **f32) if state else None
    ws = torch.full((lib.mhc_layer_dynamic_workspace_bytes(B, n, C),), 0xFF, dtype=torch.uint8, device="cuda")
    st = _lib.stream_ptr(x.device)
    check("mhc_layer_fwd_dynamic",
          lib.mhc_layer_fwd_dynamic(ptr(x), dtype_code(x), ptr(w), dtype_code(w), ptr(phi), dtype_code(phi), ptr(bias), ptr(alpha),
                                    ptr(f) if inject else None, ptr(y), dtype_code(y), ptr(Hp), ptr(Ho), ptr(M), ptr(P), ptr(r), ptr(q),
                                    ptr(sk) if state else None, B, n, C, T, EPS, ptr(ws), ws.numel(), st))
    nan = lambda *s, dt=torch.float32: torch.full(s, float("nan"), device="cuda", dtype=dt)
    out = dict(dx=nan(B, n, C, dt=xt), dphi=nan(D, n * C), dbias=nan(D), dalpha=nan(3))
    if inject:
        out["df"] = nan(B, C, dt=xt)
    else:
        out["dw"] = nan(C)
    check("mhc_layer_bwd_dynamic",
          lib.mhc_layer_bwd_dynamic(ptr(dy), dtype_code(dy), ptr(x), dtype_code(x), ptr(w), dtype_code(w), ptr(phi), dtype_code(phi),
                                    ptr(bias), ptr(alpha), ptr(f) if inject else None, ptr(Hp), ptr(Ho), ptr(M), ptr(P), ptr(r), ptr(q),
                                    ptr(sk) if state else None, ptr(out["dx"]), ptr(out["df"]) if inject else None,
                                    None if inject else ptr(out["dw"]), ptr(out["dphi"]), ptr(out["dbias"]), ptr(out["dalpha"]),
                                    B, n, C, T, EPS, ptr(ws), ws.numel(), st))
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("xt,yt", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 8])
def test_one_launch_is_the_two(n, xt, yt):
    for B, C, inject, state in ((1, 5, False, True), (3, 64, False, False), (2, 515, True, True), (7, 1030, False, True), (2, 2048, True, False),
                                (65, 1028, False, True)):
        want, got = (_run(B, n, C, xt, yt, inject, state, one) for one in (1, 2))
        wave = _run(B, n, C, xt, yt, inject, state, 3) if n <= 4 else None
        for k in want:
            assert torch.isfinite(got[k].float()).all(), (B, C, k)
            if xt == torch.bfloat16 and yt == xt and C % 8 == 0:
                continue  # whole bf16 rows: the sums come from the matrix cores, in either order
            exact = state or n <= 4
            assert not exact or torch.equal(got[k], want[k]), (B, C, k)
            for other in ([] if exact else [got]) + ([wave] if wave else []):
                if k != "dalpha":  # (sums of terms of both signs, over the batch)
                    e = rel_err(other[k].float().cpu(), want[k].float().cpu())
                    assert e <= (2.0 ** -7 if other[k].dtype == torch.bfloat16 else 2e-5), (B, C, k, e)

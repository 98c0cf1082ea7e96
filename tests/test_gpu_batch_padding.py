"""The columns of dP^T behind a batch that is no multiple of 32 are cleared by the last samples' workgroups, up to seven single
ones and then whole groups of eight: whatever the workspace held before, the gradients are the same, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

T, EPS = 20, 1e-6


def _backward(B, n, C, fill):
    from mhc import _lib
    from mhc._lib import check, dtype_code, lib, ptr

    g = torch.Generator(device="cuda").manual_seed(B + n + C)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    D = n * n + 2 * n
    x, dy, w = rn(B, n, C).bfloat16(), rn(B, n, C).bfloat16(), (1 + 0.1 * rn(C)).bfloat16()
    phi, bias, alpha = (0.02 * rn(D, n * C)).bfloat16(), 0.5 * rn(D), torch.full((3,), 0.3, device="cuda")
    f32 = dict(device="cuda")
    y, Hp, Ho, M = torch.empty_like(x), torch.empty(B, n, **f32), torch.empty(B, n, **f32), torch.empty(B, n, n, **f32)
    P, r, q = torch.empty(B, D, **f32), torch.empty(B, **f32), torch.empty(B, **f32)
    sk = torch.empty(lib.mhc_layer_sinkhorn_state_floats(B, n, T), **f32)
    ws = torch.empty(lib.mhc_layer_dynamic_workspace_bytes(B, n, C), dtype=torch.uint8, device="cuda")
    st = _lib.stream_ptr(x.device)
    check("mhc_layer_fwd_dynamic",
          lib.mhc_layer_fwd_dynamic(ptr(x), dtype_code(x), ptr(w), dtype_code(w), ptr(phi), dtype_code(phi), ptr(bias),
                                    ptr(alpha), None, ptr(y), dtype_code(y), ptr(Hp), ptr(Ho), ptr(M), ptr(P), ptr(r), ptr(q),
                                    ptr(sk), B, n, C, T, EPS, ptr(ws), ws.numel(), st))
    ws.fill_(fill)
    out = dict(dx=torch.empty_like(x), dw=torch.empty(C, **f32), dphi=torch.empty(D, n * C, **f32),
               dbias=torch.empty(D, **f32), dalpha=torch.empty(3, **f32))
    check("mhc_layer_bwd_dynamic",
          lib.mhc_layer_bwd_dynamic(ptr(dy), dtype_code(dy), ptr(x), dtype_code(x), ptr(w), dtype_code(w), ptr(phi),
                                    dtype_code(phi), ptr(bias), ptr(alpha), None, ptr(Hp), ptr(Ho), ptr(M), ptr(P), ptr(r),
                                    ptr(q), ptr(sk), ptr(out["dx"]), None, ptr(out["dw"]), ptr(out["dphi"]),
                                    ptr(out["dbias"]), ptr(out["dalpha"]), B, n, C, T, EPS, ptr(ws), ws.numel(), st))
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("n,C", [(4, 256), (3, 123), (8, 512), (12, 256), (32, 256)])
def test_columns_behind_the_batch(n, C):
    for B in (1, 2, 3, 7, 8, 9, 15, 17, 24, 25, 31, 32, 33, 41, 63, 65):
        want, got = _backward(B, n, C, 0), _backward(B, n, C, 0xFF)  # 0xFF..: NaN in either float type
        for k in want:
            assert torch.isfinite(got[k]).all(), (B, k)
            assert torch.equal(got[k], want[k]), (B, k)


def test_columns_behind_a_large_batch():
    """The tiled kernels (channel sums and slab), several samples per workgroup."""
    for B in (1281, 2003):
        want, got = _backward(B, 4, 512, 0), _backward(B, 4, 512, 0xFF)
        for k in want:
            assert torch.equal(got[k], want[k]), (B, k)

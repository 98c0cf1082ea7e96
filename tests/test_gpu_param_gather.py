"""The dynamic forward on the parameters as a layer stores them: read by the projection kernels themselves or
packed by a launch of their own, forced through the experiment hook, bit for bit the same; and dw handed back in
bfloat16 equals the float32 one rounded once."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

K_GATHER = 10


class Params(ctypes.Structure):  # struct mhc_dynamic_params
    _fields_ = [("phi_pre", ctypes.c_void_p), ("phi_post", ctypes.c_void_p), ("phi_res", ctypes.c_void_p),
                ("phi_dtype", ctypes.c_int), ("b_pre", ctypes.c_void_p), ("b_post", ctypes.c_void_p),
                ("b_res", ctypes.c_void_p), ("alpha_pre", ctypes.c_void_p), ("alpha_post", ctypes.c_void_p),
                ("alpha_res", ctypes.c_void_p)]


def _inputs(B, n, C, mixed):
    g = torch.Generator(device="cuda").manual_seed(7)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = r(B, n, C) if mixed else r(B, n, C).bfloat16()
    return x, r(C).bfloat16(), [r(n, n * C), r(n, n * C), r(n * n, n * C)], [r(n), r(n), r(n * n), r(()), r(()), r(())]


def _forward(x, w, phi, small, gather=0):
    from mhc import _lib
    from mhc._lib import check, ptr

    lib = _lib.tuning_lib()
    B, n, C = x.shape
    D, nC, T = n * n + 2 * n, n * C, 20
    p = Params(*[t.data_ptr() for t in phi], _lib.MHC_F32, *[t.data_ptr() for t in small])
    f = lambda *s: torch.full(s, float("nan"), device="cuda")
    out = [torch.full((B, n, C), float("nan"), dtype=x.dtype, device="cuda"), f(B, n), f(B, n), f(B, n, n), f(B, D), f(B),
           f(B), f(lib.mhc_layer_sinkhorn_state_floats(B, n, T)), f(D, nC).bfloat16(), f(D), f(3)]
    y, Hp, Ho, M, P, rr, q, sk, phi_o, bias, alpha = out
    ws = torch.empty(lib.mhc_layer_dynamic_workspace_bytes(B, n, C), dtype=torch.uint8, device="cuda")
    try:
        assert lib.mhc_tuning_set(K_GATHER, gather) == 0
        check("mhc_layer_fwd_dynamic_params", lib.mhc_layer_fwd_dynamic_params(
            ptr(x), _lib.MHC_BF16 if x.dtype == torch.bfloat16 else _lib.MHC_F32_AS_BF16, ptr(w), _lib.MHC_BF16, ctypes.addressof(p),
            ptr(phi_o), _lib.MHC_BF16, ptr(bias), ptr(alpha), None, ptr(y), _lib.dtype_code(y), ptr(Hp), ptr(Ho), ptr(M), ptr(P),
            ptr(rr), ptr(q), ptr(sk), B, n, C, T, 1e-6, ptr(ws), ws.numel(), _lib.stream_ptr(x.device)))
        torch.cuda.synchronize()
    finally:
        lib.mhc_tuning_set(K_GATHER, 0)
    return out


@pytest.mark.parametrize("B,n,C,mixed", [
    (1, 4, 8, False), (33, 4, 72, False), (70, 3, 1288, False), (7, 4, 1280, True),  # one row tile of phi
    (5, 6, 264, False), (40, 7, 136, True), (65, 8, 520, False),                     # two and three row tiles
    (3, 12, 64, False), (130, 20, 128, False), (17, 32, 64, False),                  # wide, one and two sample groups
])
def test_parameters_read_by_the_projection_match_the_packing_launch(B, n, C, mixed):
    x, w, phi, small = _inputs(B, n, C, mixed)
    res = [_forward(x, w, phi, small, gather) for gather in (1, 2)]
    assert torch.equal(res[1][8], torch.cat(phi).bfloat16())
    assert torch.equal(res[1][9], torch.cat(small[:3])) and torch.equal(res[1][10], torch.stack(small[3:]))
    for k, (a, b) in enumerate(zip(*res)):
        assert torch.equal(a.nan_to_num(1e30), b.nan_to_num(1e30)), k


HELD = [(4112, 4, 384, False), (1700, 3, 192, True)]  # sixteen samples per workgroup, bf16 and float32 storage


@pytest.mark.parametrize("B,n,C,mixed", [
    (1, 4, 64, False), (37, 4, 64, False), (300, 4, 128, False), (3000, 2, 64, False), (9, 3, 640, False), (40, 1, 128, False),
    (1500, 4, 768, False),                              # one launch: one workgroup, fewer steps than workgroups, two row pieces, steps from each workgroup's own starting point
    *HELD,
])
def test_parameters_read_by_the_one_pass_forwards(B, n, C, mixed):
    from mhc import _lib

    one, reads, held = 1, 2, 3
    lib, code = _lib.tuning_lib(), _lib.MHC_F32_AS_BF16 if mixed else _lib.MHC_BF16
    is_held = (B, n, C, mixed) in HELD
    try:  # the two sides differ in nothing but who packs the parameters
        assert lib.mhc_tuning_set(K_GATHER, 2) == 0 and lib.mhc_tuning_route(1, code, B, n, C) == (held if is_held else reads)
        assert lib.mhc_tuning_set(K_GATHER, 1) == 0 and lib.mhc_tuning_route(1, code, B, n, C) == (held if is_held else one)
    finally:
        lib.mhc_tuning_set(K_GATHER, 0)
    test_parameters_read_by_the_projection_match_the_packing_launch(B, n, C, mixed)


@pytest.mark.parametrize("B,n,C,mixed", HELD)
def test_held_forward_of_parameters_that_are_no_whole_pieces(B, n, C, mixed):
    """Matrices that begin four bytes behind a 16-byte boundary, as views of a flat buffer do: packed by a launch of their own."""
    x, w, phi, small = _inputs(B, n, C, mixed)
    shifted = []
    for t in phi:
        flat = torch.empty(t.numel() + 1, device="cuda")
        flat[1:].copy_(t.reshape(-1))
        shifted.append(flat[1:].view_as(t))
        assert shifted[-1].data_ptr() % 16 == 4
    for k, (a, b) in enumerate(zip(_forward(x, w, phi, small), _forward(x, w, shifted, small))):
        assert torch.equal(a.nan_to_num(1e30), b.nan_to_num(1e30)), k


@pytest.mark.parametrize("dynamic", [True, False])
@pytest.mark.parametrize("B,n,C", [(5, 4, 64), (900, 4, 72), (9, 8, 136), (6, 32, 64), (4, 3, 37)])
def test_weight_gradient_in_bfloat16_is_the_rounded_float32_one(dynamic, B, n, C):
    from mhc import MHCLayer

    torch.manual_seed(11)
    layer = MHCLayer(C, n, use_dynamic_h=dynamic, output_dtype=torch.bfloat16).cuda()
    x = torch.randn(B, n, C, device="cuda").bfloat16()
    dy = torch.randn(B, n, C, device="cuda").bfloat16()
    layer(x).backward(dy)
    g16 = layer.rmsnorm_weight.grad.clone()
    layer.rmsnorm_weight = torch.nn.Parameter(layer.rmsnorm_weight.detach().float())
    layer(x).backward(dy)
    g32 = layer.rmsnorm_weight.grad
    assert g16.dtype == torch.bfloat16 and g32.dtype == torch.float32
    assert torch.equal(g16, g32.bfloat16())

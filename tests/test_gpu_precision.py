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


# ragged rows; rows of more than 2560 channels; n = 5 .. 8 with rows of at most 512, with and without a split batch; n <= 4 and
# more than 768 samples; the slab kernels (n <= 4 with 64 and 128 channels per workgroup; n = 5 .. 8 beyond the batches of which the
# resident path rounds 513 .. 2560 channels twice)
@pytest.mark.parametrize("B,n,C", [(65, 4, 203), (40, 8, 77), (33, 3, 2701), (20, 4, 2568), (9, 8, 4096), (300, 2, 2816),
                                   (1100, 5, 264), (1030, 8, 512), (2100, 7, 64), (40, 8, 512), (1100, 6, 520),
                                   (900, 4, 520), (1000, 3, 392), (900, 4, 128), (1600, 3, 256), (2000, 2, 64), (780, 4, 264)])
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



def _batch_and_single_sums(B, n, C, act, lib=None):
    """dw, dbias and dalpha of one backward call over B samples, and of B calls over one sample each on the same saved
    state, whose results are the terms of those sums; every sample comes twice, with dy and with -dy, in random order,
    so that the sums are far smaller than what is added up on the way."""
    from mhc import _lib
    lib, D, dev = _lib.lib if lib is None else lib, n * n + 2 * n, "cuda"
    x, dy, p = _dynamic(B // 2, n, C)
    order = torch.randperm(B, generator=torch.Generator().manual_seed(6))
    x, dy = torch.cat([x, x])[order].to(dev, act), torch.cat([dy, -dy])[order].to(dev, act)
    phi = torch.cat([p["phi_pre"], p["phi_post"], p["phi_res"]]).to(dev, act)
    bias = torch.cat([p["b_pre"], p["b_post"], p["b_res"].reshape(-1)]).to(dev)
    alpha, w = torch.full((3,), 0.1, device=dev), p["w"].to(dev)
    code = _lib.dtype_code(x)
    empty = lambda *s: torch.full(s, float("nan"), device=dev)
    H_pre, H_post, M, P, r, q = empty(B, n), empty(B, n), empty(B, n, n), empty(B, D), empty(B), empty(B)
    sk = empty(B, lib.mhc_layer_sinkhorn_state_floats(1, n, T))
    y, dx = torch.empty_like(x), torch.empty_like(x)
    size = lib.mhc_layer_dynamic_workspace_bytes(B, n, C)
    ws, stream = _lib.workspace(x.device, size), _lib.stream_ptr(x.device)
    at = _lib.ptr
    _lib.check("fwd", lib.mhc_layer_fwd_dynamic(at(x), code, at(w), 0, at(phi), code, at(bias), at(alpha), None, at(y), code,
                                                at(H_pre), at(H_post), at(M), at(P), at(r), at(q), at(sk), B, n, C, T, EPS,
                                                at(ws), ws.numel(), stream))

    def backward(i, count, out):
        dw, db = out[:C], out[C:]
        _lib.check("bwd", lib.mhc_layer_bwd_dynamic(
            at(dy[i]), code, at(x[i]), code, at(w), 0, at(phi), code, at(bias), at(alpha), None, at(H_pre[i]), at(H_post[i]),
            at(M[i]), at(P[i]), at(r[i:]), at(q[i:]), at(sk[i]), at(dx[i]), None, at(dw), at(dphi), at(db), at(db[D:]), count,
            n, C, T, EPS, at(ws), ws.numel(), stream))

    dphi, whole, terms = empty(D, n * C), empty(C + D + 3), empty(B, C + D + 3)
    backward(0, B, whole)
    for i in range(B):
        backward(i, 1, terms[i])
    torch.cuda.synchronize()
    return whole.double(), terms.double()


# The sums are float64 and rounded to float32 at the end; parts of 128 samples in float32 would be off by 1e-7 of the
# parts, thousands of times this bound.
def _close_to_float64(whole, terms):
    total = terms.sum(0)
    off, bound = (whole - total).abs(), 2.0 ** -23 * total.abs() + 2.0 ** -45 * terms.abs().sum(0)
    assert torch.isfinite(whole).all() and (off <= bound).all(), float((off / bound.clamp_min(1e-300)).max())


@pytest.mark.parametrize("B,n,C", [(1536, 8, 64), (2050, 6, 16), (1794, 2, 44), (1600, 7, 48), (1922, 4, 42)])
def test_split_batch_sums_stay_in_float64(B, n, C):
    _close_to_float64(*_batch_and_single_sums(B, n, C, torch.bfloat16))


# The bf16 slab kernels (n <= 4 with 64 and 128 channels per workgroup, n = 5 .. 8): up to 128 tiles of 16 samples per batch split,
# so that a float32 sum over the tiles of a lane would be off by some 2^-24 of what is added up on the way, a million times the bound.
@pytest.mark.parametrize("B,n,C,width,splits", [(2050, 4, 264, 1, 1), (1100, 4, 136, 2, 2), (1500, 3, 64, 2, 1), (1026, 1, 72, 1, 2),
                                                (1100, 8, 264, 0, 1), (1500, 5, 72, 0, 2), (700, 7, 64, 0, 1)])
def test_slab_sums_stay_in_float64(B, n, C, width, splits):
    from mhc._lib import tuning_lib

    lib = tuning_lib()
    # the tiled path; one launch of channel sums and coefficient backward, as for one sample; the slab kernel (n = 5 .. 8) for one
    # sample too; slab width and splits
    hooks = {7: 1, 2: 2, 12: 2, 11: width, 3: splits}
    try:
        for k, v in hooks.items():
            assert lib.mhc_tuning_set(k, v) == 0
        _close_to_float64(*_batch_and_single_sums(B, n, C, torch.bfloat16, lib))
    finally:
        for k in hooks:
            lib.mhc_tuning_set(k, 0)


@pytest.mark.parametrize("B,n,C", [(640, 4, 64), (770, 3, 36), (300, 1, 96), (1030, 2, 130), (2, 4, 8), (18, 4, 512)])
def test_float32_slab_sums_stay_in_float64(B, n, C):
    _close_to_float64(*_batch_and_single_sums(B, n, C, torch.float32))


# Row tiles of phi in workgroups of their own: the sums that eight waves form.  Four waves with chains twice as long were off by
# 2.2e-7 and 2.0e-7 in these shapes, eight are by 1.73e-7 and 1.74e-7 (seeds scatter by 1e-9).
@pytest.mark.parametrize("B,n,C,most", [(600, 6, 1024, 1.95e-7), (100, 8, 1280, 1.86e-7)])
def test_float32_projection_in_row_groups(B, n, C, most):
    import bench

    st = bench.Step(dict(kind="dynamic", B=B, n=n, C=C, dtype="f32", bwd=False), "L", torch)
    st.forward()
    x, p = st.host["x"].double().reshape(B, -1), st.host["p"]
    phi = torch.cat([p["phi_pre"], p["phi_post"], p["phi_res"]]).double()
    want = x @ phi.T / (x.square().mean(1, keepdim=True) + bench.EPS).sqrt()
    assert rel2(st.P.cpu(), want) <= most, rel2(st.P.cpu(), want)


# n = 4: a sum of six terms and a product of depth 24, about 9e-8; with every step of the product rounded at the size of
# dx 1.5e-7
@pytest.mark.parametrize("B,n,C", [(65, 4, 128), (40, 4, 514), (100, 3, 66)])
def test_float32_dx_adds_the_projection_term_once(B, n, C):
    x, dy, p = _dynamic(B, n, C, bf16_weight=False)
    _, ref = nm.mhc_dynamic_fwd_bwd(x, p, dy, T, EPS, dtype=torch.float64)
    _, got = hip_dynamic(x, p, dy, T, EPS)
    assert rel2(got["x"], ref["x"]) <= 1.15e-7, rel2(got["x"], ref["x"])

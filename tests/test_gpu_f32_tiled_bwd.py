"""Float32 storage of bf16 arithmetic, the tiled backward (channel sums that leave x and dy in bf16 where dx will be, then the
slab kernel): against the sample-resident backward on the same inputs and against float64, over rows that end in the middle of
a step, batches on either side of a tile, of a workgroup's samples and of a split, and both types of the weight.

Both backwards round x, dy and dP phi's operands alike and compute in float32 behind that: they differ by the order of float32
sums and by coefficients of 1 ulp, 2e-5 of the largest value at most.  In dx a dP that lies next to a rounding boundary may
become either of two bf16 neighbours: 2^-8 of its product with a phi of up to 0.1, a few of at most 80 at once, against a largest dx of
several units, 2e-4 of it."""
import pytest
import torch

from helpers import rel_err

pytestmark = pytest.mark.gpu

T, EPS = 20, 1e-6
K_GRAM, K_RESIDENT = 2, 7
F32_AS_BF16 = 2


@pytest.fixture(autouse=True)
def _reset_tuning():
    from mhc._lib import tuning_lib

    yield
    for k in (K_GRAM, K_RESIDENT):
        tuning_lib().mhc_tuning_set(k, 0)


def _inputs(B, n, C, wt):
    g = torch.Generator(device="cuda").manual_seed(B + n + C)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    D = n * n + 2 * n
    return dict(x=rn(B, n, C), dy=rn(B, n, C), w=(1 + 0.1 * rn(C)).to(wt), phi=(0.02 * rn(D, n * C)).bfloat16(), bias=0.5 * rn(D),
                alpha=torch.tensor([0.3, 0.4, 0.5], device="cuda"))


def _run(v, resident, gram=0):
    from mhc import _lib
    from mhc._lib import check, dtype_code, ptr

    lib = _lib.tuning_lib()
    assert lib.mhc_tuning_set(K_RESIDENT, resident) == 0 and lib.mhc_tuning_set(K_GRAM, gram) == 0
    x = v["x"]
    B, n, C = x.shape
    D, f32 = n * n + 2 * n, dict(device="cuda")
    y, Hp, Ho, M = torch.empty_like(x), torch.empty(B, n, **f32), torch.empty(B, n, **f32), torch.empty(B, n, n, **f32)
    P, r, q = torch.empty(B, D, **f32), torch.empty(B, **f32), torch.empty(B, **f32)
    sk = torch.empty(lib.mhc_layer_sinkhorn_state_floats(B, n, T), **f32)
    ws = torch.full((lib.mhc_layer_dynamic_workspace_bytes(B, n, C),), 0xFF, dtype=torch.uint8, device="cuda")
    st = _lib.stream_ptr(x.device)
    check("mhc_layer_fwd_dynamic",
          lib.mhc_layer_fwd_dynamic(ptr(x), F32_AS_BF16, ptr(v["w"]), dtype_code(v["w"]), ptr(v["phi"]), dtype_code(v["phi"]),
                                    ptr(v["bias"]), ptr(v["alpha"]), None, ptr(y), dtype_code(y), ptr(Hp), ptr(Ho), ptr(M), ptr(P),
                                    ptr(r), ptr(q), ptr(sk), B, n, C, T, EPS, ptr(ws), ws.numel(), st))
    nan = lambda *s: torch.full(s, float("nan"), device="cuda")
    dx = nan(B + 1, n, C)  # one sample more: nothing may be written there
    out = dict(dw=nan(C), dphi=nan(D, n * C), dbias=nan(D), dalpha=nan(3))
    check("mhc_layer_bwd_dynamic",
          lib.mhc_layer_bwd_dynamic(ptr(v["dy"]), dtype_code(v["dy"]), ptr(x), F32_AS_BF16, ptr(v["w"]), dtype_code(v["w"]),
                                    ptr(v["phi"]), dtype_code(v["phi"]), ptr(v["bias"]), ptr(v["alpha"]), None, ptr(Hp), ptr(Ho),
                                    ptr(M), ptr(P), ptr(r), ptr(q), ptr(sk), ptr(dx), None, ptr(out["dw"]), ptr(out["dphi"]),
                                    ptr(out["dbias"]), ptr(out["dalpha"]), B, n, C, T, EPS, ptr(ws), ws.numel(), st))
    torch.cuda.synchronize()
    assert torch.isnan(dx[B]).all(), "wrote behind the batch"
    out["dx"] = dx[:B]
    return out


@pytest.mark.parametrize("wt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,C", [(1, 64), (1, 640), (2, 192), (2, 4096), (3, 128), (3, 320), (4, 64), (4, 1344), (4, 2560),
                                 (5, 64), (5, 1088), (6, 192), (6, 1536), (7, 64), (7, 448), (8, 128), (8, 1344)])
def test_same_as_the_resident_backward(n, C, wt):
    for B, gram in ((1, 0), (15, 0), (17, 2), (66, 0), (131, 2)):  # gram 2: several samples per workgroup (n <= 4)
        v = _inputs(B, n, C, wt)
        want, got = _run(v, 2), _run(v, 1, gram)
        for k in want:
            assert torch.isfinite(got[k]).all(), (B, k)
            # the three dalpha and the biases' rows: sums over the batch of terms of both signs
            e = rel_err(got[k].cpu(), want[k].cpu())
            assert e <= {"dalpha": 1e-3, "dx": 2e-4}.get(k, 2e-5), (B, k, e)


@pytest.mark.parametrize("B,n,C", [(1701, 4, 320), (1150, 3, 512), (4100, 4, 256), (1000, 2, 1024), (963, 5, 576), (1001, 6, 640),
                                   (1001, 7, 512), (1029, 8, 1024), (1721, 8, 1024)])  # (n = 1: dHpre is the difference of equal sums)
def test_through_the_module(B, n, C):
    """Sizes at which the layer takes this path by itself (the last one with a wave per sample for the channel sums)."""
    import mhc
    from mhc._lib import tuning_lib
    from oracle import naive_mhc as nm

    assert tuning_lib().mhc_tuning_route(0, F32_AS_BF16, B, n, C) == 1
    torch.manual_seed(2)
    with torch.device("cuda"):
        layer = mhc.MHCLayer(C, n, compute_dtype=torch.bfloat16)
        with torch.no_grad():
            for p in (layer.b_pre, layer.b_post, layer.b_res):
                p.normal_(0.0, 0.5)
            for a in (layer.alpha_pre, layer.alpha_post, layer.alpha_res):
                a.fill_(0.3)
            for p in (layer.phi_pre, layer.phi_post, layer.phi_res):
                p.copy_(p.bfloat16())
        x = torch.randn(B, n, C).requires_grad_(True)
        dy = torch.randn(B, n, C)
    y = layer(x)
    y.backward(dy)
    torch.cuda.synchronize()
    params = {k: getattr(layer, k).detach().double() for k in nm.DYN_PARAM_NAMES if k != "w"}
    params["w"] = layer.rmsnorm_weight.detach().double()
    y_ref, g_ref = nm.mhc_dynamic_fwd_bwd(x.detach().bfloat16().double(), params, dy.bfloat16().double(), layer.sinkhorn_iters, layer.eps,
                                          dtype=torch.float64)
    rel = lambda a, b: float((a.double() - b.to(a.device)).norm() / b.norm())
    assert rel(y.detach(), y_ref) <= 1e-5
    # dP phi is a product of bf16 operands (2^-9 of a term that is a part of dx), dw leaves in bf16 (2^-8)
    assert rel(x.grad, g_ref["x"]) <= 1e-3
    assert rel(layer.rmsnorm_weight.grad, g_ref["w"]) <= 2.0 ** -8
    for k in ("phi_pre", "phi_post", "phi_res", "b_pre", "b_post", "b_res"):
        assert rel(getattr(layer, k).grad, g_ref[k]) <= 1e-4, k

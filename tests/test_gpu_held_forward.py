"""The dynamic forward that keeps sixteen samples per workgroup in registers (layer_fwd_held.hip), n = 2 .. 4: every output
against float64 of the operands as the kernel sees them, over the row lengths at which another number of chunks or waves
is chosen and batches on either side of a tile, of one round of workgroups and of a balanced second round.

Bounds: the float32 outputs are sums of at most 10240 products (pairwise between waves) behind hardware or library
functions of 1 ulp, far below 1e-5 of the largest value; a bfloat16 y is rounded once (half a unit of
8 significant bits, 2^-8 of the value at most) and mixed with coefficients that keep 16 bits (2^-16 of the sum of the terms)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

T, EPS = 20, 1e-6
K_FORWARD = 0
BF16, F32, F32_AS_BF16 = "bf16", "f32", "f32 as bf16"


@pytest.fixture(autouse=True)
def _reset_tuning():
    from mhc._lib import tuning_lib

    yield
    tuning_lib().mhc_tuning_set(K_FORWARD, 0)


def _inputs(kind, B, n, C, seed=0, wt=None):
    g = torch.Generator(device="cuda").manual_seed(seed + B + n + C)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    act = torch.bfloat16 if kind == BF16 else torch.float32
    pt = torch.float32 if kind == F32 else torch.bfloat16
    D = n * n + 2 * n
    return dict(x=rn(B, n, C).to(act), w=(1 + 0.1 * rn(C)).to(wt or pt), phi=(0.02 * rn(D, n * C)).to(pt), bias=0.5 * rn(D),
                alpha=torch.tensor([0.3, 0.4, 0.5], device="cuda"))


def _reference(kind, v, T=T):
    x = v["x"].bfloat16().double() if kind == F32_AS_BF16 else v["x"].double()
    B, n, C = x.shape
    al, b = v["alpha"].double(), v["bias"].double()
    r = (x.reshape(B, -1).square().mean(1) + EPS).sqrt()
    P = x.reshape(B, -1) @ v["phi"].double().t() / r[:, None]
    Hp = torch.sigmoid(al[0] * P[:, :n] + b[:n])
    Ho = 2 * torch.sigmoid(al[1] * P[:, n:2 * n] + b[n:2 * n])
    M = torch.exp(al[2] * P[:, 2 * n:] + b[2 * n:]).reshape(B, n, n)
    sk = []
    for _ in range(T):
        rho = M.sum(2) + EPS
        M = M / rho[:, :, None]
        s = M.sum(1) + EPS
        M = M / s[:, None, :]
        sk.append(torch.stack([rho, s], 1))
    a = (Hp[:, :, None] * x).sum(1)
    q = (a.square().mean(1) + EPS).sqrt()
    y = (M[:, :, :, None] * x[:, None]).sum(2) + Ho[:, :, None] * (a / q[:, None] * v["w"].double())[:, None]
    return dict(P=P, r=r, Hp=Hp, Ho=Ho, M=M, q=q, y=y, **(dict(sk=torch.stack(sk, 1)) if T else {}))


def _forward(kind, v, hook=3, T=T, state=True):
    from mhc import _lib
    from mhc._lib import check, dtype_code, ptr

    lib = _lib.tuning_lib()
    assert lib.mhc_tuning_set(K_FORWARD, hook) == 0
    x = v["x"]
    B, n, C = x.shape
    D, NP = n * n + 2 * n, 4
    shapes = dict(y=(n, C), Hp=(n,), Ho=(n,), M=(n, n), P=(D,), r=(), q=(), sk=(T + 1, 2, NP))
    # one more row behind the batch: nothing may be written there
    out = {k: torch.full((B + 1, *s), float("nan"), device="cuda", dtype=x.dtype if k == "y" else torch.float32)
           for k, s in shapes.items()}
    ws = torch.empty(lib.mhc_layer_dynamic_workspace_bytes(B, n, C), dtype=torch.uint8, device="cuda")
    code = 2 if kind == F32_AS_BF16 else dtype_code(x)
    check("mhc_layer_fwd_dynamic",
          lib.mhc_layer_fwd_dynamic(ptr(x), code, ptr(v["w"]), dtype_code(v["w"]), ptr(v["phi"]), dtype_code(v["phi"]),
                                    ptr(v["bias"]), ptr(v["alpha"]), None, ptr(out["y"]), dtype_code(out["y"]), ptr(out["Hp"]),
                                    ptr(out["Ho"]), ptr(out["M"]), ptr(out["P"]), ptr(out["r"]), ptr(out["q"]), ptr(out["sk"]) if state else None,
                                    B, n, C, T, EPS, ptr(ws), ws.numel(), _lib.stream_ptr(x.device)))
    torch.cuda.synchronize()
    assert all(torch.isnan(t[B]).all() for t in out.values()), "wrote behind the batch"
    out = {k: t[:B] for k, t in out.items()}
    out["sk"] = out["sk"][:, :T, :, :n]
    return out


def _check(kind, got, ref):
    for k, v in ref.items():
        o = got[k].double()
        assert torch.isfinite(o).all(), k
        if k == "y" and kind == BF16:
            assert ((o - v).abs() <= 2.0 ** -8 * v.abs() + 2.0 ** -16 * v.abs().max()).all()
        else:
            e = float((o - v).abs().max() / v.abs().max())
            assert e <= 1e-5, f"{k}: {e:.2e}"


# rows: the shortest, one and two chunks, a wave's chunks filled and not, four and eight waves, the longest
SHAPES = [(4, 64), (4, 192), (4, 256), (4, 320), (4, 576), (4, 1280), (4, 1344), (4, 2560), (3, 64), (3, 832), (3, 1536), (3, 1600),
          (3, 3072), (2, 64), (2, 640), (2, 2560), (2, 2624), (2, 4096)]


@pytest.mark.parametrize("kind", [BF16, F32, F32_AS_BF16])
@pytest.mark.parametrize("n,C", SHAPES)
def test_every_output(kind, n, C):
    if kind == F32:
        C //= 2  # chunks of 32 channels
    for B in (1, 16, 53):
        v = _inputs(kind, B, n, C)
        _check(kind, _forward(kind, v), _reference(kind, v))


@pytest.mark.parametrize("kind", [BF16, F32, F32_AS_BF16])
@pytest.mark.parametrize("B,n,C", [(4096, 4, 1344), (4097, 4, 1344), (4500, 4, 1344), (7000, 4, 1344), (12500, 2, 640)])
def test_several_rounds(kind, B, n, C):
    """One tile per workgroup, and several: tiles of fewer samples where the last round would be nearly empty."""
    if kind == F32:
        C //= 2
    v = _inputs(kind, B, n, C)
    _check(kind, _forward(kind, v), _reference(kind, v))


@pytest.mark.parametrize("kind", [BF16, F32, F32_AS_BF16])
@pytest.mark.parametrize("n,C", [(4, 64), (4, 1344), (3, 832), (2, 2624)])
def test_without_saved_state(kind, n, C):
    """As inference calls it: the same results bit for bit, and nothing is written where a state would be."""
    if kind == F32:
        C //= 2
    for B in (1, 53):
        v = _inputs(kind, B, n, C)
        want, got = _forward(kind, v), _forward(kind, v, state=False)
        assert torch.isnan(got.pop("sk")).all()
        for k in got:
            assert torch.equal(got[k], want[k]), k
        _check(kind, {**got, "sk": want["sk"]}, _reference(kind, v))


@pytest.mark.parametrize("kind", [BF16, F32, F32_AS_BF16])
@pytest.mark.parametrize("iters", [0, 1, 32])
@pytest.mark.parametrize("state", [True, False])
def test_sinkhorn_iterations(kind, iters, state):
    for n, C in ((4, 320), (3, 64), (2, 192)):
        v = _inputs(kind, 35, n, C)
        ref = _reference(kind, v, iters)
        if not state:
            ref.pop("sk", None)
        _check(kind, _forward(kind, v, T=iters, state=state), ref)


@pytest.mark.parametrize("kind", [BF16, F32, F32_AS_BF16])
def test_the_other_type_of_weight(kind):
    for n, C in ((4, 1344), (3, 192), (2, 2624)):
        v = _inputs(kind, 37, n, C, wt=torch.bfloat16 if kind == F32 else torch.float32)
        _check(kind, _forward(kind, v), _reference(kind, v))


def test_samples_are_independent():
    """A sample of infinities and one of NaN leave the others of their tile as they were, bit for bit."""
    v = _inputs(BF16, 40, 3, 192)
    want = _forward(BF16, v)
    v["x"][5], v["x"][21] = float("inf"), float("nan")
    got = _forward(BF16, v)
    keep = [b for b in range(40) if b not in (5, 21)]
    for k in want:
        assert torch.equal(got[k][keep], want[k][keep]), k


@pytest.mark.parametrize("dtype,B,n,C", [(torch.bfloat16, 4200, 4, 384), (torch.bfloat16, 4100, 2, 128), (torch.float32, 1111, 2, 96), (torch.float32, 1100, 3, 64)])
def test_through_the_module(dtype, B, n, C):
    """Sizes at which the layer takes this path by itself: the packed parameters that it leaves serve the backward.  And as inference
    calls it, without a state to keep: the same y."""
    import mhc
    from mhc._lib import tuning_lib
    from oracle import naive_mhc as nm

    assert tuning_lib().mhc_tuning_route(1, 1 if dtype == torch.bfloat16 else 0, B, n, C) == 3
    torch.manual_seed(1)
    with torch.device("cuda"):
        layer = mhc.MHCLayer(C, n, output_dtype=dtype if dtype == torch.bfloat16 else None)
        with torch.no_grad():
            for p in (layer.b_pre, layer.b_post, layer.b_res):
                p.normal_(0.0, 0.5)
            for a in (layer.alpha_pre, layer.alpha_post, layer.alpha_res):
                a.fill_(0.3)
            for p in (layer.phi_pre, layer.phi_post, layer.phi_res):
                p.copy_(p.bfloat16())
        x = torch.randn(B, n, C, dtype=dtype).requires_grad_(True)
        dy = torch.randn(B, n, C, dtype=dtype)
    y = layer(x)
    y.backward(dy)
    with torch.no_grad():
        assert torch.equal(layer(x), y)
    torch.cuda.synchronize()
    params = {k: getattr(layer, k).detach().double() for k in nm.DYN_PARAM_NAMES if k != "w"}
    params["w"] = layer.rmsnorm_weight.detach().double()
    y_ref, g_ref = nm.mhc_dynamic_fwd_bwd(x.detach().double(), params, dy.double(), layer.sinkhorn_iters, layer.eps, dtype=torch.float64)
    bar = 1e-5 if dtype == torch.float32 else 1e-2
    rel = lambda a, b: float((a.double() - b.to(a.device)).norm() / b.norm())
    assert rel(y.detach(), y_ref) <= bar
    assert rel(x.grad, g_ref["x"]) <= bar
    for k in ("phi_pre", "phi_post", "phi_res", "b_pre", "b_post", "b_res"):
        assert rel(getattr(layer, k).grad, g_ref[k]) <= bar, k

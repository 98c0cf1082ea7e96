"""The backward with shared coefficients (bf16, n <= 8) from its two kernels, one sample per workgroup or several walked by one,
forced through the experiment hook, at sizes where the second one's waves, chunks and rounds end: each against the oracle and
against each other.

Tolerances: the bf16 tier of test_gpu_parity.py against the oracle (float32 on the bf16-rounded inputs).  Between the kernels dx
and df are the same operations in the same order (up to contraction of a product with a sum: one bf16 rounding, 2^-8); the sums
over samples are float32 terms added in float64 on both sides: 1e-5 of the largest entry."""
import pytest
import torch

from helpers import rel_err
from oracle import naive_mhc as nm

pytestmark = pytest.mark.gpu

K_SPG, T_ITERS, EPS = 6, 20, 1e-6


# (rounds 0: as the library chooses, above its lines, cut workgroups and chunks among them.)
# waves per workgroup: 2 (n <= 4, C <= 256), 4, 8 (C > 2560; n > 4: C > 1024); 3 samples make a last round that is not full
@pytest.mark.parametrize("B,n,C,rounds", [(2, 4, 8, 2), (7, 3, 256, 3), (5, 1, 264, 2), (9, 2, 513, 4), (33, 4, 1024, 5), (20, 4, 1288, 3),
                                          (11, 4, 2048, 4), (13, 4, 2560, 6), (10, 3, 2555, 3), (7, 4, 2568, 2), (6, 2, 4096, 5),
                                          (5, 4, 3333, 2), (9, 8, 64, 3), (12, 5, 520, 4), (10, 7, 1023, 3), (7, 8, 1032, 2),
                                          (9, 6, 2048, 4), (5, 8, 2056, 2), (6, 5, 3080, 3), (5, 8, 4093, 2), (4, 8, 4096, 4),
                                          (4101, 2, 72, 0), (3073, 4, 264, 0), (515, 4, 2568, 0), (2051, 8, 520, 0), (769, 5, 3080, 0)])
@pytest.mark.parametrize("inject", [False, True])
@pytest.mark.parametrize("w_f32", [False, True])
def test_one_and_several_samples_per_workgroup(B, n, C, rounds, inject, w_f32):
    if inject and w_f32:
        pytest.skip("w is unused with an injected f")
    import bench
    from mhc._lib import tuning_lib

    lib = tuning_lib()
    st = bench.Step(dict(kind="static", B=B, n=n, C=C, dtype="bf16", bwd=True), "K" if inject else "L", torch, lib=lib)
    g = torch.Generator().manual_seed(B * 7 + n * 131 + C)
    p = st.host["p"]
    p["w"] = 1.0 + 0.3 * torch.randn(C, generator=g)
    if not w_f32:
        p["w"] = p["w"].bfloat16().float()
    for i, (k, shape) in enumerate((("H_pre", (n,)), ("H_post", (n,)), ("H_res", (n, n)))):
        p[k] = torch.randn(*shape, generator=g)
        st.Hl[i].copy_(p[k])
    st.w = p["w"].to(torch.float32 if w_f32 else torch.bfloat16).cuda()
    h = st.host
    y_ref, g_ref = nm.mhc_static_fwd_bwd(h["x"], p, h["dy"], T_ITERS, EPS, f_inject=h["f"], dtype=torch.float32)
    ref = dict(dx=g_ref["x"], dH_post=g_ref["H_post"], dH_res=g_ref["H_res"])
    ref.update(dict(df=g_ref["f"]) if inject else dict(dw=g_ref["w"], dH_pre=g_ref["H_pre"]))
    st.forward()
    got = []
    try:
        for spg in (1, rounds):
            assert lib.mhc_tuning_set(K_SPG, spg) == 0
            for t in [st.dx, st.dw] + st.dH + ([st.df] if inject else []):
                t.fill_(float("nan"))
            st.ws.fill_(255)
            st.backward()
            torch.cuda.synchronize()
            o = dict(dx=st.dx, dH_pre=st.dH[0], dH_post=st.dH[1], dH_res=st.dH[2])
            o.update(dict(df=st.df) if inject else dict(dw=st.dw))
            got.append({k: v.float().cpu() for k, v in o.items()})
    finally:
        lib.mhc_tuning_set(K_SPG, 0)
    for o in got:
        assert not inject or not o["dH_pre"].any()
        for k, r in ref.items():
            assert torch.isfinite(o[k]).all(), k
            if n == 1 and not inject and k == "dH_pre":
                continue  # one stream: O(eps), compared between the kernels below
            assert rel_err(o[k], r) <= 2e-2, (k, rel_err(o[k], r))
    for k in ref:
        e = rel_err(got[1][k], got[0][k])
        small = n == 1 and k == "dH_pre"  # a difference of two equal sums: bounded against the summands instead
        assert e <= (2.0 ** -8 if k in ("dx", "df") else 1e-5) or (small and (got[1][k] - got[0][k]).abs().max() <= 1e-5 * B * C), (k, e)

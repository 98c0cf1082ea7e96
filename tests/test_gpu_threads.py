"""Several host threads on one stream: the launches of one call must not come in between those of another, since the
calls of a stream share its scratch memory (projection sums, coefficients, the packed parameters of a forward without
gradients).  Each thread has its own layer and input, so a mixed-up call gives another thread's numbers."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("train", [False, True])
def test_threads_on_one_stream_do_not_mix(train):
    from mhc import MHCLayer
    work = []
    for i, (B, n, C) in enumerate([(7, 4, 512), (64, 4, 512), (33, 8, 256), (5, 12, 128)]):
        torch.manual_seed(i)
        layer, x = MHCLayer(C, n).cuda(), torch.randn(B, n, C, device="cuda")

        def call(layer=layer, x=x):
            if not train:
                with torch.no_grad():
                    return [layer(x)]
            xg = x.clone().requires_grad_(True)
            y = layer(xg)
            return [y.detach()] + list(torch.autograd.grad(y, [xg, *layer.parameters()], torch.ones_like(y)))

        work.append((call, call()))
    torch.cuda.synchronize()
    bad, start = [], threading.Barrier(len(work))

    def loop(k):
        call, want = work[k]
        start.wait()
        for _ in range(60):
            got = call()
            if not all(torch.equal(a, b) for a, b in zip(got, want)):
                bad.append(k)
                return

    threads = [threading.Thread(target=loop, args=(k,)) for k in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, f"thread {bad} got another call's values"

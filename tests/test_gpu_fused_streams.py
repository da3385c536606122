"""GPU: plans that run as persistent launches (a C2C batch, realft, an uneven
batch, correl), executing at the same time on streams of their own, give what
they give one after the other, bit by bit."""
import pytest

import numrs_amd
from numrs_amd import synth

pytestmark = pytest.mark.gpu


def test_persistent_plans_on_several_streams():
    import torch

    def real(n, seed):
        x = torch.empty(n, dtype=torch.float32, device="cuda")
        numrs_amd.gen_uniform(x, seed)
        return x

    jobs = []
    n, b = 1 << 20, 27
    c2c, cx = numrs_amd.C2CPlan("float32", [n], b), real(2 * n * b, 1)
    cy = torch.empty_like(cx)
    jobs.append((lambda s: c2c.execute(cx, cy, 1, stream=s), cy))
    rft, rx0 = numrs_amd.RealFTPlan("float32", 1 << 18, 90), real((1 << 18) * 90, 2)
    rx = rx0.clone()

    def there_and_back(s):
        with torch.cuda.stream(s):
            rx.copy_(rx0)
        rft.execute(rx, 1, stream=s)
        rft.execute(rx, -1, stream=s)

    jobs.append((there_and_back, rx))
    items = synth.uneven_shapes(7, 90)
    un = numrs_amd.UnevenPlan("float32", items)
    ux = real(2 * un.total, 3)
    uy = torch.empty_like(ux)
    jobs.append((lambda s: un.execute(ux, uy, -1, stream=s), uy))
    cor, da, db = numrs_amd.CorrelPlan("float32", 1 << 17, 140), real((1 << 17) * 140, 4), real((1 << 17) * 140, 5)
    ca = torch.empty_like(da)
    jobs.append((lambda s: cor.execute(da, db, ca, stream=s), ca))

    streams = [torch.cuda.Stream() for _ in jobs]
    want = []
    for (run, out), s in zip(jobs, streams):
        run(s)
        torch.cuda.synchronize()
        want.append(out.clone())
        out.fill_(float("nan"))
    torch.cuda.synchronize()
    for rep in range(4):
        print(f"streams rep {rep}", flush=True)
        for _ in range(3):
            for (run, _), s in zip(jobs, streams):
                run(s)
        torch.cuda.synchronize()
        for k, ((_, out), w) in enumerate(zip(jobs, want)):
            assert torch.equal(out, w), (rep, k)
            out.fill_(float("nan"))
        torch.cuda.synchronize()
    un.check()

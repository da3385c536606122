"""GPU: correl with both spectra in one persistent launch and the product with
its inverse in another, at the smallest batch that takes it and one more, with
places in the ring used again, and with the result written over either input,
against the plan of one pair (which runs in passes) and numpy in FP64.

Tolerances: a transform of n reals is within 2 eps log2 n of exact, 3e-6 (FP32)
and 1e-14 (FP64) at these lengths; a correlation is three of them and a product,
taken as four, and two forms of it are at most twice that apart: 2.4e-5 and
8e-14 relative L2."""
import numpy as np
import pytest

import numrs_amd

pytestmark = pytest.mark.gpu

TILE = {"float32": 1 << 14, "float64": 1 << 13}
TOL = {"float32": 2.4e-5, "float64": 8e-14}


def _min_batch(dtype, logl):
    return max(1, 512 * TILE[dtype] >> logl)


def _rel(a, b):
    import torch

    return float(torch.linalg.vector_norm(a.double() - b.double()) / torch.linalg.vector_norm(b.double()))


CASES = [(d, l, _min_batch(d, l) + e) for d, lo, hi in (("float32", 15, 20), ("float64", 14, 20))
         for l in range(lo, hi + 1) for e in (0, 1)]
# more slabs than ring slots (192 MiB) in both launches, a short last slab
CASES += [("float32", 15, 771), ("float32", 19, 51), ("float64", 14, 770), ("float64", 19, 25)]


@pytest.mark.parametrize("dtype,logl,batch", CASES)
def test_fused_correl(dtype, logl, batch):
    import torch

    n = 2 << logl
    a = torch.empty(n * batch, dtype=getattr(torch, dtype), device="cuda")
    b, ans = torch.empty_like(a), torch.empty_like(a)
    numrs_amd.gen_uniform(a, 600 + logl)
    numrs_amd.gen_uniform(b, 700 + logl)
    plan, one = numrs_amd.CorrelPlan(dtype, n, batch), numrs_amd.CorrelPlan(dtype, n, 1)
    print(f"fused correl {dtype} 2^{logl} x {batch}: workspace {plan.workspace_bytes}", flush=True)
    for rep in range(2):  # the state is left as it was found
        ans.fill_(float("nan"))
        plan.execute(a, b, ans)
        for i in sorted({0, 1 % batch, batch // 2, batch - 1}):
            seg = slice(n * i, n * (i + 1))
            x, y, ref = a[seg].clone(), b[seg].clone(), torch.empty(n, dtype=a.dtype, device="cuda")
            one.execute(x, y, ref)
            assert _rel(ans[seg], ref) < TOL[dtype], (rep, i)
    fa, fb = (np.fft.rfft(t[:n].double().cpu().numpy()) for t in (a, b))
    want = np.fft.irfft(fa * np.conj(fb), n)
    got = ans[:n].double().cpu().numpy()
    assert np.linalg.norm(got - want) < TOL[dtype] * np.linalg.norm(want)
    for over in (0, 1):
        x, y = a.clone(), b.clone()
        plan.execute(x, y, (x, y)[over])
        assert torch.equal((x, y)[over], ans), over
        assert torch.equal((y, x)[over], (b, a)[over]), over

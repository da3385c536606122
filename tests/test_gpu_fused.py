"""GPU tests of the four-step C2C that runs both passes in one persistent
launch: every length and precision that has such a kernel, at the smallest
batch that takes it, with a last slab that is not full, and with more slabs
than the ring has slots; both signs, in place, on tensors that start at an odd
element, and under graph replay.  Every transform is compared with the
pass-by-pass form of the same plan, some with the oracle.

Tolerances: two FFTs of N points in precision eps differ by at most a few eps
per radix-2 level each, 2 eps log2 N here: 2.5e-6 (FP32, N = 2^21) and 4.5e-15
(FP64, N = 2^20) relative L2, rounded up to 3e-6 and 1e-14; against the oracle
2e-6 and 1e-12 as elsewhere."""
import numpy as np
import pytest

import numrs_amd
import oracle
from conftest import rel_l2
from numrs_amd import synth

pytestmark = pytest.mark.gpu

TILE = {"float32": 1 << 14, "float64": 1 << 13}
TOL = {"float32": 3e-6, "float64": 1e-14}
TOL_ORACLE = {"float32": 2e-6, "float64": 1e-12}


def _min_batch(dtype, logn):
    tiles = 1024 if dtype == "float64" and logn >= 18 else 640
    return max(1, tiles * TILE[dtype] >> logn)


def _rel(a, b):
    import torch

    return float(torch.linalg.vector_norm(a.double() - b.double()) / torch.linalg.vector_norm(b.double()))


def _cases():
    out = []
    for dtype, lo, hi in (("float32", 15, 21), ("float64", 14, 20)):
        for logn in range(lo, hi + 1):
            b = _min_batch(dtype, logn)
            out += [(dtype, logn, b), (dtype, logn, b + 1)]
    # more slabs than ring slots (192 MiB), a short last slab
    out += [("float32", 15, 3077), ("float32", 20, 27), ("float32", 21, 14), ("float64", 14, 773), ("float64", 20, 13)]
    return out


@pytest.mark.parametrize("dtype,logn,batch", _cases())
def test_fused_matches_passes(dtype, logn, batch):
    import torch

    n = 1 << logn
    x = torch.empty(2 * n * batch, dtype=getattr(torch, dtype), device="cuda")
    numrs_amd.gen_uniform(x, 300 + logn)
    plan = numrs_amd.C2CPlan(dtype, [n], batch)
    print(f"fused case {dtype} 2^{logn} x {batch}: workspace {plan.workspace_bytes}", flush=True)
    y, ref = torch.empty_like(x), torch.empty_like(x)
    for isign in (1, -1):
        plan.execute_launches(x, ref, isign, 0, plan.num_launches)
        for _ in range(2):  # the state is left as it was found
            y.fill_(float("nan"))
            plan.execute(x, y, isign)
        worst = max(_rel(y[2 * n * i:2 * n * (i + 1)], ref[2 * n * i:2 * n * (i + 1)])
                    for i in {0, 1 % batch, batch // 2, batch - 1})
        assert worst < TOL[dtype], (isign, worst)
        assert _rel(y, ref) < TOL[dtype], isign
    for i in {0, batch - 1}:
        seg = slice(2 * n * i, 2 * n * (i + 1))
        want = oracle.four1_nr(x[seg].cpu().numpy().astype(np.float64), -1)
        assert rel_l2(y[seg].cpu().numpy().astype(np.float64), want) < TOL_ORACLE[dtype], i
    z = x.clone()
    plan.execute(z, z, -1)
    assert torch.equal(z, y)


@pytest.mark.parametrize("dtype,logn", [("float32", 16), ("float64", 15)])
def test_fused_odd_element_offset(dtype, logn):
    # complex values that start at an odd real element of their buffer
    import torch

    n, batch = 1 << logn, _min_batch(dtype, logn)
    base = torch.empty(2 * n * batch + 1, dtype=getattr(torch, dtype), device="cuda")
    numrs_amd.gen_uniform(base, 21)
    x = base[1:]
    out = torch.zeros(2 * n * batch + 2, dtype=x.dtype, device="cuda")
    plan = numrs_amd.C2CPlan(dtype, [n], batch)
    plan.execute(x, out[1:-1], 1)
    ref = torch.empty(2 * n * batch, dtype=x.dtype, device="cuda")
    plan.execute(x.clone(), ref, 1)
    assert torch.equal(out[1:-1], ref)
    assert out[0] == 0 and out[-1] == 0


def test_fused_graph_replay():
    # captured once, replayed with the program's own eager executions between
    import torch

    dtype, n, batch = "float32", 1 << 18, 48
    x = torch.empty(2 * n * batch, dtype=torch.float32, device="cuda")
    numrs_amd.gen_uniform(x, 5)
    plan = numrs_amd.C2CPlan(dtype, [n], batch)
    y, ref = torch.empty_like(x), torch.empty_like(x)
    plan.execute(x, ref, 1)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        plan.execute(x, y, 1)
    for k in range(4):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref), k
        plan.execute(x, ref, 1)
        torch.cuda.synchronize()


@pytest.mark.parametrize("dtype,n,batch", [("float32", 1 << 17, 160), ("float64", 1 << 16, 161)])
def test_fused_inside_real_plans(dtype, n, batch):
    # convlv in both directions, correl, realft both ways and twofft at sizes
    # whose inner C2C runs as one launch: first, middle and last signal
    # against the oracle (the spectra's direction is not the call's isign).
    import torch

    tdt = getattr(torch, dtype)
    tol = 5 * TOL_ORACLE[dtype]
    idx = (0, batch // 2, batch - 1)
    a = torch.empty(n * batch, dtype=tdt, device="cuda")
    b = torch.empty_like(a)
    numrs_amd.gen_uniform(a, 31)
    numrs_amd.gen_uniform(b, 32)
    m = 65
    r = np.zeros((batch, m))
    r[:, m // 2] = 1.0
    r += 0.002 * synth.uniform(33, batch * m).reshape(batch, m)
    r = r.astype(dtype)
    rt = torch.from_numpy(r.reshape(-1)).cuda()
    ans = torch.empty_like(a)
    plan = numrs_amd.ConvlvPlan(dtype, n, m, batch)

    def seg(t, i, k=n):
        return t[k * i:k * (i + 1)].cpu().numpy().astype(np.float64)

    for isign in (1, -1):
        plan.execute(a, rt, ans, isign)
        for i in idx:
            want = oracle.convlv(seg(a, i), r[i].astype(np.float64), isign)
            assert rel_l2(seg(ans, i), want) < tol, ("convlv", isign, i)
    numrs_amd.CorrelPlan(dtype, n, batch).execute(a, b, ans)
    for i in idx:
        assert rel_l2(seg(ans, i), oracle.correl(seg(a, i), seg(b, i))) < tol, ("correl", i)
    rp = numrs_amd.RealFTPlan(dtype, n, batch)
    for isign in (1, -1):
        z = a.clone()
        rp.execute(z, isign)
        for i in idx:
            assert rel_l2(seg(z, i), oracle.realft(seg(a, i), isign)) < tol, ("realft", isign, i)
    f1 = torch.empty(2 * n * batch, dtype=tdt, device="cuda")
    f2 = torch.empty_like(f1)
    numrs_amd.TwofftPlan(dtype, n, batch).execute(a, b, f1, f2)
    for i in idx:
        for src, f in ((a, f1), (b, f2)):
            z = np.zeros(2 * n)
            z[0::2] = seg(src, i)
            assert rel_l2(seg(f, i, 2 * n), oracle.four1_nr(z, 1)) < tol, ("twofft", i)

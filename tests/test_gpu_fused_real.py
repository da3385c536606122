"""GPU: realft of either direction in one persistent launch, at the smallest
batch that takes it and one more, with places in the ring used again, at an odd
element offset and under graph replay, against the plan of one signal (which
runs in passes) and against numpy in FP64.

Tolerances: two transforms of n reals in precision eps differ by at most a few
eps per radix-2 level each, 2 eps log2 n: 2.6e-6 (FP32, n = 2^22) and 9.4e-15
(FP64, n = 2^21), rounded up to 3e-6 and 1e-14; there and back twice that."""
import numpy as np
import pytest

import numrs_amd

pytestmark = pytest.mark.gpu

TILE = {"float32": 1 << 14, "float64": 1 << 13}
TOL = {"float32": 3e-6, "float64": 1e-14}


def _min_batch(dtype, logl):
    late = 20 if dtype == "float32" else 18
    return max(1, (1024 if logl >= late else 640) * TILE[dtype] >> logl)


def _rel(a, b):
    import torch

    return float(torch.linalg.vector_norm(a.double() - b.double()) / torch.linalg.vector_norm(b.double()))


def _spectrum(x):
    z = np.conj(np.fft.rfft(x))
    out = np.empty_like(x)
    out[0], out[1] = z[0].real, z[-1].real
    out[2::2], out[3::2] = z[1:-1].real, z[1:-1].imag
    return out


def _check(dtype, logl, batch, offset=0):
    import torch

    n = 2 << logl
    buf = torch.empty(n * batch + offset, dtype=getattr(torch, dtype), device="cuda")
    x = buf[offset:]
    numrs_amd.gen_uniform(x if offset == 0 else buf, 500 + logl)
    plan, one = numrs_amd.RealFTPlan(dtype, n, batch), numrs_amd.RealFTPlan(dtype, n, 1)
    print(f"fused real {dtype} 2^{logl} x {batch}: workspace {plan.workspace_bytes}", flush=True)
    x0, keep = x.clone(), buf[:offset].clone()
    picks = sorted({0, 1 % batch, batch // 2, batch - 1})
    for rep in range(2):  # the state is left as it was found
        x.copy_(x0)
        plan.execute(x, 1)
        for i in picks:
            seg = slice(n * i, n * (i + 1))
            ref = x0[seg].clone()
            one.execute(ref, 1)
            assert _rel(x[seg], ref) < TOL[dtype], (rep, i)
    want = _spectrum(x0[:n].double().cpu().numpy())
    assert np.linalg.norm(x[:n].double().cpu().numpy() - want) < TOL[dtype] * np.linalg.norm(want)
    spec = x.clone()
    plan.execute(x, -1)
    for i in picks:
        seg = slice(n * i, n * (i + 1))
        ref = spec[seg].clone()
        one.execute(ref, -1)
        assert _rel(x[seg], ref) < TOL[dtype], i
    assert _rel(x * (2.0 / n), x0) < 2 * TOL[dtype]
    assert torch.equal(buf[:offset], keep)


CASES = [(d, l, _min_batch(d, l) + e) for d, lo, hi in (("float32", 15, 21), ("float64", 14, 20))
         for l in range(lo, hi + 1) for e in (0, 1)]
# more slabs than ring slots (192 MiB), a short last slab
CASES += [("float32", 15, 770), ("float32", 19, 51), ("float32", 21, 14), ("float64", 14, 1541), ("float64", 20, 13)]


@pytest.mark.parametrize("dtype,logl,batch", CASES)
def test_fused_real(dtype, logl, batch):
    _check(dtype, logl, batch)


@pytest.mark.parametrize("dtype,logl", [("float32", 16), ("float64", 15)])
def test_fused_real_odd_offset(dtype, logl):
    _check(dtype, logl, _min_batch(dtype, logl), offset=1)


def test_fused_real_graph_replay():
    import torch

    logl, batch = 17, 130
    n = 2 << logl
    x = torch.empty(n * batch, dtype=torch.float32, device="cuda")
    numrs_amd.gen_uniform(x, 77)
    x0 = x.clone()
    plan = numrs_amd.RealFTPlan("float32", n, batch)
    plan.execute(x, 1)
    want = x.clone()
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        plan.execute(x, 1, stream=s)
        plan.execute(x, -1, stream=s)
        plan.execute(x, 1, stream=s)
    for rep in range(4):
        x.copy_(x0 * (2.0 / n))
        g.replay()
        torch.cuda.synchronize()
        assert _rel(x, want) < 3 * TOL["float32"], rep
        plan.execute(x, -1)  # eager work between replays
        torch.cuda.synchronize()

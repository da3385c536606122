"""GPU: convlv and correl where one group holds one signal (the product is
formed on the halves of each bin pair): the lengths of that form, responses of
1, 2, few and n values, with and without the short-response window, against the
oracle.

Tolerances: three transforms of n reals, each within 2 eps log2 n of exact, and
a product, taken as four: 1.5e-5 (FP32) and 3e-14 (FP64) relative L2."""
import numpy as np
import pytest

import numrs_amd
import oracle
from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = {"float32": 1.5e-5, "float64": 3e-14}


@pytest.mark.parametrize("dtype,n", [("float32", 1 << 13), ("float32", 1 << 14), ("float32", 1 << 15),
                                     ("float64", 1 << 12), ("float64", 1 << 13), ("float64", 1 << 14)])
def test_convlv_halves(dtype, n):
    import torch

    batch = 3
    rng = np.random.default_rng(n)
    x = rng.standard_normal((batch, n)).astype(dtype)
    xt = torch.from_numpy(x.reshape(-1)).cuda()
    for m in (1, 2, 257, 513, n):
        r = rng.standard_normal((batch, m))
        r[:, 1:] *= 0.5 / max(1.0, np.abs(r[:, 1:]).sum(axis=1).max())
        r[:, 0] = 1.0
        r = r.astype(dtype)
        plan = numrs_amd.ConvlvPlan(dtype, n, m, batch)
        rt, y = torch.from_numpy(r.reshape(-1)).cuda(), torch.empty_like(xt)
        plan.execute(xt, rt, y, 1)
        got = y.cpu().numpy().reshape(batch, n).astype(np.float64)
        for i in range(batch):
            want = oracle.convlv(x[i].astype(np.float64), r[i].astype(np.float64), 1)
            assert rel_l2(got[i], want) < TOL[dtype], (m, i)
    z = torch.from_numpy(x[::-1].copy().reshape(-1)).cuda()
    y = torch.empty_like(xt)
    numrs_amd.CorrelPlan(dtype, n, batch).execute(xt, z, y)
    got = y.cpu().numpy().reshape(batch, n).astype(np.float64)
    for i in range(batch):
        want = oracle.correl(x[i].astype(np.float64), x[batch - 1 - i].astype(np.float64))
        assert rel_l2(got[i], want) < TOL[dtype], i

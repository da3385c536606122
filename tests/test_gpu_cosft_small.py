"""GPU: batched cosft1 and cosft2 of the shortest lengths, whose bin pairs a group
enumerates in two ways, with a last group that is not full, against scipy's DCTs.

Tolerances: a transform of 2 n reals in precision eps is within 2 eps log2 2n of
exact, 1.7e-6 (FP32) and 3.1e-15 (FP64) at n = 64: 3e-6 and 6e-15 relative L2."""
import numpy as np
import pytest
import scipy.fft as sfft

import numrs_amd
from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = {"float32": 3e-6, "float64": 6e-15}


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("n", [2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("batch", [1, 1237])
def test_cosft_small(dtype, n, batch):
    import torch

    rng = np.random.default_rng(n + batch)

    def run(plan, width, *args):
        x = rng.standard_normal((batch, width)).astype(dtype)
        t = torch.from_numpy(x.reshape(-1)).cuda()
        y = torch.full_like(t, float("nan"))
        plan.execute(t, y, *args)
        return x.astype(np.float64), y.cpu().numpy().reshape(batch, width).astype(np.float64)

    x, y = run(numrs_amd.Cosft1Plan(dtype, n, batch), n + 1)
    want = 0.5 * sfft.dct(x, type=1)
    assert max(rel_l2(y[i], want[i]) for i in range(batch)) < 4 * TOL[dtype]
    assert rel_l2(y, want) < TOL[dtype]
    plan = numrs_amd.Cosft2Plan(dtype, n, batch)
    for isign, kind in ((1, 2), (-1, 3)):
        x, y = run(plan, n, isign)
        want = 0.5 * sfft.dct(x, type=kind)
        assert max(rel_l2(y[i], want[i]) for i in range(batch)) < 4 * TOL[dtype], isign
        assert rel_l2(y, want) < TOL[dtype], isign

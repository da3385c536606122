"""GPU: convlv and correl of one signal a group over the range of FP32: a response
(second signal) near the smallest normal values and data near the largest, and the
other way round; the products are ordinary.  Values are powers of two times ordinary
ones, so the result is that of the ordinary values, scaled.

Tolerances as for ordinary values: three transforms of n reals, each within 2 eps
log2 n of exact, and a product, taken as four: 1.5e-5 relative L2."""
import numpy as np
import pytest

import numrs_amd
import oracle
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1 << 13, 1 << 14, 1 << 15])
@pytest.mark.parametrize("small_second", [True, False])
def test_range(n, small_second):
    import torch

    rng = np.random.default_rng(n)
    down, up = 2.0**-122, 2.0**90
    sx, sr = (up, down) if small_second else (down, up)
    # few non-zero values where the scale is small: spectra of the size of the values
    x = rng.standard_normal(n)
    if not small_second:
        x[5:] = 0.0
    x = (x + np.sign(x)).astype(np.float32)
    for m in (5, 700):
        r = rng.uniform(0.5, 1.0, m)
        r[5:m - 2] = 0.0
        r = r.astype(np.float32)
        xt = torch.from_numpy((x * np.float32(sx)).astype(np.float32)).cuda()
        rt = torch.from_numpy((r * np.float32(sr)).astype(np.float32)).cuda()
        y = torch.empty_like(xt)
        numrs_amd.ConvlvPlan("float32", n, m, 1).execute(xt, rt, y, 1)
        want = oracle.convlv(x.astype(np.float64), r.astype(np.float64), 1)
        assert rel_l2(y.cpu().numpy().astype(np.float64) / (sx * sr), want) < 1.5e-5, m
    z = np.zeros(n, np.float32)
    z[:5] = r[:5]
    if not small_second:
        z = (rng.standard_normal(n) + 2).astype(np.float32)
    zt = torch.from_numpy((z * np.float32(sr)).astype(np.float32)).cuda()
    numrs_amd.CorrelPlan("float32", n, 1).execute(xt, zt, y)
    want = oracle.correl(x.astype(np.float64), z.astype(np.float64))
    assert rel_l2(y.cpu().numpy().astype(np.float64) / (sx * sr), want) < 1.5e-5

"""GPU: rlft3 forward plans whose last axis runs with the untangle, at the edges
of the row pairs' enumeration (rows that are their own mirrors only, one middle
plane or none, a last tile that is not full), batched, against the oracle.

Tolerances: a transform of n reals in precision eps is within 2 eps log2 n of
exact: 5e-6 (FP32) and 1e-14 (FP64) relative L2 up to 2^20 values."""
import numpy as np
import pytest

import numrs_amd
import oracle
from conftest import rel_l2
from numrs_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,tol", [(np.float32, 5e-6), (np.float64, 1e-14)])
@pytest.mark.parametrize("shape", [(1, 2, 32), (2, 2, 32), (1, 4, 4096), (2, 2, 4096), (4, 2, 64), (2, 64, 128)])
def test_rlft3_rows(dt, tol, shape):
    import torch

    nn1, nn2, nn3 = shape
    vol, ns, batch = nn1 * nn2 * nn3, 2 * nn1 * nn2, 5
    x = synth.uniform(31, vol * batch).astype(dt)
    plan = numrs_amd.Rlft3Plan(np.dtype(dt).name, nn1, nn2, nn3, batch)
    d = torch.from_numpy(x.copy()).cuda()
    s = torch.empty(ns * batch, dtype=d.dtype, device="cuda")
    plan.execute(d, s, 1)
    gd, gs = d.cpu().numpy(), s.cpu().numpy()
    for i in range(batch):
        seg = x[i * vol:(i + 1) * vol].astype(np.float64)
        rd, rs = oracle.rlft3(seg, np.zeros(ns), nn1, nn2, nn3, 1)
        assert rel_l2(gd[i * vol:(i + 1) * vol].astype(np.float64), rd.reshape(-1)) < tol, i
        assert rel_l2(gs[i * ns:(i + 1) * ns].astype(np.float64), rs.reshape(-1)) < tol, i

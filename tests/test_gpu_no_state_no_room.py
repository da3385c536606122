"""GPU: plans that would run as persistent launches but find no counters left (every
one of the pool is held by a plan) or no room for their ring run in passes."""
import pytest

import numrs_amd
from test_gpu_lanes_given_back import CHILD_HEAD, run_child

pytestmark = pytest.mark.gpu

POOL = 256  # plans with counters of their own at a time


def test_no_counters_left():
    import torch

    n, b = 1 << 15, 320  # a ring of 80 MiB each
    x = torch.empty(2 * n * b, dtype=torch.float32, device="cuda")
    numrs_amd.gen_uniform(x, 17)
    y, ref = torch.empty_like(x), torch.empty_like(x)
    plans = []
    while len(plans) <= POOL:
        plans.append(numrs_amd.C2CPlan("float32", [n], b))
        if plans[-1].launch_info()["ring_slabs"] == 0:
            break
    assert len(plans) > POOL - 64, len(plans)  # (other tests' plans may not be gone yet)
    last = plans.pop()
    info = last.launch_info()
    assert info["ring_slabs"] == 0 and info["launches"] > 1 and info["expired"] is None
    plans[0].execute(x, ref, 1)
    last.execute(x, y, 1)
    last.check()
    assert float((y - ref).norm() / ref.norm()) < 3e-6
    real = numrs_amd.RealFTPlan("float32", 2 * n, b)
    assert real.launch_info()["ring_slabs"] == 0
    z = x.clone()
    real.execute(z, 1)
    real.execute(z, -1)
    assert float((z / n - x).norm() / x.norm()) < 6e-6
    plans.pop().destroy()
    assert numrs_amd.C2CPlan("float32", [n], b).launch_info()["ring_slabs"] > 0


CHILD = CHILD_HEAD + r"""
assert _lib.lib().nrfft_init(0) == 0 and _lib.lib().nrfft_trim() == 0
x = torch.empty(2 * 48 << 18, dtype=torch.float32, device="cuda")
numrs_amd.gen_uniform(x, 3)
y, ref = torch.empty_like(x), torch.empty_like(x)
one, passes = plan(0), plan(1)
assert one.launch_info()["ring_slabs"] > 0 and passes.launch_info()["ring_slabs"] == 0
one.execute(x, ref, -1)
passes.execute(x, y, -1)
assert float((y - ref).norm() / ref.norm()) < 3e-6
try:
    plan(2)  # nor for the passes' workspace
except numrs_amd.NrfftError as e:
    assert e.code == _lib.E_NOMEM, e.code
else:
    raise AssertionError("no error")
assert plan(0).launch_info()["ring_slabs"] > 0  # the counters went back
print("passes", flush=True)
"""


def test_no_room_for_the_ring(tmp_path):
    run_child(tmp_path, CHILD, "passes")

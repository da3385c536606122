"""GPU: a plan gets its counters cleared, whatever the plan that had them before
left there (a caller that ran one plan on two streams at once must not spoil the
plans of others).  The counters are overwritten by the host before their plan, which
runs no more, is destroyed."""
import ctypes

import pytest

import numrs_amd

pytestmark = pytest.mark.gpu


def test_counters_are_cleared_for_the_next_plan():
    import torch

    n, b = 1 << 18, 48
    x = torch.empty(2 * n * b, dtype=torch.float32, device="cuda")
    numrs_amd.gen_uniform(x, 9)
    y, ref = torch.empty_like(x), torch.empty_like(x)
    plan = numrs_amd.C2CPlan("float32", [n], b)
    word = plan.launch_info()["expired"]
    plan.execute(x, ref, 1)
    torch.cuda.synchronize()
    hip = ctypes.CDLL("libamdhip64.so.7")
    junk = (ctypes.c_uint32 * 96)(*([7] * 96))  # the flag, the tickets, the groups that have left: a line each
    assert hip.hipMemcpy(ctypes.c_void_p(word), junk, ctypes.c_size_t(ctypes.sizeof(junk)), 1) == 0
    plan.destroy()
    plan = numrs_amd.C2CPlan("float32", [n], b)
    assert plan.launch_info()["expired"] == word  # the same counters
    plan.check()
    for _ in range(2):
        y.zero_()
        plan.execute(x, y, 1)
        plan.check()
        assert torch.equal(y, ref)

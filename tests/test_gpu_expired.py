"""GPU: a wait inside a persistent launch that has given up is reported by the
plan's check, once, and by none before.  The word a group sets in that case is
written by the host here; no launch is disturbed."""
import ctypes

import pytest

import numrs_amd
from numrs_amd import _lib

pytestmark = pytest.mark.gpu


def _set_word(address):
    import torch

    torch.cuda.synchronize()
    hip = ctypes.CDLL("libamdhip64.so.7")
    one = ctypes.c_uint32(1)
    assert hip.hipMemcpy(ctypes.c_void_p(address), ctypes.byref(one), ctypes.c_size_t(4), 1) == 0
    torch.cuda.synchronize()


def _plans():
    import torch

    def real(n, seed=1):
        x = torch.empty(n, dtype=torch.float32, device="cuda")
        numrs_amd.gen_uniform(x, seed)
        return x

    n, b = 1 << 18, 48
    x = real(2 * n * b)
    y = torch.empty_like(x)
    c2c = numrs_amd.C2CPlan("float32", [n], b)
    yield "c2c", c2c, lambda: c2c.execute(x, y, 1)
    rft, r = numrs_amd.RealFTPlan("float32", 2 * n, b), real(2 * n * b, 2)
    yield "realft", rft, lambda: rft.execute(r, 1)
    cor, a, d = numrs_amd.CorrelPlan("float32", n, 100), real(n * 100, 3), real(n * 100, 4)
    out = torch.empty_like(a)
    yield "correl", cor, lambda: cor.execute(a, d, out)
    un = numrs_amd.UnevenPlan("float32", [(512, 512)] * 3 + [(1 << 16,)] * 5)
    u = real(2 * un.total, 5)
    v = torch.empty_like(u)
    yield "uneven", un, lambda: un.execute(u, v, 1)


def test_expired_wait_is_reported():
    for name, plan, run in _plans():
        print(f"expired: {name}", flush=True)
        word = plan.launch_info()["expired"]
        assert word, name
        run()
        plan.check()
        _set_word(word)
        run()  # an execution does not clear it
        with pytest.raises(numrs_amd.NrfftError):
            plan.check()
        plan.check()  # reported once
        run()
        plan.check()


def test_noalloc_check_and_plans_without_waits():
    import torch

    assert _lib.lib().nrfft_init(0) == _lib.OK
    x = torch.zeros(2 * 48 << 18, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    assert _lib.lib().nrfft_execute_four1_batch_noalloc(_lib.F32, x.data_ptr(), x.data_ptr(), 1 << 18, 48, 1, s) == 0
    assert _lib.lib().nrfft_four1_batch_noalloc_check(s) == _lib.OK
    plan = numrs_amd.C2CPlan("float32", [256], 4)
    assert plan.launch_info() == {"launches": 1, "ring_slots": 0, "ring_slabs": 0, "expired": None}
    plan.check()

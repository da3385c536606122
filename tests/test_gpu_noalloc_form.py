"""GPU: the allocation-free four1 on either side of the batch from which its two
passes run as one launch, against the passes of a plan.

Tolerances: two FFTs of N points in precision eps differ by at most 2 eps log2 N:
3e-6 (FP32, N = 2^21) and 1e-14 (FP64, N = 2^20) relative L2."""
import pytest

import numrs_amd
from numrs_amd import _lib

pytestmark = pytest.mark.gpu

CASES = [("float32", 15, 768), ("float32", 18, 72), ("float32", 19, 28), ("float32", 20, 10), ("float32", 21, 23),
         ("float64", 14, 576), ("float64", 19, 18), ("float64", 20, 13)]


@pytest.mark.parametrize("dtype,logn,batch", CASES)
def test_noalloc_forms(dtype, logn, batch):
    import torch

    assert _lib.lib().nrfft_init(0) == _lib.OK
    code, tol = (_lib.F32, 3e-6) if dtype == "float32" else (_lib.F64, 1e-14)
    n, s = 1 << logn, torch.cuda.current_stream().cuda_stream
    for b in (batch - 1, batch, batch + 1):
        x = torch.empty(2 * n * b, dtype=getattr(torch, dtype), device="cuda")
        numrs_amd.gen_uniform(x, 40 + logn)
        y, ref = torch.full_like(x, float("nan")), torch.empty_like(x)
        plan = numrs_amd.C2CPlan(dtype, [n], b)
        for isign in (1, -1):
            plan.execute_launches(x, ref, isign, 0, plan.num_launches)
            for _ in range(2):
                assert _lib.lib().nrfft_execute_four1_batch_noalloc(code, x.data_ptr(), y.data_ptr(), n, b, isign, s) == 0
            assert float((y - ref).norm() / ref.norm()) < tol, (b, isign)
            assert _lib.lib().nrfft_four1_batch_noalloc_check(s) == _lib.OK

"""GPU: the one-launch forms are no further from 64-bit results than the separate
passes: C2C against execute_launches of the same plan, realft against the plan of
one signal, there and back too; and their FP32 outputs are not short by a common
factor.

Tolerances: the error of 2^18 or more values has a spread far below 1%, so the
one-launch form's mean error may exceed the other's by 1% at most.  Common factor:
less than half a unit of a 24-bit value next to 1, 2^-25 (rounded down, the stages'
constants give 4 to 7e-8)."""
import numpy as np
import pytest

import numrs_amd

pytestmark = pytest.mark.gpu


def _complex(t):
    z = t.cpu().numpy().astype(np.float64)
    return z[0::2] + 1j * z[1::2]


def _spectrum(x):
    z = np.conj(np.fft.rfft(x))
    out = np.empty_like(x)
    out[0], out[1] = z[0].real, z[-1].real
    out[2::2], out[3::2] = z[1:-1].real, z[1:-1].imag
    return out


@pytest.mark.parametrize("logn", range(15, 22))
def test_c2c_error(logn):
    import torch

    n, batch = 1 << logn, max(1, (700 << 14) >> logn)
    x = torch.empty(2 * n * batch, dtype=torch.float32, device="cuda")
    numrs_amd.gen_uniform(x, 900 + logn)
    y, ref = torch.empty_like(x), torch.empty_like(x)
    plan = numrs_amd.C2CPlan("float32", [n], batch)
    assert plan.launch_info()["ring_slabs"] > 0
    for isign in (1, -1):
        plan.execute(x, y, isign)
        plan.execute_launches(x, ref, isign, 0, plan.num_launches)
        one, passes, gain = [], [], []
        for i in range(min(batch, max(2, (1 << 19) >> logn))):
            seg = slice(2 * n * i, 2 * n * (i + 1))
            z = _complex(x[seg])
            want = np.fft.ifft(z) * n if isign > 0 else np.fft.fft(z)
            got = _complex(y[seg])
            one.append(np.linalg.norm(got - want))
            passes.append(np.linalg.norm(_complex(ref[seg]) - want))
            gain.append(np.vdot(want, got) / np.vdot(want, want) - 1)
        assert np.mean(one) < 1.01 * np.mean(passes), (isign, np.mean(one) / np.mean(passes))
        assert abs(np.mean(gain)) < 2.0**-25, (isign, np.mean(gain))


@pytest.mark.parametrize("logl", range(15, 22))
def test_realft_error(logl):
    import torch

    n, batch = 2 << logl, max(1, (1160 << 14) >> logl)
    x0 = torch.empty(n * batch, dtype=torch.float32, device="cuda")
    numrs_amd.gen_uniform(x0, 950 + logl)
    plan, one = numrs_amd.RealFTPlan("float32", n, batch), numrs_amd.RealFTPlan("float32", n, 1)
    assert plan.launch_info()["ring_slabs"] > 0 and one.launch_info()["ring_slabs"] == 0
    x = x0.clone()
    plan.execute(x, 1)
    spec = x.clone()
    plan.execute(x, -1)
    err = np.zeros((2, 2))
    for i in range(min(batch, max(2, (1 << 19) >> logl))):
        seg = slice(n * i, n * (i + 1))
        src = x0[seg].cpu().numpy().astype(np.float64)
        r = x0[seg].clone()
        one.execute(r, 1)
        rs = r.clone()
        one.execute(r, -1)
        for k, (s, b) in enumerate(((spec[seg], x[seg]), (rs, r))):
            want = _spectrum(src)
            err[k] += (np.linalg.norm(s.cpu().numpy() - want) / np.linalg.norm(want),
                       np.linalg.norm(b.cpu().numpy() * (2.0 / n) - src) / np.linalg.norm(src))
    assert (err[0] < 1.01 * err[1]).all(), err[0] / err[1]

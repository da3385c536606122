"""GPU: host-pointer calls through lanes: buffers of a few bytes, around the
staging limit (1 MiB) and the lane limit (32 MiB), and more threads than lanes,
against numpy in FP64.

Tolerances: a transform of n points in precision eps is within 2 eps log2 n of
exact (relative L2): 6e-6 (FP32) and 1.2e-14 (FP64) up to 2^25 points; a
correlation is three and a product, taken as four of them."""
import threading

import numpy as np
import pytest

import numrs_amd

pytestmark = pytest.mark.gpu

TOL = {np.float32: 6e-6, np.float64: 1.2e-14}


def _rel(a, b):
    return float(np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b))


def _four1(rng, dt, n):
    x = rng.standard_normal(2 * n).astype(dt)
    z = x[0::2].astype(np.float64) + 1j * x[1::2].astype(np.float64)
    want = np.fft.ifft(z) * n
    y = x.copy()
    numrs_amd.four1(y, n, 1)
    got = y[0::2].astype(np.float64) + 1j * y[1::2].astype(np.float64)
    assert np.linalg.norm(got - want) < TOL[dt] * np.linalg.norm(want), (dt, n)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("logn", [1, 2, 5, 10, 15, 16, 17, 20, 21, 22])
def test_host_sizes(dt, logn):
    _four1(np.random.default_rng(logn), dt, 1 << logn)


def test_host_threads():
    errors = []

    def work(seed):
        try:
            rng = np.random.default_rng(seed)
            for k in range(12):
                dt = (np.float32, np.float64)[(seed + k) % 2]
                _four1(rng, dt, 1 << int(rng.integers(1, 18)))
                n = 1 << int(rng.integers(8, 16))
                x = rng.standard_normal(n).astype(dt)
                y = numrs_amd.correl(x, x) if n > 32 else x
                f = np.fft.rfft(x.astype(np.float64))
                want = np.fft.irfft(f * np.conj(f), n)
                assert _rel(np.asarray(y), want) < 4 * TOL[dt], (seed, k, n)
        except Exception as e:  # noqa: BLE001 -- reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(7)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]

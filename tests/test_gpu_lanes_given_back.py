"""GPU: the memory that host-pointer calls keep is given back: by nrfft_trim, and when
a plan finds no room (a stand-in for hipMalloc in a child process fails once)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import numrs_amd
from numrs_amd import _lib

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
static int fails;
void fail_next(int n) { fails = n; } /* the next n allocations of 1 MiB and more */
int hipMalloc(void** p, size_t bytes) {
    static int (*real)(void**, size_t);
    if (!real) real = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD), "hipMalloc");
    if (bytes >= (1u << 20) && fails > 0) {
        --fails;
        *p = 0;
        return 2; /* hipErrorOutOfMemory */
    }
    return real(p, bytes);
}
"""

CHILD_HEAD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before anything that allocates on the GPU
import numpy as np
import torch
import numrs_amd
from numrs_amd import _lib

def host_call():
    a = np.zeros(2 << 12)
    a[0] = 1
    numrs_amd.four1(a, 1 << 12, 1)
    assert np.allclose(a[0::2], 1)

def plan(fails):
    shim.fail_next(fails)
    p = numrs_amd.C2CPlan("float32", [1 << 18], 48)
    shim.fail_next(0)
    return p
"""

CHILD = CHILD_HEAD + r"""
host_call()
assert plan(1).launch_info()["ring_slabs"] > 0  # the lane's memory, then the ring
print("given back", flush=True)
host_call()  # a new lane
"""


def run_child(tmp_path, code, says):
    src, lib = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src), "-ldl"], check=True)
    run = subprocess.run([sys.executable, "-c", code, str(lib)], cwd=ROOT, capture_output=True, text=True, timeout=110)
    assert run.returncode == 0 and says in run.stdout, run.stdout + run.stderr


def test_trim():
    import torch

    x = np.zeros(2 << 20, np.float32)
    x[0] = 1
    numrs_amd.four1(x, 1 << 20, 1)  # 16 MiB of device memory
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    assert _lib.lib().nrfft_trim() == _lib.OK
    assert torch.cuda.mem_get_info()[0] - before >= 16 << 20
    x[:] = 0
    x[0] = 1
    numrs_amd.four1(x, 1 << 20, 1)
    assert np.allclose(x[0::2], 1)


def test_given_back_to_a_plan(tmp_path):
    run_child(tmp_path, CHILD, "given back")

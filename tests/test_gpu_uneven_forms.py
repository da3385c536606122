"""GPU: the two forms of an uneven batch (one list, or one launch a pass), at the
edges of the rule that chooses between them, against the pass-by-pass C2C plan of
each item; and a batch whose ring finds no room.

Tolerances: two FFTs of the same data by different factorisations, each within
eps sqrt(log2 N) of exact in relative L2 (eps: 2^-23, 2^-52), differ by less than
2 eps sqrt(26) < 11 eps.
"""
import math
import os
import subprocess
import sys

import pytest

import numrs_amd

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIST, PASSES = 1, 3  # launches

CASES = [
    ("float32", [(1 << 21,)] * 2, PASSES), ("float32", [(1 << 21,)] * 3, LIST),
    ("float32", [(1 << 22,)], PASSES), ("float32", [(1 << 22,)] * 3, LIST),
    ("float32", [(1 << 23,)], PASSES), ("float32", [(1 << 24,)], PASSES),
    ("float32", [(2048, 2048)], PASSES), ("float32", [(2048, 2048)] * 2, LIST),
    ("float32", [(1024, 2048)], LIST), ("float32", [(1024, 2048)] * 2, PASSES), ("float32", [(1024, 2048)] * 3, LIST),
    ("float32", [(4096, 4096)], PASSES), ("float32", [(4096, 2048)] * 2, LIST),
    ("float32", [(8192, 64)], PASSES), ("float32", [(64, 8192)], PASSES),
    # most of the work decides
    ("float32", [(1 << 22,)] + [(1 << 16,), (64, 64), (1 << 12,)] * 9, PASSES),
    ("float32", [(1 << 22,)] + [(1 << 20,), (512, 512), (1 << 12,)] * 4, LIST),
    ("float32", [(1 << 13,)] * 128, 2), ("float32", [(1 << 13,)] * 129, LIST),
    # the shapes of the other form as the smaller part of a list
    ("float32", [(8192, 64), (64, 8192), (8192, 128)] + [(1024, 1024)] * 4, LIST),
    ("float32", [(1 << 22,), (1 << 23,)] + [(1 << 20,)] * 16, LIST),
    ("float32", [(4096, 4096)] + [(1 << 20,)] * 20, LIST),
    ("float64", [(64, 8192), (1 << 22,), (4096, 1024)] + [(1 << 18,)] * 48, LIST),
    ("float64", [(1 << 20,)], LIST), ("float64", [(1 << 20,)] * 2, PASSES), ("float64", [(1 << 20,)] * 3, LIST),
    ("float64", [(1 << 22,)], PASSES), ("float64", [(1 << 22,)] * 2, LIST),
    ("float64", [(4096, 1024)], PASSES), ("float64", [(4096, 512)] * 2, LIST), ("float64", [(2048, 2048)] * 2, LIST),
    ("float64", [(1 << 13,)] * 128, LIST), ("float64", [(1 << 13,)] * 129, 2), ("float64", [(1 << 13,)] * 700, LIST),
]


@pytest.mark.parametrize("k", range(len(CASES)))
def test_forms(k):
    import torch

    dtype, items, launches = CASES[k]
    print(f"uneven form {dtype} {len(items)} items, first {items[0]}", flush=True)
    gap, offsets, at = 3, [], 0
    for it in items:
        offsets.append(at)
        at += math.prod(it) + gap
    plan = numrs_amd.UnevenPlan(dtype, items, offsets)
    assert plan.launch_info()["launches"] == launches
    two_pass_1d = sum(it[0] for it in items if len(it) == 1 and it[0] > 1 << 13)
    if launches != LIST:  # 2-D items need no workspace
        assert plan.workspace_bytes == two_pass_1d * (8 if dtype == "float32" else 16)
    x = torch.empty(2 * at, dtype=getattr(torch, dtype), device="cuda")
    numrs_amd.gen_uniform(x, 70 + k)
    tol = 11 * torch.finfo(x.dtype).eps
    plans = {it: numrs_amd.C2CPlan(dtype, list(it), 1) for it in set(items)}
    for isign in (1, -1):
        y = torch.full_like(x, 7.0)
        for _ in range(2):
            plan.execute(x, y, isign)
            plan.check()
        z = x.clone()
        plan.execute(z, z, isign, graph=False)
        for it, o in list(zip(items, offsets))[:40]:
            n = math.prod(it)
            ref = torch.empty(2 * n, dtype=x.dtype, device="cuda")
            plans[it].execute_launches(x[2 * o:2 * (o + n)].clone(), ref, isign, 0, plans[it].num_launches)
            for out in (y, z):
                assert float((out[2 * o:2 * (o + n)] - ref).norm() / ref.norm()) < tol, (isign, it)
            assert bool((y[2 * (o + n):2 * (o + n + gap)] == 7.0).all()), (isign, it)


SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
static size_t limit = (size_t)-1;
void no_room_above(size_t bytes) { limit = bytes; }
int hipMalloc(void** p, size_t bytes) {
    static int (*real)(void**, size_t);
    if (!real) real = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD), "hipMalloc");
    if (bytes > limit) {
        *p = 0;
        return 2; /* hipErrorOutOfMemory */
    }
    return real(p, bytes);
}
"""

CHILD = r"""
import ctypes, math, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before anything that allocates on the GPU
shim.no_room_above.argtypes = [ctypes.c_size_t]
import torch
import numrs_amd

def limited(make, bytes_):
    shim.no_room_above(bytes_)
    try:
        return make()
    finally:
        shim.no_room_above(2**64 - 1)

def data(n):
    x = torch.empty(n, dtype=torch.float32, device="cuda")
    numrs_amd.gen_uniform(x, 3)
    return x

x = data(2 * 4 << 20)
y, ref = torch.empty_like(x), torch.empty_like(x)
items = [(1024, 1024)] * 4
plan = numrs_amd.UnevenPlan("float32", items)
assert plan.launch_info()["launches"] == 1 and plan.workspace_bytes == 4 << 23
plan.execute(x, ref, 1)
small = limited(lambda: numrs_amd.UnevenPlan("float32", items), 1 << 20)
assert small.launch_info()["launches"] == 3 and small.workspace_bytes == 0
small.execute(x, y, 1)
small.check()
assert float((y - ref).norm() / ref.norm()) < 11 * 2.0**-23
try:  # a 1-D item of two passes needs memory in either form
    limited(lambda: numrs_amd.UnevenPlan("float32", [(1 << 20,)]), 1 << 20)
except numrs_amd.NrfftError as e:
    assert e.code == -8, e.code
else:
    raise AssertionError("no error")
print("no room ok", flush=True)
"""


def test_ring_finds_no_room(tmp_path):
    src, lib = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src), "-ldl"], check=True)
    run = subprocess.run([sys.executable, "-c", CHILD, str(lib)], cwd=ROOT, capture_output=True, text=True, timeout=110)
    assert run.returncode == 0 and "no room ok" in run.stdout, run.stdout + run.stderr

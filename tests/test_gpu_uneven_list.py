"""GPU: the tile list of an uneven batch at its edges (every tile length and
mode, packed single-pass items with gaps, ring places handed out again, few and
many tiles), against the pass-by-pass C2C plan of each item.

Tolerances: two FFTs of the same data by different factorisations, each within
eps sqrt(log2 N) of exact in relative L2 (eps: 2^-23, 2^-52), so they differ by
less than 2 eps sqrt(22) < 10 eps.
"""
import math

import pytest

import numrs_amd

pytestmark = pytest.mark.gpu

CASES = {
    # single-pass items of every length, more than a tile holds, at odd offsets
    "rows": [(1 << k,) for k in range(6, 14) for _ in range(3 + (300 >> (k - 6)))],
    # first and second passes of every length
    "sides": [(1 << a, 1 << b) for a in range(6, 12) for b in range(6, 12)],
    "long_rows": [(64, 8192), (128, 8192), (64, 4096)],
    "long_cols": [(4096, 64), (4096, 128)],
    "lengths": [(1 << k,) for k in range(13, 23)],
    # places in the ring handed out again: to slabs of the same size, of smaller ones
    "reuse_even": [(1 << 20,)] * 27,
    "reuse_mixed": [(2048, 2048)] * 7 + [(1 << 19,), (512, 512), (64, 64), (4096,)] * 40 + [(1 << 16,)] * 30,
    "one": [(1 << 14,)],
}


def _check(dtype, items, gap):
    import torch

    offsets, at = [], 0
    for it in items:
        offsets.append(at)
        at += math.prod(it) + gap
    plan = numrs_amd.UnevenPlan(dtype, items, offsets)
    x = torch.empty(2 * at, dtype=getattr(torch, dtype), device="cuda")
    numrs_amd.gen_uniform(x, 900 + len(items))
    tol = 10 * torch.finfo(x.dtype).eps
    plans = {it: numrs_amd.C2CPlan(dtype, list(it), 1) for it in set(items)}
    for isign in (1, -1):
        y = torch.full_like(x, 7.0)
        for _ in range(2):  # the counters are left as they were found
            plan.execute(x, y, isign)
            plan.check()
        z = x.clone()
        plan.execute(z, z, isign, graph=False)
        for k, (it, o) in enumerate(zip(items, offsets)):
            n = math.prod(it)
            ref = torch.empty(2 * n, dtype=x.dtype, device="cuda")
            src = x[2 * o:2 * (o + n)].clone()
            plans[it].execute_launches(src, ref, isign, 0, plans[it].num_launches)
            for out in (y, z):
                got = out[2 * o:2 * (o + n)]
                assert float((got - ref).norm() / ref.norm()) < tol, (dtype, isign, k, it)
            if gap:  # nothing between the items is written
                assert bool((y[2 * (o + n):2 * (o + n + gap)] == 7.0).all()), (dtype, isign, k, it)


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("dtype", ["float32", "float64"])
def test_uneven_list(dtype, name):
    items = CASES[name]
    print(f"uneven list {dtype} {name}: {len(items)} items", flush=True)
    _check(dtype, items, 0 if name.startswith("reuse") else 3)


def test_uneven_rows_8192_columns():
    _check("float32", [(8192, 64), (8192, 128)], 1)

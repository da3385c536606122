"""GPU: which plans run as persistent launches.  At the smallest batch that takes
one the plan has it, one below it runs in passes; and the batches by which the
other tests mean to use places of the ring again do so."""
import pytest

import numrs_amd

pytestmark = pytest.mark.gpu

TILE = {"float32": 1 << 14, "float64": 1 << 13}
RANGE = {"float32": (15, 22), "float64": (14, 21)}  # log2 points of a fused C2C


def _batch(dtype, logn, tiles):
    return max(1, -(-(tiles * TILE[dtype]) >> logn))


def _fused(plan, isign=1):
    return plan.launch_info(isign)["ring_slabs"] > 0


@pytest.mark.parametrize("dtype", ["float32", "float64"])
def test_c2c(dtype):
    for logn in range(*RANGE[dtype]):
        b = _batch(dtype, logn, 1024 if dtype == "float64" and logn >= 18 else 640)
        info = numrs_amd.C2CPlan(dtype, [1 << logn], b).launch_info()
        assert info["launches"] == 1 and info["ring_slabs"] > 0 and info["expired"], (logn, b, info)
        info = numrs_amd.C2CPlan(dtype, [1 << logn], b - 1).launch_info()
        assert info["launches"] > 1 and info["ring_slabs"] == 0 and info["expired"] is None, (logn, b - 1, info)
    for logn in (RANGE[dtype][0] - 1, RANGE[dtype][1]):
        assert not _fused(numrs_amd.C2CPlan(dtype, [1 << logn], _batch(dtype, logn, 1100))), logn


@pytest.mark.parametrize("dtype", ["float32", "float64"])
def test_realft(dtype):
    for logl in range(*RANGE[dtype]):
        late, last = (20, 21) if dtype == "float32" else (18, 20)
        b = _batch(dtype, logl, 1152 if logl == last else 1024 if logl >= late else 640)
        at, below = (numrs_amd.RealFTPlan(dtype, 2 << logl, k) for k in (b, b - 1))
        for isign in (1, -1):
            info = at.launch_info(isign)
            assert info["launches"] == 1 and info["ring_slabs"] > 0, (logl, isign, info)
            assert not _fused(below, isign), (logl, isign)


@pytest.mark.parametrize("dtype", ["float32", "float64"])
def test_correl(dtype):
    for logl in range(RANGE[dtype][0], 20):
        b = _batch(dtype, logl, 512)
        info = numrs_amd.CorrelPlan(dtype, 2 << logl, b).launch_info()
        assert info["launches"] == 2 and info["ring_slabs"] > 0, (logl, info)
        assert not _fused(numrs_amd.CorrelPlan(dtype, 2 << logl, b - 1)), logl
    # longer spectra: passes, and a pass for the product
    assert numrs_amd.CorrelPlan(dtype, 2 << 20, _batch(dtype, 20, 1100)).launch_info()["launches"] > 2


def test_inside_other_plans():
    for dtype, n, b in (("float32", 1 << 17, 160), ("float64", 1 << 16, 161)):
        assert _fused(numrs_amd.ConvlvPlan(dtype, n, 65, b)), dtype
        assert _fused(numrs_amd.TwofftPlan(dtype, n, b)), dtype


def test_ring_places_used_again():
    def reuse(plan):
        for isign in (1, -1):
            info = plan.launch_info(isign)
            assert 0 < info["ring_slots"] < info["ring_slabs"], info

    for dtype, logn, b in (("float32", 15, 3077), ("float32", 20, 27), ("float32", 21, 14), ("float64", 14, 773),
                           ("float64", 20, 13)):
        reuse(numrs_amd.C2CPlan(dtype, [1 << logn], b))
    for dtype, logl, b in (("float32", 15, 770), ("float32", 19, 51), ("float32", 21, 14), ("float64", 14, 1541),
                           ("float64", 20, 13)):
        reuse(numrs_amd.RealFTPlan(dtype, 2 << logl, b))
    for dtype, logl, b in (("float32", 15, 771), ("float32", 19, 51), ("float64", 14, 770), ("float64", 19, 25)):
        reuse(numrs_amd.CorrelPlan(dtype, 2 << logl, b))
    for items in ([(1 << 20,)] * 27, [(2048, 2048)] * 7 + [(1 << 16,)] * 30):
        assert numrs_amd.UnevenPlan("float32", items).launch_info()["ring_reused"]
    assert not numrs_amd.UnevenPlan("float32", [(1 << 20,)] * 4).launch_info()["ring_reused"]

"""xpu_gemm's choice of tile and K ranges (gemm_api.cpp), asked without a GPU:
what every plan has to keep, and plans of measured shapes."""
import ctypes
import random

import pytest

import xpu_playground_amd as xpu

CUS = 256  # MI355X
STAGES = {32: 4, 64: 3}  # slices per group of the tiles that are split (kernels/gemm.hip)


def gemm_plan(m, n, k, cus=CUS):
    """rows, cols, splits, slices per range, largest number of ranges"""
    v = [ctypes.c_uint32() for _ in range(5)]
    xpu.library().xpu_internal_gemm_plan(cus, m, n, k, *map(ctypes.byref, v))
    return tuple(x.value for x in v)


def log_random(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def test_plans_cover_k_and_stay_within_the_limit():
    rng, split = random.Random(1), 0
    for _ in range(20000):
        m, n, k = (log_random(rng, 1, 8192) for _ in range(3))
        rows, cols, splits, slices, limit = gemm_plan(m, n, k, rng.choice([1, 64, CUS, 304]))
        assert 1 <= splits <= limit
        if splits >= 2:
            split += 1
            assert cols == 128 and slices % STAGES[rows] == 0
            assert (splits - 1) * slices < (k + 63) // 64 <= splits * slices  # no empty range
    assert split > 1000


@pytest.mark.parametrize("m,n,k,plan", [
    (24, 4096, 4096, (32, 128, 8)), (1024, 1024, 1024, (32, 128, 1)), (512, 512, 512, (32, 128, 1)),
    (1500, 1000, 600, (64, 128, 1)), (33, 1000, 1537, (32, 128, 7)), (768, 768, 8192, (64, 128, 3)),
    (118, 2632, 3942, (32, 128, 3)), (4096, 4096, 4096, (256, 256, 1)), (3000, 4097, 2050, (224, 256, 1))])
def test_plans_of_measured_shapes(m, n, k, plan):
    assert gemm_plan(m, n, k)[:3] == plan

"""The GEMM's small block tiles (32x128, 64x128): launched by name on ragged
shapes and 2-byte offsets against the 128x128 tile (the same k-order per MFMA
chain: the same bits) and, through xpu_gemm, in the plans that the dispatch
takes around its limits (whole K, K split at stage groups and past K) against
the FP64 oracle at the GEMM bar."""
import numpy as np
import pytest

import oracle_lib as orc
import test_gpu_gemm_edges as edges
import xpu_playground_amd as xpu
from test_gpu_gemm import check, gpu_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [xpu.BF16, xpu.FP16])
@pytest.mark.parametrize("m,n,k,offsets", [
    (1, 1, 1, (0, 0, 0)), (31, 127, 63, (2, 6, 2)), (32, 128, 64, (0, 0, 0)), (33, 129, 65, (4, 2, 0)),
    (64, 128, 192, (0, 0, 0)), (65, 136, 193, (0, 0, 0)), (63, 263, 256, (6, 14, 4)), (100, 96, 257, (0, 0, 2)),
    (129, 392, 520, (0, 0, 0)), (300, 77, 1031, (10, 2, 0))])
def test_small_tiles_equal_128_tile(rt, monkeypatch, dtype, m, n, k, offsets):
    monkeypatch.setitem(edges.TILES, "_m32", (32, 128))
    monkeypatch.setitem(edges.TILES, "_m64", (64, 128))
    a = orc.uniform(m * k, 3 * m + k, dtype)
    b = orc.uniform(k * n, 5 * n + k, dtype)
    want = edges.launch_tile(rt, "_t128", dtype, a, b, m, n, k, offsets)
    check(want, a, b, m, n, k, dtype)
    for tag in ("_m32", "_m64"):
        assert np.array_equal(edges.launch_tile(rt, tag, dtype, a, b, m, n, k, offsets), want)


@pytest.mark.parametrize("m,n,k", [
    (4, 4096, 4096), (24, 130, 2050), (32, 64, 4095), (33, 1000, 1537), (64, 1024, 1600), (257, 500, 1991),
    (96, 3001, 513), (512, 640, 448), (1025, 513, 200), (1500, 1001, 601), (4, 64, 511), (4, 64, 513)])
def test_dispatch_around_its_limits(rt, m, n, k):
    dtype = xpu.FP16 if (m + n + k) % 2 else xpu.BF16
    print(f"xpu_gemm {m}x{n}x{k} dtype={dtype}", flush=True)
    a = orc.uniform(m * k, m + 1, dtype)
    b = orc.uniform(k * n, n + 2, dtype)
    rows = None if m * n * k < 1 << 28 else np.arange(0, m, 11)
    check(gpu_gemm(rt, a, b, m, n, k, dtype), a, b, m, n, k, dtype, rows=rows)

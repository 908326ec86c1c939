"""The GEMM's small block tiles (32x128, 64x128): launched by name on ragged
shapes and 2-byte offsets against the 128x128 tile (the same k-order per MFMA
chain: the same bits), whole K and in K ranges, and, through xpu_gemm, in the
plans that the dispatch takes around its limits (whole K, K split at stage
groups and past K, in each tile) against the FP64 oracle at the GEMM bar."""
import numpy as np
import pytest

import oracle_lib as orc
import test_gpu_gemm_edges as edges
import xpu_playground_amd as xpu
from test_gemm_plan import gemm_plan
from test_gpu_gemm import check, gpu_gemm
from xpu_playground_amd import Args

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [xpu.BF16, xpu.FP16])
@pytest.mark.parametrize("m,n,k,offsets", [
    (1, 1, 1, (0, 0, 0)), (31, 127, 63, (2, 6, 2)), (32, 128, 64, (0, 0, 0)), (33, 129, 65, (4, 2, 0)),
    (64, 128, 192, (0, 0, 0)), (65, 136, 193, (0, 0, 0)), (63, 263, 256, (6, 14, 4)), (100, 96, 257, (0, 0, 2)),
    (129, 392, 520, (0, 0, 0)), (300, 77, 1031, (10, 2, 0)),
    # more tile-columns than tile-rows, no multiple of 8 tiles: dealt to the XCDs in ranges
    (5, 2100, 70, (0, 0, 0)), (70, 1300, 130, (2, 4, 2)), (97, 520, 65, (0, 0, 0))])
def test_small_tiles_equal_128_tile(rt, monkeypatch, dtype, m, n, k, offsets):
    monkeypatch.setitem(edges.TILES, "_m32", (32, 128))
    monkeypatch.setitem(edges.TILES, "_m64", (64, 128))
    a = orc.uniform(m * k, 3 * m + k, dtype)
    b = orc.uniform(k * n, 5 * n + k, dtype)
    want = edges.launch_tile(rt, "_t128", dtype, a, b, m, n, k, offsets)
    check(want, a, b, m, n, k, dtype)
    for tag in ("_m32", "_m64"):
        assert np.array_equal(edges.launch_tile(rt, tag, dtype, a, b, m, n, k, offsets), want)


def launch_ranges(rt, rows, dtype, a, b, m, n, k, slices, offsets):
    """One launch of a split kernel and of the reduction: the FP32 partials and C."""
    tag = {32: "_m32", 64: "_m64"}[rows]
    splits, pitch = ((k + 63) // 64 + slices - 1) // slices, (n + 3) // 4 * 4
    words = splits * m * pitch
    da, db = rt.alloc(a.size * 2 + 32), rt.alloc(b.size * 2 + 32)
    dp, dc = rt.alloc(words * 4 + 64), rt.alloc(m * n * 2 + 64)
    try:
        rt.copy_to(da + offsets[0], a)
        rt.copy_to(db + offsets[1], b)
        rt.copy_to(dp, np.full(words + 16, 0x7FC12345, np.uint32))
        rt.copy_to(dc, np.full(m * n + 32, edges.GUARD, np.uint16))
        name = f"xpu_gemm_{'fp16' if dtype else 'bf16'}{tag}_part_dma{'_edge' if k % 8 or n % 2 else ''}"
        grid = (m + rows - 1) // rows * ((n + 127) // 128) * splits
        print(f"{name} {m}x{n}x{k} {splits} ranges of {slices} slices, offsets {offsets}, grid {grid}", flush=True)
        rt.launch_grid(name, grid, 256, 0, Args().ptr(da + offsets[0]).ptr(db + offsets[1]).ptr(dp).u32(m).u32(n)
                       .u32(k).u32(slices).u32(pitch).u32(n))
        rt.launch_grid("xpu_gemm_splitk_reduce_any", (m * pitch // 4 + 255) // 256, 256, 0,
                       Args().ptr(dp).ptr(dc + offsets[2]).u32(m).u32(n).u32(pitch).u32(n).u32(splits).u32(dtype))
        rt.synchronize()
        parts, out = rt.download(dp, words + 16, np.uint32), rt.download(dc, m * n + 32, np.uint16)
    finally:
        for p in (da, db, dp, dc):
            rt.free(p)
    o = offsets[2] // 2
    assert np.all(parts[words:] == 0x7FC12345), "store outside the partials"
    assert np.all(out[:o] == edges.GUARD) and np.all(out[o + m * n:] == edges.GUARD), "store outside C"
    return parts[:words].reshape(splits, m, pitch)[:, :, :n], out[o:o + m * n].reshape(m, n)


@pytest.mark.parametrize("dtype", [xpu.BF16, xpu.FP16])
@pytest.mark.parametrize("m,n,k,slices,offsets", [
    (33, 130, 64 * 24, 12, (0, 0, 0)),        # two whole ranges
    (65, 129, 64 * 13, 12, (4, 2, 2)),        # the last range has one live slice
    (31, 257, 64 * 13 + 5, 12, (2, 6, 0)),    # and one more with five live columns
    (100, 72, 64 * 23 + 63, 12, (0, 0, 4)),   # the last group partly past K
    (64, 128, 64 * 96, 12, (0, 0, 0)),        # 8 ranges: the reduction's first batch of seven
    (40, 96, 64 * 97 + 1, 12, (0, 0, 0)),     # 9: into its second
    (70, 1300, 64 * 26, 12, (0, 0, 0)),       # 33 and 22 tiles a range, dealt to the XCDs in ranges
    (5, 66, 64 * 180 + 2, 12, (10, 2, 2))])   # 16: past its second
def test_range_kernels_give_the_same_partials(rt, dtype, m, n, k, slices, offsets):
    a = orc.uniform(m * k, 7 * m + k, dtype)
    b = orc.uniform(k * n, 9 * n + k, dtype)
    want, out = launch_ranges(rt, 64, dtype, a, b, m, n, k, slices, offsets)
    check(out, a, b, m, n, k, dtype)
    parts, c = launch_ranges(rt, 32, dtype, a, b, m, n, k, slices, offsets)
    assert np.array_equal(parts, want) and np.array_equal(c, out)
    # the partials themselves: each range's product, in 64 bits
    fa = orc.decode(a, dtype).reshape(m, k).astype(np.float64)
    fb = orc.decode(b, dtype).reshape(k, n).astype(np.float64)
    for s, part in enumerate(want.view(np.float32)):
        r = slice(s * slices * 64, min(k, (s + 1) * slices * 64))
        # FP32 sums of up to 768 products: gamma_768 sum|a b|
        bound = 768 * 2.0 ** -24 * (np.abs(fa[:, r]) @ np.abs(fb[r])) * 1.01 + 1e-30
        assert np.all(np.abs(part - fa[:, r] @ fb[r]) <= bound)


# (m, n, k, rows of the tile, K ranges) that the dispatch takes on 256 compute units
@pytest.mark.parametrize("m,n,k,rows,splits", [
    (24, 4096, 4096, 32, 8), (33, 1000, 1537, 32, 7), (118, 2632, 3942, 32, 3), (3043, 66, 1666, 64, 5),
    (768, 768, 8192, 64, 3), (1000, 1001, 5001, 64, 2)])
def test_dispatch_splits_in_each_tile(rt, m, n, k, rows, splits):
    if rt.compute_units == 256:
        assert gemm_plan(m, n, k)[::2][:2] == (rows, splits)
    for dtype in (xpu.BF16, xpu.FP16):
        print(f"xpu_gemm {m}x{n}x{k} dtype={dtype}", flush=True)
        a = orc.uniform(m * k, m + 3, dtype)
        b = orc.uniform(k * n, n + 4, dtype)
        some = np.arange(0, m, max(1, m // 40))
        check(gpu_gemm(rt, a, b, m, n, k, dtype), a, b, m, n, k, dtype, rows=some)


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

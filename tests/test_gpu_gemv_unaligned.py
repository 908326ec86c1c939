"""xpu_gemv on rows that are not 16-byte aligned (16-byte loads at any element,
the slice that crosses K shifted into place) and on row lengths around the
512-column chunk and the two- and four-chunk batches, against the oracle's
canonical order bit for bit. Columns K .. lda - 1, the codes before the matrix
and those after its last row hold NaN, which one wrong column would spread."""
import numpy as np
import pytest

import oracle_lib as orc
import xpu_playground_amd as xpu

pytestmark = pytest.mark.gpu

NAN = {xpu.BF16: 0x7FC0, xpu.FP16: 0x7E00}


@pytest.mark.parametrize("dtype", [xpu.BF16, xpu.FP16])
@pytest.mark.parametrize("k,pad,offset", [
    (1, 0, 0), (7, 0, 1), (8, 3, 1), (9, 0, 0), (13, 2, 3), (505, 0, 1), (511, 1, 0), (512, 1, 0), (513, 0, 7),
    (519, 8, 8), (520, 0, 0), (1023, 0, 1), (1024, 3, 0), (1030, 0, 5), (1536, 0, 8), (1537, 0, 0), (2050, 0, 1),
    (3001, 4, 0), (8191, 0, 1), (8192, 1, 0), (8193, 0, 0), (10241, 0, 3), (16383, 0, 1)])
@pytest.mark.parametrize("m", [1, 9])
def test_unaligned_rows(rt, dtype, m, k, pad, offset):
    lda = k + pad
    a = np.full((m, lda), NAN[dtype], np.uint16)
    a[:, :k] = orc.uniform(m * k, 3 * k + offset, dtype).reshape(m, k)
    x = orc.uniform(k, 5 * k + m, dtype)
    want = orc.gemv_canonical(a.reshape(-1), x, m, k, lda, dtype)
    guard = np.full(16, NAN[dtype], np.uint16)
    da = rt.upload(np.concatenate([guard[:offset], a.reshape(-1), guard]))
    dx = rt.upload(np.concatenate([guard[:offset], x, guard]))
    dy = rt.upload(np.full(m + 16, 0x7FC1, np.uint16))
    print(f"gemv {m}x{k} lda {lda} offset {offset}", flush=True)
    try:
        rt.gemv(dtype, da + 2 * offset, dx + 2 * offset, dy, m, k, lda)
        rt.synchronize()
        y = rt.download(dy, m + 16, np.uint16)
    finally:
        for p in (da, dx, dy):
            rt.free(p)
    assert np.array_equal(y[:m], want)
    assert np.all(y[m:] == 0x7FC1)


@pytest.mark.parametrize("dtype", [xpu.BF16, xpu.FP16])
@pytest.mark.parametrize("k", [8, 504, 1024, 1032, 2048, 3072, 4088, 4096, 4104, 5120, 7168, 7680, 8184, 8192, 8200])
@pytest.mark.parametrize("m", [1, 9])
def test_aligned_rows_with_and_without_ends(rt, dtype, m, k):
    """Aligned rows around the change of kernels: row ends loaded ahead of the
    batches, except where 4096 columns or more are whole batches."""
    test_unaligned_rows(rt, dtype, m, k, 8, 8)


def test_many_rows_of_whole_batches(rt):
    """A matrix past 400 MB: one block a compute unit instead of four."""
    test_unaligned_rows(rt, xpu.BF16, (200 << 20) // 7168 + 1, 7168, 0, 0)

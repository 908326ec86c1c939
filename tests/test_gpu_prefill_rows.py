"""The batched prompt projections on the FP32 MFMA (xpu_q3_pf_rows_*) against
the oracle's canonical GEMV, bit for bit: token counts around the 16-token
tile, row counts around the 8-tile XCD groups, one and several token groups,
and inputs whose products cancel or are FP32 subnormals (an MFMA that flushed
them, or rounded a chain's sum more than once, would differ)."""
import numpy as np
import pytest

import oracle_lib as orc
import xpu_playground_amd as xpu
from xpu_playground_amd import Args, qwen3

pytestmark = pytest.mark.gpu

KERNELS = [(0, 2, 8), (0, 4, 4), (0, 8, 8), (1, 2, 8), (1, 4, 4), (1, 6, 4), (1, 8, 8), (2, 2, 4), (2, 4, 8), (2, 8, 8)]
GUARD = 0x7FC1


def inputs(rows, T, K, seed):
    w = orc.decode(orc.uniform(rows * K, seed, xpu.BF16), xpu.BF16).reshape(rows, K)
    x = orc.decode(orc.uniform(T * K, seed + 1, xpu.BF16), xpu.BF16).reshape(T, K)
    # one row and one token each of tiny values: products about 2^-140
    w[rows // 2] *= np.float32(2.0 ** -70)
    x[T // 2] *= np.float32(2.0 ** -70)
    # a row of wide magnitudes, and one that cancels against every token pair
    w[rows - 1] *= np.exp2(np.arange(K) % 41 - 20).astype(np.float32)
    x[:, 1::2] = np.where(np.arange(K // 2) % 3 == 0, -x[:, ::2], x[:, 1::2])
    return (orc.encode(w.reshape(-1), xpu.BF16).reshape(rows, K), orc.encode(x.reshape(-1), xpu.BF16).reshape(T, K))


@pytest.mark.parametrize("epi,nc,waves", KERNELS)
@pytest.mark.parametrize("T,M,groups", [(1, 16, 1), (16, 144, 1), (17, 16, 2), (33, 48, 1), (50, 16, 3), (50, 16, 5)])
def test_rows_bits(rt, epi, nc, waves, T, M, groups):
    K = 512 * nc
    rows = 2 * M if epi == 2 else M
    w, x = inputs(rows, T, K, 1000 * epi + 10 * nc + T)
    y = np.stack([orc.gemv_canonical(w.reshape(-1), x[t].copy(), rows, K, K, xpu.BF16) for t in range(T)])
    start = orc.uniform(T * M, 5, xpu.BF16).reshape(T, M) if epi == 1 else np.full((T, M), GUARD, np.uint16)
    if epi == 0:
        want = y
    elif epi == 1:
        want = orc.add(start.reshape(-1).copy(), y.reshape(-1).copy()).reshape(T, M)
    else:
        want = orc.silu_mul(y[:, :M].reshape(-1).copy(), y[:, M:].reshape(-1).copy()).reshape(T, M)
    dw, dx = rt.upload(w), rt.upload(x)
    do = rt.upload(np.concatenate([start.reshape(-1), np.full(64, GUARD, np.uint16)]))
    name = f"xpu_q3_pf_rows_e{epi}_c{nc}_w{waves}"
    grid = (M // 16 + 7) // 8 * 8 * groups
    print(f"{name} T={T} M={M} groups={groups} grid={grid}", flush=True)
    try:
        rt.launch_grid(name, grid, 64 * waves, 0, Args().ptr(dw).ptr(dx).ptr(do).u32(M).u32(T).u32(groups))
        rt.synchronize()
        out = rt.download(do, T * M + 64, np.uint16)
    finally:
        for p in (dw, dx, do):
            rt.free(p)
    assert np.all(out[T * M:] == GUARD)
    assert np.array_equal(out[: T * M].reshape(T, M), want)


def test_prompt_of_a_wide_model(rt):
    """The K = 4096 kernels through the engine: hidden and query width 4096
    with an intermediate size that has a kernel. Batched and stepwise prompts
    give the same bits, below and above the token count that takes the MFMA."""
    cfg = qwen3.preset("small")
    cfg.hidden, cfg.intermediate, cfg.heads, cfg.kv_heads, cfg.layers, cfg.vocab = 4096, 2048, 32, 8, 1, 1000
    eng = qwen3.Engine(cfg, max_seq=64, seed=3, gain_std=0.1, runtime=rt)
    try:
        for n in (20, 50):
            ids, got = qwen3.prompt_tokens(n, 11, cfg.vocab), []
            for form in ("stepwise", "batched"):
                eng.set_prefill(form)
                tokens, _, _ = eng.generate(ids, 3, stop_on_eos=False)
                got.append((tokens, eng.logits(), eng.hidden()))
            for a, b in zip(*got):
                assert np.array_equal(a, b)
    finally:
        eng.close()

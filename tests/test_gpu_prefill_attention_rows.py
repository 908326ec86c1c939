"""The batched prompt form's attention on the FP32 MFMA
(xpu_q3_pf_attention_rows) against the one-block-per-token kernel
(xpu_q3_pf_attention, itself checked against the oracle), bit for bit:
query and key counts around the 16-query tile, the 64-key score tile, the
512-position softmax lanes and the 4096-position limit; an infinite V row at
a query's own position, which earlier queries must not see; and NaN codes
past the chunk. Then whole prompts across the 1024-position chunk against the
stepwise prompt."""
import numpy as np
import pytest

import oracle_lib as orc
import xpu_playground_amd as xpu
from xpu_playground_amd import Args, qwen3

pytestmark = pytest.mark.gpu

NAN, INF = 0x7FC0, 0x7F80


@pytest.mark.parametrize("p0,T,heads,kv,gain,inf_at", [
    (0, 1, 4, 2, 1.0, None), (0, 16, 2, 2, 1.0, 5), (0, 17, 4, 1, 8.0, 16), (0, 63, 2, 1, 1.0, 40),
    (0, 65, 4, 2, 30.0, 64), (0, 250, 2, 1, 4.0, 245), (496, 33, 2, 1, 4.0, 500), (1024, 70, 2, 2, 1.0, 1030),
    (2048, 16, 1, 1, 8.0, None), (4064, 32, 2, 1, 1.0, 4090)])
def test_attention_rows_bits(rt, p0, T, heads, kv, gain, inf_at):
    n = p0 + T
    max_seq = n + 5
    q = orc.encode(orc.decode(orc.uniform(T * heads * 128, 1, xpu.BF16), xpu.BF16) * np.float32(gain), xpu.BF16)
    k = np.full((kv, max_seq, 128), NAN, np.uint16)
    v = np.full((kv, max_seq, 128), NAN, np.uint16)
    k[:, :n] = orc.uniform(kv * n * 128, 2, xpu.BF16).reshape(kv, n, 128)
    v[:, :n] = orc.uniform(kv * n * 128, 3, xpu.BF16).reshape(kv, n, 128)
    if inf_at is not None:
        v[:, inf_at, ::7] = INF
    chunked = [np.ascontiguousarray(a.reshape(kv, max_seq, 16, 8).transpose(0, 2, 1, 3)) for a in (k, v)]
    dq, dk, dv = rt.upload(q), rt.upload(chunked[0]), rt.upload(chunked[1])
    da = rt.alloc((T * heads * 128 + 64) * 2)
    scale = float(np.float32(1.0 / np.sqrt(128.0)))
    outs = []
    try:
        for rows in (False, True):
            rt.memset(da, 0xFF, (T * heads * 128 + 64) * 2)
            args = Args().ptr(dq).ptr(dk).ptr(dv).ptr(da).u32(p0)
            print(f"attention {'rows' if rows else 'token blocks'} p0={p0} T={T} heads={heads} kv={kv}", flush=True)
            if rows:
                lds = 16 * ((n + 63) // 64 * 128 + 32) + 8 * 2048
                rt.launch_grid("xpu_q3_pf_attention_rows", heads * ((T + 15) // 16), 512, lds,
                               args.u32(T).u32(heads).u32(kv).u32(max_seq).f32(scale))
            else:
                rt.launch_grid("xpu_q3_pf_attention", heads, 256, 0,
                               args.u32(heads).u32(kv).u32(max_seq).f32(scale), grid_y=T)
            rt.synchronize()
            outs.append(rt.download(da, T * heads * 128 + 64, np.uint16))
    finally:
        for p in (dq, dk, dv, da):
            rt.free(p)
    assert np.all(outs[1][T * heads * 128:] == 0xFFFF)
    got, want = (o[: T * heads * 128].reshape(T, heads, 128) for o in (outs[1], outs[0]))
    bad = (want & 0x7F80) == 0x7F80  # an infinite V row's own outputs: infinite or NaN on both
    assert np.array_equal((got & 0x7F80) == 0x7F80, bad)
    assert np.array_equal(got[~bad], want[~bad])
    if inf_at is not None:
        assert not np.any(bad[: inf_at - p0])  # earlier queries do not see it


@pytest.mark.parametrize("prompt", [129, 1024, 1025, 1061])
def test_prompt_chunks_equal_stepwise(rt, prompt):
    """Every position's K and V through the next decode step's bits, across
    the 1024-position chunk of the batched form."""
    eng = qwen3.Engine(qwen3.preset("small"), max_seq=1100, seed=3, gain_std=0.1, runtime=rt)
    try:
        ids = qwen3.prompt_tokens(prompt, 11, 4096)
        rows = []
        for form in ("stepwise", "batched"):
            eng.set_prefill(form)
            tokens, _, _ = eng.generate(ids, 4, stop_on_eos=False)
            rows.append((tokens, eng.logits(), eng.hidden()))
        for a, b in zip(*rows):
            assert np.array_equal(a, b)
    finally:
        eng.close()

"""The split attention's P.V kernel at the edges of its load batches (512
positions), of the batches in flight (2048) and of the softmax chunks (4096):
logits and hidden state equal those of the one-block-per-head kernel bit for
bit (both state the oracle's order, test_gpu_qwen3_engine.py)."""
import numpy as np
import pytest

import oracle_lib as orc
from xpu_playground_amd import qwen3

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 511, 512, 513, 2047, 2048, 2049, 2575, 4095, 4096, 4097, 4609, 6144, 6163, 8191, 8200]


@pytest.mark.parametrize("shape,positions", [("tiny", EDGES), ("small", [511, 512, 2047, 2100, 4096, 6163])])
def test_split_pv_equals_single_block(rt, shape, positions):
    cfg = orc.config(shape)
    eng = qwen3.Engine(qwen3.config_from(cfg), max_seq=8201, seed=3, gain_std=0.1, runtime=rt)
    ids = qwen3.prompt_tokens(max(positions) + 1, 5, cfg.vocab)
    for p in positions:
        print(f"{shape} position {p}", flush=True)
        got = []
        eng.generate(ids[:p], 1, stop_on_eos=False)  # fills the caches below p
        for split_from in (0, 1):
            eng.set_attention_split(split_from)
            tok = eng.decode(int(ids[p]), p)
            got.append((tok, eng.logits(), eng.hidden()))
        assert got[0][0] == got[1][0]
        assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])
    eng.close()

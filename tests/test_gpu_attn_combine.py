"""The decode o projection's combine of attention segments beyond the four it keeps in registers (exps on a thread per
(segment, head), four outputs per thread) against the CPU oracle, bit for bit: one head to more than the threads hold
(48 heads: the outputs one by one), the fifth segment's first positions, segment counts off the groups of four, and a
position past one batch of 64 segments."""
import numpy as np
import pytest

import lq8
import oracle
from test_gpu_prefill_attention import config, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,positions", [
    (1, 1, (255, 256, 257, 319, 320)), (3, 1, (256, 511, 512, 513)), (6, 2, (256, 448, 700)), (16, 8, (256, 600)),
    (32, 8, (257, 576)), (48, 16, (256, 390)), (2, 1, (1030, 4096, 4097)),
])
def test_decode_past_four_segments(ctx, heads, kv, positions):
    cfg = config(heads, kv, 64 * (max(positions) // 64 + 1), layers=1)
    tensors = oracle.random_q8_tensors(cfg, seed=heads, layer_std=0.1, norm_jitter=0.1)
    model, ref = lq8.Qwen3ForCausalLM.load(ctx, cfg, tensors), oracle.Model(cfg, tensors)
    ids = np.random.default_rng(heads).integers(0, cfg.vocab_size, max(positions) + 1).astype(np.uint32)
    at = 0
    for p in positions:
        for m in (model, ref):
            if p > at:
                m.forward(ids[at:p], at)
        got, want = model.forward(ids[p:p + 1], p), ref.forward(ids[p:p + 1], p)
        assert same_bits(got, want), f"position {p}"
        at = p + 1
    model.free()
    ref.close()

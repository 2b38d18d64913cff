"""The MoE router (k_moe_route: ranks picked round by round, expert lists numbered by count) against the oracle at the
edges of its lane entries: expert counts around 64 and 128 (two and four entries per lane), one expert, every expert
chosen, the largest top-k and batch, tied and underflowing scores, and scores that are not finite."""
import numpy as np
import pytest

import lq8
import oracle
from test_gpu_moe import assert_bits, lq8_cfg
from test_oracle_moe import MoeCfg, moe_tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,k,T", [
    (1, 1, 1), (2, 2, 3), (63, 8, 5), (64, 8, 16), (65, 3, 17), (128, 8, 1), (128, 16, 64), (129, 16, 2), (200, 5, 33),
    (256, 16, 64), (16, 16, 4),
])
def test_routes_match_oracle(ctx, experts, k, T):
    cfg = MoeCfg(hidden_size=32, expert_intermediate_size=32, num_heads=1, num_kv_heads=1, num_experts=experts, top_k=k,
                 max_positions=64, max_batch=64, num_layers=2)
    tens = moe_tensors(cfg, experts + k)
    gpu, orc = lq8.Qwen3MoeLayers.load(ctx, lq8_cfg(cfg), tens), oracle.MoeStack(cfg, tens)
    rng = np.random.default_rng(experts * 100 + T)
    base = rng.standard_normal((2, T, experts)).astype(np.float32)
    # spread, ties between most experts, all equal, and weights that underflow to zero (ties at p = 0)
    for step, scores in enumerate((base, np.round(base), np.zeros_like(base), base * np.float32(200))):
        x = rng.standard_normal((T, cfg.hidden_size)).astype(np.float32)
        pos = np.full(T, step, np.int32)
        y = gpu.forward(x, scores, pos)
        assert_bits(y, orc.forward(x, scores, pos.astype(np.uint32)), f"step {step} hidden")
        ids, w = gpu.routing(T)
        for l in range(2):
            rid, rw = oracle.moe_route(scores[l], k)
            assert np.array_equal(ids[l], rid), f"step {step} layer {l} experts"
            assert_bits(w[l], rw, f"step {step} layer {l} weights")
    gpu.free()
    orc.close()


@pytest.mark.parametrize("experts,k,T", [(65, 5, 1), (65, 5, 6), (128, 8, 6), (256, 16, 6)])
def test_scores_not_finite(ctx, experts, k, T):
    """An infinite or NaN score makes every probability of its row NaN: no entry is larger than another, so the experts
    are the lowest indices in order, whatever the NaNs' bits are.  -inf alone is a probability of zero."""
    cfg = MoeCfg(hidden_size=32, expert_intermediate_size=32, num_heads=1, num_kv_heads=1, num_experts=experts, top_k=k,
                 max_positions=64, max_batch=8, num_layers=2)
    gpu = lq8.Qwen3MoeLayers.load(ctx, lq8_cfg(cfg), moe_tensors(cfg, experts))
    rng = np.random.default_rng(experts + T)
    rows = rng.standard_normal((6, experts)).astype(np.float32)
    rows[0, 9] = np.inf
    rows[1, [7, 40, 64]] = np.array([0x7FC00001, 0x7FFFFFFF, 0xFFC01234], np.uint32).view(np.float32)
    rows[2, ::3] = -np.inf
    rows[3] = -np.inf
    rows[4, [3, 50]] = np.nan, np.inf
    rows[5, k - 1:] = -np.inf  # fewer than k probabilities above zero
    for first in range(0, 6, T):
        scores = np.stack([rows[first:first + T], rows[::-1][first:first + T]])
        gpu.forward(rng.standard_normal((T, cfg.hidden_size)).astype(np.float32), scores, np.zeros(T, np.int32))
        ids, w = gpu.routing(T)
        for l in range(2):
            rid, rw = oracle.moe_route(scores[l], k)
            assert np.array_equal(ids[l], rid), f"rows from {first} layer {l} experts"
            nan = np.isnan(rw)
            assert np.array_equal(np.isnan(w[l]), nan) and np.array_equal(w[l][~nan], rw[~nan]), f"layer {l} weights"
    gpu.free()

"""Prefill attention (k_attn_rows: products on the matrix cores, outputs quantized into the o projection's operand)
against the CPU oracle, bit for bit, where its tiles can go wrong: head groups that do not divide the 16 (or 32) query
vectors of a workgroup, odd head counts (padding blocks of the operand), rows around the tiles and the 64-position
segments, chunks that start inside a segment, a few rows behind a long cache, both vector counts per workgroup, score
differences over the whole range of the exp (its subnormal results and its cutoff among them), and keys and values that
are not finite.  One case takes the GEMM of many tiles with a residual (the o and down projections of a long prompt)."""
import numpy as np
import pytest

import lq8
import oracle

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    nan = np.isnan(a) & np.isnan(b)  # NaNs carry no defined payload
    return a.shape == b.shape and bool(np.all((a.view(np.uint32) == b.view(np.uint32)) | nan))


def config(heads, kv, positions, layers=2):
    return lq8.Qwen3Config(vocab_size=96, hidden_size=96, intermediate_size=64, num_hidden_layers=layers,
                           num_attention_heads=heads, num_key_value_heads=kv, head_dim=128,
                           max_position_embeddings=positions)


# (heads, kv heads, chunk lengths): 32 vectors per workgroup in the 64-head cases (kv heads * tiles >= 1024), else 16
@pytest.mark.parametrize("heads,kv,chunks", [
    (2, 2, (2, 15, 17)), (3, 1, (64, 2)), (5, 5, (65,)), (7, 1, (63, 3, 130)), (6, 2, (31, 34, 64)),
    (16, 1, (70,)), (12, 4, (100, 93)), (64, 64, (513,)), (64, 64, (40, 500)), (66, 33, (600,)), (2, 1, (2300, 3, 2)),
])
def test_prefill_rows_match_oracle(ctx, heads, kv, chunks):
    cfg = config(heads, kv, 64 * ((sum(chunks) + 63) // 64), layers=1 if heads > 16 else 2)
    tensors = oracle.random_q8_tensors(cfg, seed=heads * 100 + kv, layer_std=0.1, norm_jitter=0.1)
    compare_chunks(ctx, cfg, tensors, chunks)


def compare_chunks(ctx, cfg, tensors, chunks):
    model, ref = lq8.Qwen3ForCausalLM.load(ctx, cfg, tensors), oracle.Model(cfg, tensors)
    ids = np.random.default_rng(cfg.num_attention_heads).integers(0, cfg.vocab_size, sum(chunks)).astype(np.uint32)
    at = 0
    for n in chunks:
        got, want = (m.forward_with_intermediates(ids[at:at + n], at) for m in (model, ref))
        for g, w, what in zip(got, want, ("hidden", "final norm", "logits")):
            assert same_bits(g, w), f"chunk at {at}: {what}"
        at += n
    model.free()
    ref.close()


# kv heads * tiles >= 1024 (32 vectors per workgroup) in the cases of 63 heads and more, whose groups of 3, 7 and 11 heads
# leave spare vectors
@pytest.mark.parametrize("heads,kv,chunks", [(4, 2, (70, 130)), (3, 1, (300,)), (66, 22, (480,)), (63, 9, (460,)),
                                             (66, 6, (345,))])
def test_score_differences_past_the_exp_range(ctx, heads, kv, chunks):
    """Large q and k norm weights: scores of a row lie up to hundreds apart, so that exps of differences to the maximum
    are subnormal (below -87.3), zero (below about -104) and past the cutoff (-110), in the first and in later segments,
    with the running maximum rising by as much."""
    cfg = config(heads, kv, 64 * ((sum(chunks) + 63) // 64), layers=1)
    tensors = oracle.random_q8_tensors(cfg, seed=heads + kv, layer_std=0.1, norm_jitter=0.1)
    tensors[4] = (tensors[4] * np.float32(6.0)).astype(np.float32)
    tensors[5] = (tensors[5] * np.float32(6.0)).astype(np.float32)
    compare_chunks(ctx, cfg, tensors, chunks)


def test_long_prompt_residual_gemms(ctx):
    """o and down of 1025 rows into 2016 columns: 33 x 63 output tiles (a ragged last row tile) at 5 and 6 groups of
    blocks, so both run k_gemm_lds with the residual added in place."""
    cfg = lq8.Qwen3Config(vocab_size=96, hidden_size=2016, intermediate_size=1312, num_hidden_layers=1,
                          num_attention_heads=9, num_key_value_heads=3, head_dim=128, max_position_embeddings=1088)
    compare_chunks(ctx, cfg, oracle.random_q8_tensors(cfg, seed=21, layer_std=0.05, norm_jitter=0.1), (1025,))


@pytest.mark.parametrize("heads,kv,n,at", [(4, 2, 50, 40), (4, 2, 130, 70), (64, 64, 513, 500)])
def test_rows_before_a_nonfinite_value_are_not_touched(ctx, heads, kv, n, at):
    """A token whose normed hidden state overflows the activation's f16 scale (one large element under a large norm
    weight) has keys and values that are not finite: the rows before it keep their bits, and the rows from it on have
    NaN attention outputs (which the o projection's quantizer takes as zeros)."""
    cfg = config(heads, kv, 64 * ((n + 63) // 64), layers=1)
    tensors = oracle.random_q8_tensors(cfg, seed=9, norm_jitter=0.1)
    H = cfg.hidden_size
    table = oracle.dequantize_q8_0(tensors[0], cfg.vocab_size * H).reshape(cfg.vocab_size, H).copy()
    table[7] = 0.0
    table[7, 5] = 1.0  # normed to sqrt(96): 2e6 sqrt(96) / 127 is above 65504, an ordinary row's 3 * 2e6 / 127 is not
    tensors[0] = oracle.quantize_q8_0(table)
    tensors[2] = np.full(H, 2e6, np.float32)
    model, ref = lq8.Qwen3ForCausalLM.load(ctx, cfg, tensors), oracle.Model(cfg, tensors)
    ids = np.random.default_rng(3).integers(8, cfg.vocab_size, n).astype(np.uint32)
    ids[at] = 7
    got, want = (m.forward_with_intermediates(ids, 0)[0] for m in (model, ref))
    scales = oracle.quantize_q8_0(oracle.rms_norm(want[0], tensors[2], cfg.rms_norm_eps)).reshape(n, H // 32, 34)
    inf = np.ascontiguousarray(scales[:, :, :2]).view(np.float16)[..., 0] == np.inf
    assert inf[at].any() and not np.delete(inf, at, axis=0).any()
    assert same_bits(got, want)
    model.free()
    ref.close()

"""The GEMM of many tiles (k_gemm_lds: operands shared through LDS) against the oracle at the edges of its range: the
smallest tile counts that take each of its block shapes, ragged rows and columns (one row or column in the last tile,
a last block of one 32-row tile), one block, odd block and pair counts, a group of 8 blocks and one more; and f16 scales
that are infinite, zero or subnormal beside a padding block."""
import numpy as np
import pytest

import lq8
import oracle
from test_gpu_q8 import assert_parity, gemm_case, normal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (353, 5441, 32), (383, 5473, 64), (513, 3841, 96), (1023, 2049, 256), (1024, 2048, 1312), (2047, 1025, 544),
    (2049, 1000, 1024), (1025, 3940, 1056),           # 64 x 64 blocks: from 12 m-tiles and 2048 tiles
    (97, 98273, 32), (129, 78625, 96), (1023, 12289, 64), (2049, 6049, 288), (160, 78656, 544),  # 64 x 128: 12288 tiles
    (33, 32769, 64), (2, 65505, 96), (352, 5985, 64),  # few m-tiles: the other kernels
    (1024, 2048, 320),                                 # 2 to 4 groups of blocks below 8192 tiles: the other kernels
    (65536, 32, 64), (129, 78625, 512),                # one n-tile, 5 m-tiles of whole groups: the other kernels
])
def test_many_tiles_match_oracle(ctx, m, n, k):
    y, ref = gemm_case(ctx, m, n, k, m + n + k)
    assert_parity(y, ref)


# the last tile count of the other kernels and the first of k_gemm_lds, at 2 to 4 groups of blocks, at 5, and at more with
# three, four, five and seven 64 x 64 blocks on the fullest CU
@pytest.mark.parametrize("m,k,below,above", [
    (1024, 320, 8160, 8192), (2048, 288, 1568, 1600), (2051, 288, 2016, 2048), (416, 1056, 7552, 7584),
    (416, 1312, 5152, 5216), (410, 1312, 8960, 8992), (1248, 1312, 2720, 2752), (416, 1312, 9824, 9856),
    (416, 1312, 14624, 14656),
])
def test_both_sides_of_the_tile_rule(ctx, m, k, below, above):
    for n in (below, above):
        y, ref = gemm_case(ctx, m, n, k, m + n + k)
        assert_parity(y, ref)


@pytest.mark.parametrize("m,n,k", [(354, 5441, 96), (98, 98273, 96)])
def test_scale_edges(ctx, m, n, k):
    wf = normal((n, k), 0.02, 40)
    wf[::3] *= np.float32(1e-3)   # f16 subnormal scales
    wf[5, 32:] = 0.0              # zero blocks
    wf[n - 1, 64:] = 9e6          # the scale overflows f16
    x = normal((m, k), 1.0, 41)
    x[0] *= np.float32(1e-6)
    x[1, 64:] = 0.0
    x[2, :32] = -9e6
    blocks = oracle.quantize_q8_0(wf)
    w = lq8.Q8Weight.from_blocks(ctx, blocks, n, k)
    y = lq8.Linear.new(w).forward(x).reshape(m, n)
    w.free()
    ref = oracle.gemm_q8_0(blocks, n, k, x)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(y), nan)
    assert np.array_equal(y.view(np.uint32)[~nan], ref.view(np.uint32)[~nan])

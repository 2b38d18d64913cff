"""The activation quantizers at their edges.  RMSNorm fused (k_rms_quantize_act, a workgroup per row, and
k_rms_quantize_waves, a wave per row, for more rows): one block, odd block counts, 1024 and one block more, the largest
width, row counts around the 32-row padding, the last row count of one kernel and the first of the other, and more rows
than a launch of one workgroup per row may have threads.  Plain rows: both kernels (by rows up to 1024 waves of the
tile-shaped one), odd block counts, one row, and 1024 waves and the next."""
import numpy as np
import pytest

import lq8
import oracle
from test_gpu_q8 import act_operand, assert_blocks_equal, edge_blocks, normal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(2, 32), (33, 96), (31, 288), (32, 992), (5, 1024), (65, 1056), (3, 1824), (64, 2016),
                                 (1, 2048), (130, 2048)])
def test_rms_quantize_widths(ctx, m, k):
    x = normal((m, k), 1.0, 11 * k + m)
    x[0, : k // 2] = 0.0   # zero blocks
    x[m - 1] *= np.float32(1e-6)  # the mean beside eps
    w = (1.0 + 0.1 * normal(k, 1.0, k)).astype(np.float32)
    ref = oracle.quantize_q8_0(oracle.rms_norm(x, w, 1e-6))
    assert_blocks_equal(act_operand(ctx, lq8.ACT_RMSNORM, x, m, k, w), ref)


@pytest.mark.parametrize("m,k", [(1280, 32), (1281, 32), (1280, 1024), (1281, 1024), (1300, 480), (1536, 1056), (1537, 1056),
                                 (1536, 2048), (1537, 2048), (4099, 224)])
def test_rms_quantize_many_rows(ctx, m, k):
    x = normal((m, k), 1.0, 17 * k + m)
    x[m // 2] = 0.0
    x[m - 1] *= np.float32(1e-6)
    w = (1.0 + 0.1 * normal(k, 1.0, k)).astype(np.float32)
    ref = oracle.quantize_q8_0(oracle.rms_norm(x, w, 1e-6))
    assert_blocks_equal(act_operand(ctx, lq8.ACT_RMSNORM, x, m, k, w), ref)


def test_rms_quantize_rows_past_a_grid(ctx):
    """2^24 rows: a workgroup of 256 threads per row would be 2^32 threads, which a launch refuses."""
    tile, k = 4096, 32
    x = normal((tile, k), 1.0, 3)
    w = (1.0 + 0.1 * normal(k, 1.0, k)).astype(np.float32)
    ref = oracle.quantize_q8_0(oracle.rms_norm(x, w, 1e-6))
    got = act_operand(ctx, lq8.ACT_RMSNORM, np.tile(x, (4096, 1)), 4096 * tile, k, w).reshape(4096, -1)
    assert np.array_equal(got, np.broadcast_to(ref, got.shape))


@pytest.mark.parametrize("m,k", [(1, 32), (2, 288), (33, 2080), (31, 12256), (512, 2048), (513, 2048), (1100, 1056),
                                 (4096, 256), (4097, 224)])
def test_plain_quantize_kernels(ctx, m, k):
    x = normal((m, k), 1.0, 13 * k + m)
    x[m - 1, : k // 2] = 0.0
    e = edge_blocks()
    if x.size >= e.size:
        x.reshape(-1)[x.size - e.size:] = e.reshape(-1)
    assert_blocks_equal(act_operand(ctx, lq8.ACT_PLAIN, x, m, k), oracle.quantize_q8_0(x))

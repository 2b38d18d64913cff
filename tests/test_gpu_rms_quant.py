"""RMSNorm fused into the activation quantizer (k_rms_quantize_act, a workgroup per row) at the edges of its two widths:
one block, odd block counts, 1024 and one block more, the largest width, and row counts around the 32-row padding."""
import numpy as np
import pytest

import lq8
import oracle
from test_gpu_q8 import act_operand, assert_blocks_equal, normal

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

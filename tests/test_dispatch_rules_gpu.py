"""The rules by which a launch picks its kernel form or tile, at the sizes where they change over (against the oracle)."""
import numpy as np
import pytest

import oracle
from helpers import make_qweight, normal_bf16, rel_l2, to_device
from test_attention_gpu import _sdpa_case

pytestmark = pytest.mark.gpu


def test_gemv_tiling_is_looked_up_by_shape_and_policy(fk):
    """Shapes and tile policies in turn, each twice: what one call looked up is never another's."""
    cases = [(n, 64 * g, rows) for n, g, rows in ((896, 14, 0), (897, 14, 0), (896, 76, 0), (896, 14, 3), (64, 14, 0))]
    kept = [(W := make_qweight(7 + i, n, k, 4), to_device(fk, W), normal_bf16(i, k), fk.DeviceBuffer(2 * n), rows)
            for i, (n, k, rows) in enumerate(cases)]
    try:
        for _ in range(2):
            for W, dW, x, y, rows in kept:
                fk.set_gemv_policy(rows, 0)
                fk.qgemv(dW, fk.DeviceBuffer.from_numpy(x), None, y)
                assert rel_l2(y.to_numpy(np.uint16), oracle.linear_acc(W, x)) <= 5e-3
    finally:
        fk.set_gemv_policy(0, 0)


@pytest.mark.parametrize("heads,length", [((14, 2, 64), 4096), ((14, 2, 64), 4097), ((10, 2, 64), 130), ((16, 2, 128), 4200)])
def test_attention_tiles_of_groups_of_more_than_four_heads(fk, heads, length):
    n_heads, n_kv, dim = heads
    _sdpa_case(fk, n_heads, n_kv, dim, dim, length, length + 3, seed=length)

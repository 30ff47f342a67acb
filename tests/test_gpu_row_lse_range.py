"""row_lse's operands (packing, mask and the range check in one launch): results against float64 where the units do not
fill the launch's workgroups or take several rounds of them, and one value out of range at each corner of either
operand refused."""

import numpy as np
import pytest
import torch

from oracle import brute
from test_gpu_kernels import _lse_tol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,m,K", [(1, 1, 1), (31, 33, 16), (33, 31, 17), (32, 64, 128), (40_000, 70, 100)])
def test_operands_of_every_size(hip, rows, m, K):
    rng = np.random.default_rng(rows + m + K)
    xa, ya = rng.normal(size=(rows, K)).astype(np.float32), rng.normal(size=(m, K)).astype(np.float32)
    out = hip.row_lse(torch.from_numpy(xa).cuda(), torch.from_numpy(ya).cuda()).cpu().numpy()
    assert out.shape == (rows,)
    assert np.all(np.abs(out - brute.row_lse(xa, ya)) <= _lse_tol(xa, ya))


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -1e14])
@pytest.mark.parametrize("rows,m,K", [(1, 1, 1), (70, 45, 19)])
def test_one_value_out_of_range_is_refused(hip, bad, rows, m, K):
    for which in (0, 1):
        for corner in ((0, 0), (-1, -1)):
            ab = [torch.ones(rows, K, device="cuda"), torch.ones(m, K, device="cuda")]
            ab[which][corner] = bad
            with pytest.raises(ValueError, match="coordinates must be finite"):
                hip.row_lse(*ab)

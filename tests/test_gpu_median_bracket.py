"""The exact median's bracket: two passes over approximate costs from the fp16 matrix cores find the few pairs whose
float64 costs are needed. Against the median of the dense float64 costs at the edges of the tiles (32 points), of the row
blocks (64 rows, 32 above 64 coordinates) and of the K chunks (16 coordinates), at scales far outside float32, and where
the bracket cannot narrow (a point so far out that every other cost falls into the lowest bin), which sends the call to
the passes over every cost. The two sums differ in their order only: 1e-12 relative (128 terms, 2^-53 each, with a margin
of 70)."""

import numpy as np
import pytest

from test_gpu_median import dense_median

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(1, 33), (31, 32), (33, 31), (63, 65), (64, 64), (65, 63), (129, 1), (1025, 700)])
@pytest.mark.parametrize("d", [1, 8, 16, 17, 64, 65, 81, 97, 113, 128])
def test_bracket_at_tile_edges(hip, n, m, d):
    rng = np.random.default_rng(n * 7 + m * 3 + d)
    x, y = rng.standard_normal((n, d)), rng.standard_normal((m, d)) * 0.7 + 0.3
    want = dense_median(x, y)
    assert abs(hip.cost_median(x, y, "cuda") - want) <= 1e-12 * want


@pytest.mark.parametrize("e", [-400, -140, 140, 400])
def test_a_power_of_two_scales_the_median_exactly(hip, e):
    rng = np.random.default_rng(3)
    x, y = rng.standard_normal((900, 20)), rng.standard_normal((700, 20)) + 0.5
    one = hip.cost_median(x, y, "cuda")
    assert hip.cost_median(np.ldexp(x, e), np.ldexp(y, e), "cuda") == np.ldexp(one, 2 * e)


@pytest.mark.parametrize("n,far", [(300, 1e8), (2100, 1e8), (2100, 30.0)])
def test_one_point_far_out(hip, n, far):
    rng = np.random.default_rng(n)
    x, y = rng.standard_normal((n, 3)), rng.standard_normal((n, 3))
    x[n // 2, 1] = far
    want = dense_median(x, y)
    assert abs(hip.cost_median(x, y, "cuda") - want) <= 1e-12 * want

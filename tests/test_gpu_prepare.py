"""A solve's clouds prepared on the GPU (sk_cloud_stats_f64, sk_centre_f64, sk_prepare_cloud_f64) against the host's own
steps: the centre and the sampled mean cost to the rounding of a float64 sum (1e-13 relative: up to 2e4 terms of one sign,
or of the points' size, 2^-53 each, added in another order), the packed pieces, scale and norms bit for bit from the same
normalisation, and what was refused stays refused."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("n,m", [(1, 1), (1, 70), (63, 65), (1000, 37), (9001, 4003)])
@pytest.mark.parametrize("d", [1, 3, 16, 64, 65, 127, 128])
def test_stats_and_packing_match_the_host(hip, n, m, d):
    from trnopt.sinkhorn import _sample_pairs, normalization
    rng = np.random.default_rng(n + 3 * m + d)
    x, y = rng.standard_normal((n, d)) * 2.0 + 0.5, rng.standard_normal((m, d)) - 0.25
    X, Y = hip.to_device_f64(x, DEV), hip.to_device_f64(y, DEV)
    stat = torch.empty(d + 3, dtype=torch.float64, device=DEV)
    hip.cloud_stats(X, Y, stat, _sample_pairs(n, m))
    center, scale = normalization(x, y)
    got = stat.cpu().numpy()
    assert np.abs(got[:d] - center).max() <= 1e-13 * np.abs(np.concatenate([x, y])).max()
    assert abs(got[d] - scale) <= 1e-13 * scale
    np.testing.assert_array_equal(hip.centred(X, stat).cpu().numpy(), x - got[:d])
    # packing from the same centre and scale
    lw = np.full(n, -np.log(n))
    a = hip.HipCloud.prepared(X, stat, stat[d + 1:d + 2], lw)
    xs = (x - got[:d]) / np.sqrt(got[d])
    b = hip.HipCloud(xs, lw, DEV)
    own = hip.PACKED_HEADER_BYTES + (b.pk.numel() - hip.PACKED_HEADER_BYTES) // 2
    assert torch.equal(a.pk[:8], b.pk[:8])                                       # max |coordinate| and scale
    assert torch.equal(a.pk[hip.PACKED_HEADER_BYTES:own], b.pk[hip.PACKED_HEADER_BYTES:own])
    sa, sb = a.sq.cpu().numpy(), b.sq.cpu().numpy()
    assert np.all(np.abs(sa - sb) <= np.spacing(sb)) and not sa[n:].any()        # sums in another order, one cast each
    assert float(stat[d + 1]) == np.abs(xs).max()
    assert all(torch.equal(getattr(a, k), getattr(b, k)) for k in ("log_w", "w", "log_w_lo"))


def test_points_that_all_coincide_keep_unit_scale(hip):
    from trnopt import Backend, SinkhornOptions, sinkhorn
    x, y = np.full((40, 5), 3.0), np.full((30, 5), 3.0)
    for how in ("mean", "median"):
        r = sinkhorn(x, y, opts=SinkhornOptions(kernel="hip", backend=Backend.preset("rocm"), normalize=how, max_iters=3,
                                                fixed_iters=True))
        assert r.cost_scale == 1.0 and np.isfinite(r.f).all()


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 1e16])
@pytest.mark.parametrize("how", ["mean", "median", False, (np.zeros(4), 1.0)])
def test_points_out_of_range_are_refused(hip, bad, how):
    from trnopt import Backend, SinkhornOptions, sinkhorn
    x, y = np.random.default_rng(0).standard_normal((50, 4)), np.random.default_rng(1).standard_normal((60, 4))
    y[7, 2] = bad
    if how in ("mean", "median") and bad == 1e16:
        how = (np.zeros(4), 1.0)             # (normalised, one far point is in range)
    opts = SinkhornOptions(kernel="hip", backend=Backend.preset("rocm"), normalize=how, max_iters=3, fixed_iters=True)
    with pytest.raises(ValueError, match="coordinates must be finite"):
        sinkhorn(x, y, opts=opts)


@pytest.mark.parametrize("center", [0.5, np.full(4, 0.5), np.full((1, 4), 0.5), np.full((50, 1), 0.5)])
def test_given_centres_of_every_shape(hip, center):
    """normalize=(center, scale) takes whatever broadcasts against the points, as the host's subtraction does."""
    from trnopt import Backend, SinkhornOptions, sinkhorn
    x, y = np.random.default_rng(0).standard_normal((50, 4)), np.random.default_rng(1).standard_normal((50, 4))
    kw = dict(eps=0.3, max_iters=20, fixed_iters=True)
    hipr = sinkhorn(x, y, opts=SinkhornOptions(kernel="hip", backend=Backend.preset("rocm"), normalize=(center, 2.0), **kw))
    cpu = sinkhorn(x, y, opts=SinkhornOptions(normalize=(center, 2.0), **kw))
    assert np.abs(hipr.f - cpu.f).max() <= 1e-5 * np.abs(cpu.f).max()
    np.testing.assert_array_equal(hipr.center, cpu.center)

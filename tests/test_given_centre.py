"""normalize=(centre, scale) on the fused path means (x - centre) / sqrt(scale) as numpy broadcasts it, whatever the
centre's shape: one number, one per coordinate, or one per point. What the set-up hands to the GPU preparation (points,
and the centre and scale that it takes off them, one per coordinate of those points) is checked on the host."""

import sys

import numpy as np
import pytest
import torch

import trnopt
from trnopt import hip_sinkhorn as hk

sk = sys.modules["trnopt.sinkhorn"]            # (trnopt.sinkhorn the name is the function)
CPU = torch.device("cpu")


class _Stop(Exception):
    pass


def _normalised(monkeypatch, x, y, center, scale):
    """The points of both clouds as the preparation would see them."""
    opts = sk.SinkhornOptions(normalize=(center, scale))
    seen = []

    def prepared(pts, stat, rng, log_w, off=None, role=0):
        n, d = pts.shape
        stat = stat.numpy()
        assert stat.size >= d + 1 + 2, "the statistics end before the points' last coordinate"
        seen.append((pts.numpy() - stat[:d]) / np.sqrt(stat[d]))
        if len(seen) == 2:
            raise _Stop

    monkeypatch.setattr(hk, "to_device_f64", lambda p, dev: torch.from_numpy(np.array(p, dtype=np.float64)))
    monkeypatch.setattr(hk.HipCloud, "prepared", prepared)
    p = sk._prepare(x, y, None, None, opts, None, None, True)
    with pytest.raises(_Stop):
        sk._hip_setup(p, opts, CPU)
    return seen


@pytest.mark.parametrize("n,d,shape", [(6, 4, ()), (6, 4, (1,)), (6, 4, (4,)), (6, 4, (1, 1)), (6, 4, (1, 4)), (6, 4, (6, 1)),
                                       (6, 4, (6, 4)), (4, 4, (4, 1)), (4, 4, (1, 4)), (4, 4, (4, 4)), (1, 1, (1, 1)),
                                       (1, 5, (1, 5)), (5, 1, (5, 1)), (5, 1, (7,)), (5, 1, (1, 7)), (5, 1, (5, 7)), (5, 1, (5,))])
def test_a_centre_is_taken_off_as_numpy_broadcasts_it(monkeypatch, n, d, shape):
    rng = np.random.default_rng(n * 10 + d)
    x, y, center = rng.normal(size=(n, d)), rng.normal(size=(n, d)), rng.normal(size=shape)
    for got, p in zip(_normalised(monkeypatch, x, y, center, 2.25), (x, y)):
        np.testing.assert_array_equal(got, (p - center) / 1.5)


@pytest.mark.parametrize("n,m,d,shape", [(6, 5, 4, (4, 1)), (6, 6, 4, (3,)), (6, 6, 4, (4, 1)), (6, 6, 4, (2, 6, 4)), (6, 6, 4, (1, 1, 4))])
def test_a_centre_that_does_not_fit_is_refused(monkeypatch, n, m, d, shape):
    rng = np.random.default_rng(0)
    with pytest.raises(ValueError):
        _normalised(monkeypatch, rng.normal(size=(n, d)), rng.normal(size=(m, d)), rng.normal(size=shape), 1.0)


@pytest.mark.gpu
@pytest.mark.parametrize("n,d,shape", [(24, 24, (24, 1)), (24, 24, (24,)), (30, 1, (5,)), (30, 1, (1, 70))])
def test_a_solve_agrees_with_the_torch_path(hip, n, d, shape):
    """1e-5 of the largest potential: the float32 loop's rounding (as the solver tests)."""
    print(f"given centre {shape}: {n} x {n}, d {d}", flush=True)
    rng = np.random.default_rng(n + d)
    x, y, center = rng.normal(size=(n, d)), rng.normal(size=(n, d)), rng.normal(size=shape)
    kw = dict(eps=0.5, max_iters=15, fixed_iters=True, normalize=(center, float(2 * d)))
    got = sk.sinkhorn(x, y, opts=sk.SinkhornOptions(kernel="hip", backend=trnopt.Backend.preset("rocm"), **kw))
    want = sk.sinkhorn(x, y, opts=sk.SinkhornOptions(**kw))
    assert np.abs(got.f - want.f).max() <= 1e-5 * np.abs(want.f).max()
    assert np.abs(got.g - want.g).max() <= 1e-5 * np.abs(want.g).max()
    np.testing.assert_array_equal(got.center, center)


@pytest.mark.gpu
def test_a_batch_needs_one_number_of_normalised_coordinates(hip):
    x, y = np.random.default_rng(0).normal(size=(2, 20, 1))
    rocm = trnopt.Backend.preset("rocm")
    opts = [sk.SinkhornOptions(kernel="hip", backend=rocm, normalize=(c, 1.0)) for c in (np.ones(1), np.ones(20))]
    with pytest.raises(ValueError, match="one d"):
        sk.sinkhorn_batch([dict(x=x, y=y, opts=o) for o in opts])

"""Points that may not be written to (memory-mapped files, broadcast views) go to the GPU without a warning, as they did while
the host made a copy of them; torch warns about a tensor over such memory, which a caller may have turned into an error."""

import warnings

import numpy as np
import pytest
import torch

from trnopt import hip_sinkhorn as hk


def _readonly(kind, tmp_path):
    x = np.random.default_rng(0).normal(size=(60, 5))
    if kind == "mapped":
        np.save(tmp_path / "x.npy", x)
        return np.load(tmp_path / "x.npy", mmap_mode="r"), x
    if kind == "broadcast":
        return np.broadcast_to(x[0], (60, 5)), np.tile(x[0], (60, 1))
    x.setflags(write=False)
    return x, x


@pytest.mark.parametrize("kind", ["mapped", "broadcast", "flag"])
def test_copied_without_a_warning(kind, tmp_path):
    r, want = _readonly(kind, tmp_path)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        got = hk.to_device_f64(r, torch.device("cpu"))
    np.testing.assert_array_equal(got.numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["mapped", "broadcast", "flag"])
def test_a_solve_takes_them(hip, kind, tmp_path):
    from trnopt import Backend, SinkhornOptions, sinkhorn
    from trnopt.sinkhorn import normalization
    r, want = _readonly(kind, tmp_path)
    y = np.random.default_rng(1).normal(size=(70, 5))
    opts = SinkhornOptions(kernel="hip", backend=Backend.preset("rocm"), eps=0.3, max_iters=10, fixed_iters=True)
    big = np.broadcast_to(y[0], (20_000, 5))
    with warnings.catch_warnings():
        warnings.simplefilter("error", UserWarning)
        got = sinkhorn(r, y, opts=opts)
        normalization(big, r, how="median", device="cuda")
    np.testing.assert_array_equal(got.f, sinkhorn(want.copy(), y, opts=opts).f)

"""The loop of small problems as one resident launch (sk_loop_run_resident_f32 wherever it fits, TRNOPT_HIP_LOOP=1) against
the launch-by-launch loop: potentials, iteration counts, errors and convergence bit for bit, over the forms the loop has
(fixed, to convergence, eps schedule, stages, unbalanced with targets, weights), sizes at the edges of the 32-row blocks,
256-row groups and its largest (192 tiles), every width of kernel, one to four workgroups per row block, calls of several lengths, and clouds without a
log2-unit copy; and from several streams and threads."""

import ctypes

import numpy as np
import pytest
import torch

from trnopt import Backend
from trnopt import hip_sinkhorn as hk
from trnopt.sinkhorn import SinkhornOptions, sinkhorn

pytestmark = pytest.mark.gpu
ROCM = Backend.preset("rocm")

FORMS = {
    "fixed": dict(eps=0.1, max_iters=12, fixed_iters=True),
    "raw": dict(eps=0.1, max_iters=12, fixed_iters=True, normalize=False),
    "converged": dict(eps=0.1, tol=1e-5, max_iters=400),
    "schedule": dict(eps=0.05, eps_start=1.0, eps_decay=0.8, max_iters=30, fixed_iters=True),
    "schedule-checked": dict(eps=0.1, eps_start=0.5, eps_decay=0.7, max_iters=300, tol=1e-4, check_every=3),
    "stages": dict(eps=0.05, rho=(1.0, 50.0), eps_stages=(1.0, 0.4, 0.15), check_every=5, tol=1e-5, max_iters=600),
    "unbalanced": dict(eps=0.1, rho=(1.0, 50.0), tol=1e-6, max_iters=600),
}


def _clouds(n, m, d):
    rng = np.random.default_rng(n * 31 + m * 7 + d)
    a, b = rng.uniform(0.5, 1.5, n), rng.uniform(0.5, 1.5, m)
    return rng.normal(size=(n, d)), rng.normal(size=(m, d)) * 0.9 + 0.3, a / a.sum(), b / b.sum()


def _both(monkeypatch, n, m, d, o, x=None):
    x0, y, a, b = _clouds(n, m, d)
    kw = dict(a_target=a[::-1].copy(), b_target=b) if "rho" in o else {}
    out = []
    lib = hk.lib()
    run = lib.sk_loop_try_resident_f32
    for v in ("0", "1"):
        resident = []                        # the form that each call of the loop's iterations takes
        monkeypatch.setenv("TRNOPT_HIP_LOOP", v)
        monkeypatch.setattr(lib, "sk_loop_try_resident_f32",
                            lambda L, k, stream: (resident.append(lib.sk_loop_resident(L)), run(L, k, stream))[1])
        out.append(sinkhorn(x0 if x is None else x, y, a, b, SinkhornOptions(kernel="hip", backend=ROCM, **o), **kw))
        assert resident and set(resident) == {int(v)}
    monkeypatch.setattr(lib, "sk_loop_try_resident_f32", run)
    return out


def _same(p, q):
    assert (p.iterations, p.converged) == (q.iterations, q.converged)
    assert p.error == q.error or (np.isnan(p.error) and np.isnan(q.error))
    np.testing.assert_array_equal(p.f, q.f)
    np.testing.assert_array_equal(p.g, q.g)


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("n,m,d", [(137, 91, 5), (700, 900, 30), (257, 31, 64), (1300, 400, 40)])
def test_every_form_bit_for_bit(hip, monkeypatch, form, n, m, d):
    print(f"resident {form} {n} x {m} d {d}", flush=True)
    _same(*_both(monkeypatch, n, m, d, FORMS[form]))


@pytest.mark.parametrize("n,m,d", [(1, 1, 1), (31, 33, 16), (32, 32, 17), (33, 1, 40), (255, 256, 48), (256, 257, 80),
                                   (513, 100, 96), (64, 6144, 8), (6144, 64, 112), (6144, 6100, 33), (2000, 1900, 128),
                                   (2700, 2600, 40), (4000, 3900, 20), (280, 4096, 64)])
def test_sizes_bit_for_bit(hip, monkeypatch, n, m, d):
    print(f"resident {n} x {m} d {d}", flush=True)
    _same(*_both(monkeypatch, n, m, d, dict(eps=0.3, max_iters=5, fixed_iters=True)))


@pytest.mark.parametrize("n,m,fits", [(6144, 6144, 1), (6145, 40, 0), (40, 6145, 0)])
def test_the_largest_loop_that_fits(hip, monkeypatch, n, m, fits):
    monkeypatch.setenv("TRNOPT_HIP_LOOP", "1")
    x, y, a, b = _clouds(n, m, 3)
    loop = hip.DeviceLoop(hip.HipCloud(x, np.log(a), "cuda"), hip.HipCloud(y, np.log(b), "cuda", role=1), eps=1.0, rho_x=None,
                          rho_y=None, sched=[], stages=[], tol=0.0, stage_tol=0.0, max_iters=1, check_every=1,
                          stage_max_iters=1, fixed_iters=True, balanced=True)
    assert hip.lib().sk_loop_resident(ctypes.byref(loop._L)) == fits
    assert (hip.lib().sk_loop_repairs_offset(ctypes.byref(loop._L)) > 0) == bool(fits)


def test_clouds_without_a_log2_copy(hip, monkeypatch):
    """All-zero coordinates have no log2-unit copy: the loop then works in accumulator units."""
    _same(*_both(monkeypatch, 50, 40, 4, dict(eps=0.5, max_iters=7, fixed_iters=True, normalize=False), x=np.zeros((50, 4))))


def test_mixed_calls_continue_one_loop(hip, monkeypatch):
    """Iterations in calls of 1, 2, 5, ... (1 runs as launches, more as one) over a schedule, against all in launches."""
    x, y, a, b = _clouds(300, 200, 20)
    got = []
    for v in ("0", "1"):
        monkeypatch.setenv("TRNOPT_HIP_LOOP", v)
        X = hip.HipCloud(x, np.log(a), "cuda", role=0)
        Y = hip.HipCloud(y, np.log(b), "cuda", role=1)
        loop = hip.DeviceLoop(X, Y, eps=0.2, rho_x=None, rho_y=None, sched=[2.0, 1.5, 1.0, 0.7, 0.5], stages=[], tol=0.0,
                              stage_tol=0.0, max_iters=100, check_every=4, stage_max_iters=10, fixed_iters=False, balanced=True)
        loop.init()
        for k in (2, 1, 1, 3, 1, 5, 2, 4):
            loop.enqueue(k)
        st = loop.read_state()
        got.append((loop.fh.cpu(), loop.gh.cpu(), st.it, st.err, st.checks, st.eps, bytes(X.pk[:40].cpu().numpy())))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert got[0][2:6] == got[1][2:6]
    assert got[0][6][:28] == got[1][6][:28]              # the copy's tag as the launches leave it


@pytest.mark.parametrize("form", ["fixed", "converged", "stages"])
def test_a_launch_that_gives_up_is_run_again_as_launches(hip, monkeypatch, form):
    """With a single poll allowed, any wait gives up: the solve goes on in launches from there with the same result."""
    monkeypatch.setenv("TRNOPT_HIP_LOOP_POLLS", "1")
    loops, init = [], hip.DeviceLoop.init
    monkeypatch.setattr(hip.DeviceLoop, "init", lambda loop: (loops.append(loop), init(loop))[1])
    _same(*_both(monkeypatch, 400, 900, 30, FORMS[form]))
    assert [l.repairs() > 0 for l in loops] == [False, True]


def test_threads_and_streams_side_by_side(hip, monkeypatch):
    """Four threads, two on the default stream (resident launches) and two on streams of their own (launches)."""
    import threading
    monkeypatch.setenv("TRNOPT_HIP_LOOP", "1")
    o = SinkhornOptions(kernel="hip", backend=ROCM, eps=0.1, max_iters=60, fixed_iters=True)
    data = [_clouds(400 + 50 * k, 350, 12) for k in range(4)]
    want = [sinkhorn(x, y, a, b, o) for x, y, a, b in data]
    got = [None] * 4

    def run(k):
        x, y, a, b = data[k]
        with torch.cuda.stream(torch.cuda.Stream() if k % 2 else torch.cuda.default_stream()):
            for _ in range(3):
                got[k] = sinkhorn(x, y, a, b, o)

    ts = [threading.Thread(target=run, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for p, q in zip(want, got):
        _same(p, q)

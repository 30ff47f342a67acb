"""Two on-device loops on the same packed clouds, stepped in turn over different eps schedules and stages. x's one log2-unit
copy changes hands: a loop that finds a copy another loop has still to make, for an eps that is not its own, must not
declare it made: after every step the header's copy is either none or the tiles of its own eps."""

import numpy as np
import pytest
import torch

from conftest import inf_rel

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
KW = dict(rho_x=None, rho_y=None, tol=0.0, stage_tol=1e9, max_iters=40, check_every=1, stage_max_iters=1000, fixed_iters=True,
          balanced=True)
FORMS = {     # (first loop, second loop): eps, sched, stages
    "other eps": ((0.1, [0.8, 0.4, 0.2], []), (0.15, [0.6, 0.3], [])),
    "one fixed": ((0.1, [0.8, 0.4, 0.2], []), (0.3, [], [])),
    "crossing": ((0.2, [0.8, 0.4], []), (0.2, [0.4, 0.8, 0.4, 0.4, 0.4], [])),
    "stages": ((0.1, [], [0.8, 0.4]), (0.4, [], [])),
}


def _clouds(hip, n, m, d):
    rng = np.random.default_rng(n + m + d)
    x, y = rng.normal(size=(n, d)) * 0.3, rng.normal(size=(m, d)) * 0.3 + 0.1
    return (hip.HipCloud(x, np.full(n, -np.log(n)), DEV, role=0), hip.HipCloud(y, np.full(m, -np.log(m)), DEV, role=1))


def _loop(hip, X, Y, form):
    eps, sched, stages = form
    return hip.DeviceLoop(X, Y, eps=eps, sched=sched, stages=stages, **KW)


def _header_is_true(hip, X, n, m, d, known):
    """The header's copy is none, or the copy of one of the loops' eps."""
    w = X.pk[:64].cpu().numpy()
    c, pending = float(w.view(np.float32)[2]), int(w.view(np.int32)[6])
    if c == 0.0:
        return
    assert pending == 0
    head = hip.PACKED_HEADER_BYTES
    tiles = X.pk[head + (X.pk.numel() - head) // 2:].cpu()
    for e in known:
        A, B = _clouds(hip, n, m, d)
        hip.bake_log2(A, B, hip.scalars(e, 1.0, DEV))
        if float(A.pk[:64].cpu().numpy().view(np.float32)[2]) == c:
            assert torch.equal(tiles, A.pk[head + (A.pk.numel() - head) // 2:].cpu()), e
            return
    raise AssertionError(f"a copy of no loop's eps (c {c})")


@pytest.mark.parametrize("step", [1, 2])
@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("n,m,d", [(300, 200, 20), (1300, 900, 64), (10_273, 300, 30)])
def test_the_header_says_what_the_tiles_are(hip, monkeypatch, n, m, d, form, step):
    print(f"two loops in turn: {form}, {n} x {m}, d {d}, {step} at a time", flush=True)
    monkeypatch.setenv("TRNOPT_HIP_LOOP", "1")
    X, Y = _clouds(hip, n, m, d)
    loops = [_loop(hip, X, Y, f) for f in FORMS[form]]
    known = sorted({e for eps, sched, stages in FORMS[form] for e in (eps, *sched, *stages)})
    for l in loops:
        l.init()
    for _ in range(8 // step):
        for l in loops:
            l.enqueue(step)
            _header_is_true(hip, X, n, m, d, known)


def _step_in_turn(hip, X, Y, forms, step):
    loops = [_loop(hip, X, Y, f) for f in forms]
    for l in loops:
        l.init()
    for _ in range(8 // step):
        for l in loops:
            l.enqueue(step)
    return loops


@pytest.mark.parametrize("step", [1, 2])
@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("n,m,d", [(300, 200, 20), (1300, 900, 64), (10_273, 300, 30)])
def test_each_loop_gets_the_potentials_it_has_alone(hip, monkeypatch, n, m, d, form, step):
    """Alone, the scores come from the copy in every iteration, here from the general path in some: float32 rounding of the
    scores apart (1e-5 relative, as in the solver tests). A loop whose copy comes back carries on from the potentials of
    the iterations without it."""
    print(f"two loops in turn: {form}, {n} x {m}, d {d}, {step} at a time", flush=True)
    monkeypatch.setenv("TRNOPT_HIP_LOOP", "1")
    for l, f in zip(_step_in_turn(hip, *_clouds(hip, n, m, d), FORMS[form], step), FORMS[form]):
        alone = _loop(hip, *_clouds(hip, n, m, d), f)
        alone.init()
        alone.enqueue(8)
        assert (l.read_state().it, l.read_state().eps) == (alone.read_state().it, alone.read_state().eps)
        for got, want, k in ((l.fh, alone.fh, n), (l.gh, alone.gh, m)):
            assert inf_rel(got[:k].cpu(), want[:k].cpu()) <= 1e-5

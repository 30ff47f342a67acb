"""A resident launch whose waits run out (TRNOPT_HIP_LOOP_POLLS: a few polls each) is made good on the device: whoever
enqueued the iterations finds them done, without having looked at the state, bit for bit as launches do them. A whole run,
which reads the state, goes on as launches from where that launch began, with the same results."""

import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)

FORMS = {
    "fixed": dict(eps=0.1, sched=[], stages=[], fixed_iters=True),
    "schedule": dict(eps=0.1, sched=[0.9, 0.6, 0.4, 0.3, 0.2], stages=[], fixed_iters=True),
    "stages": dict(eps=0.1, sched=[], stages=[0.8, 0.4, 0.2], fixed_iters=False),
    "checked": dict(eps=0.4, sched=[], stages=[], fixed_iters=False),
}


def _loop(hip, n, m, d, form):
    rng = np.random.default_rng(n * 31 + m * 7 + d)
    x, y = rng.normal(size=(n, d)) * 0.4, rng.normal(size=(m, d)) * 0.4 + 0.1
    a, b = rng.uniform(0.5, 1.5, n), rng.uniform(0.5, 1.5, m)
    X = hip.HipCloud(x, np.log(a / a.sum()), DEV, role=0)
    Y = hip.HipCloud(y, np.log(b / b.sum()), DEV, role=1)
    return hip.DeviceLoop(X, Y, rho_x=None, rho_y=None, tol=1e-3, stage_tol=0.05, max_iters=90, check_every=2,
                          stage_max_iters=8, balanced=True, **FORMS[form])


def _state(st):
    return [getattr(st, k) for k, _ in st._fields_ if k not in ("sc_x", "sc_y")] + list(st.sc_x) + list(st.sc_y)


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("n,m,d", [(400, 900, 30), (33, 31, 5), (1300, 1000, 64), (600, 700, 128)])
def test_enqueued_iterations_are_done(hip, monkeypatch, n, m, d, form):
    print(f"give-up {form} {n} x {m} d {d}", flush=True)
    got = []
    for loop_env, polls in (("0", None), ("1", "1")):
        monkeypatch.setenv("TRNOPT_HIP_LOOP", loop_env)
        if polls:
            monkeypatch.setenv("TRNOPT_HIP_LOOP_POLLS", polls)
        loop = _loop(hip, n, m, d, form)
        assert hip.lib().sk_loop_resident(ctypes.byref(loop._L)) == int(loop_env)
        loop.init()
        fh, gh, seen = loop.fh, loop.gh, []        # held from before the launches
        for k in (2, 1, 30, 7):
            loop.enqueue(k)
            seen += [fh.clone(), gh.clone()]
        got.append((seen, _state(loop.read_state()), loop.X.pk[:36].cpu()))
        assert (loop.repairs() > 0) == (polls is not None)
    for p, q in zip(got[0][0], got[1][0]):
        assert torch.equal(p, q)
    np.testing.assert_array_equal(got[0][1], got[1][1])
    assert torch.equal(got[0][2][:28], got[1][2][:28])


@pytest.mark.parametrize("polls", [2, 4, 6, 9, 14])
@pytest.mark.parametrize("form", list(FORMS))
def test_a_give_up_on_the_way_changes_nothing(hip, monkeypatch, form, polls):
    """With a few polls a wait runs out in some iteration or in none: enqueued calls and whole runs alike."""
    n, m, d = 700, 500, 30
    print(f"give-up on the way {form} {polls} polls", flush=True)
    monkeypatch.setenv("TRNOPT_HIP_LOOP", "0")
    want = _loop(hip, n, m, d, form)
    end = _state(want.run())
    monkeypatch.setenv("TRNOPT_HIP_LOOP", "1")
    monkeypatch.setenv("TRNOPT_HIP_LOOP_POLLS", str(polls))
    runs, calls = _loop(hip, n, m, d, form), _loop(hip, n, m, d, form)
    np.testing.assert_array_equal(_state(runs.run()), end)
    calls.init()
    for _ in range(9):
        calls.enqueue(10)
    np.testing.assert_array_equal(_state(calls.read_state()), end)
    for l in (runs, calls):
        assert torch.equal(l.fh, want.fh) and torch.equal(l.gh, want.gh)
    print("runs made good:", runs.repairs(), calls.repairs(), flush=True)


def test_no_launch_gives_up_by_itself(hip, monkeypatch):
    monkeypatch.setenv("TRNOPT_HIP_LOOP", "1")
    loop = _loop(hip, 1300, 1000, 64, "fixed")
    loop.init()
    loop.enqueue(40)
    assert (loop.read_state().it, loop.repairs()) == (40, 0)

"""The log2-unit copy of the first cloud when the on-device loop moves to a new eps: the control only marks it, and the
next f update makes its tiles, each workgroup its own rows. The tiles must be those that sk_bake_log2_f32 makes for that
eps on a fresh cloud, bit for bit, and while they are still to be made the header must offer no copy to anyone else."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _clouds(hip, n, m, d):
    rng = np.random.default_rng(n + m + d)
    x = rng.normal(size=(n, d)) * 0.3
    y = rng.normal(size=(m, d)) * 0.3 + 0.1
    return (hip.HipCloud(x, np.full(n, -np.log(n)), DEV, role=0), hip.HipCloud(y, np.full(m, -np.log(m)), DEV, role=1))


def _tag(cloud):
    w = cloud.pk[:64].cpu().numpy()
    f, i = w.view(np.float32), w.view(np.int32)
    return float(f[2]), float(f[4]), int(i[6])


def _copy_tiles(cloud, hip):
    head = hip.PACKED_HEADER_BYTES
    half = (cloud.pk.numel() - head) // 2
    return cloud.pk[head + half:].cpu()


@pytest.mark.parametrize("n,m,d", [(33, 40, 5), (1300, 900, 64), (255, 2100, 30), (10_273, 300, 100)])
@pytest.mark.parametrize("stages", [False, True])
def test_a_new_eps_remakes_the_copy(hip, n, m, d, stages):
    print(f"copy remade: {n} x {m}, d {d}, stages {stages}", flush=True)
    X, Y = _clouds(hip, n, m, d)
    eps = [0.8, 0.4, 0.1]
    loop = hip.DeviceLoop(X, Y, eps=eps[-1], rho_x=None, rho_y=None, sched=[] if stages else eps[:-1],
                          stages=eps[:-1] if stages else [], tol=0.0, stage_tol=1e9, max_iters=9, check_every=1,
                          stage_max_iters=1000, fixed_iters=True, balanced=True)
    loop.init()
    for k, e in enumerate(eps):
        # iteration k runs at eps[k]: its f update makes the copy (k > 0), its control hands on the next eps
        loop.enqueue(1)
        c, t, pending = _tag(X)
        last = k == len(eps) - 1
        assert pending == (0 if last else 1) and (c == 0.0) == (not last), (k, c, pending)
        A, B = _clouds(hip, n, m, d)
        hip.bake_log2(A, B, hip.scalars(e, 1.0, DEV))
        want = _tag(A)
        assert want[0] > 0.0
        if last:
            assert (c, t) == want[:2]
        assert torch.equal(_copy_tiles(X, hip), _copy_tiles(A, hip)), k
    loop.enqueue(3)
    assert torch.isfinite(loop.fh).all() and torch.isfinite(loop.gh).all()

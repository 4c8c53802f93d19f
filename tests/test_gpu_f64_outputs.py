"""What a float64 step is asked to leave besides the poses does not change them:
steps with fields and diagnostics, with either, and with neither move the agents
identically, and the increments in the diagnostics are the sums of their parts
within the float64 path's 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one, two, four and eight waves a replica; both orders
@pytest.mark.parametrize("N, R, replicas", [(50, 500, 4), (70, 512, 300), (100, 1024, 2), (30, 4000, 3)])
@pytest.mark.parametrize("order", ["sequential", "synchronous"])
def test_outputs_do_not_move_agents(gpu, N, R, replicas, order):
    from abm_amd.vf import VFConfig, VFSwarm
    rng = np.random.RandomState(N + R)
    side = 50.0 * np.sqrt(N)
    cfgs = [VFConfig(n_agents=N, n_rays=R, width=side, height=side, boundary=("infinite", "walls")[b % 2],
                     ALP0=0.5 + b % 3, BET0=0.5) for b in range(replicas)]
    n = N * replicas
    start = [30 + rng.uniform(0, side, n), 30 + rng.uniform(0, side, n), rng.uniform(0, 2 * np.pi, n), rng.uniform(0, 2, n)]
    kinds = [dict(), dict(fields=True), dict(diag=True), dict(fields=True, diag=True)]
    swarms = [VFSwarm(cfgs, *start, radius=5, precision="f64") for _ in kinds]
    gam, v0 = cfgs[0].GAM, cfgs[0].V0
    for step in range(3):
        v = swarms[0].state_numpy()[3]
        for sw, kw in zip(swarms, kinds):
            sw.step(order=order, **kw)
        want = swarms[0].state_numpy()
        for sw, kw in zip(swarms[1:], kinds[1:]):
            for p, q in zip(sw.state_numpy(), want):
                assert np.array_equal(p, q), (step, kw)
        d = swarms[2].diag_numpy()
        assert np.array_equal(d, swarms[3].diag_numpy()), step
        parts = np.stack([gam * (v0 - v) + d[:, 2] + d[:, 3], d[:, 4] + d[:, 5]], axis=1)
        assert np.max(np.abs(d[:, :2] - parts) / np.maximum(np.abs(parts), 1.0)) <= 1e-12, step

"""The push kernel sums agent k + 1's field ahead with the rays that agent k
would set if it kept its heading and speed, and again where it did not.  Fast,
sharply turning agents (guesses mostly wrong), slow ones (mostly right) and
agents that start on one place, at the smallest sizes of the chain: fields,
diagnostics, poses and speeds equal the one-wave per-replica kernel's bit for
bit, in the plain step and in the one with outputs."""
import numpy as np
import pytest

from test_gpu_push import swarm
from test_gpu_vf_f32 import uniform_start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rays", [64, 250, 1000, 2048])
@pytest.mark.parametrize("turn, speed, together", [(40.0, 25.0, False), (0.1, 0.2, False), (3.0, 2.0, True)])
def test_sums_taken_ahead(gpu, n_rays, turn, speed, together):
    import torch
    from abm_amd.vf import VFConfig
    cfgs, states = [], []
    for n in (1, 2, 3, 9, 65):
        for boundary in ("infinite", "walls"):
            side = 60.0 * np.sqrt(n) + 40.0
            cfgs.append(VFConfig(n_agents=n, n_rays=n_rays, width=side, height=side, boundary=boundary,
                                 ALP0=1.0, BET0=turn, V0=speed))
            s = uniform_start(n, side, side, 15, seed=7 * n + n_rays, v=speed)
            if together:
                s[0][:] = s[0][0]
                s[1][:] = s[1][0]
            states.append(s)
    a, b, c, d = (swarm(cfgs, states, launch) for launch in (32, 1, 32, 1))
    for step in range(4):
        print(f"  sums ahead R={n_rays} turn={turn} together={together} step {step}", flush=True)
        a.step(fields=True, diag=True)
        b.step(fields=True, diag=True)
        c.step()
        d.step()
        assert a.last_kernels() == c.last_kernels() == {"push"}
        assert b.last_kernels() == d.last_kernels() == {"per_replica"}
        torch.cuda.synchronize()
        assert torch.equal(a.fields, b.fields) and torch.equal(a.diag, b.diag), step
        for x, y in ((a, b), (c, d)):
            for p, q in zip(x.state_numpy(), y.state_numpy()):
                assert np.array_equal(p, q), step

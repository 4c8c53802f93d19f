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


@pytest.mark.parametrize("rays", [(64, 250), (300, 512), (1024, 700), (2048, 1100)])
@pytest.mark.parametrize("sizes", [(1, 9, 33, 64), (1, 9, 30), (200, 8, 9, 10, 64, 65, 33, 12, 2),
                                   (200, 8, 9, 10, 30, 65, 22, 12, 2)])
def test_whole_batches_on_the_push_kernel(gpu, sizes, rays):
    # the automatic launch gives a batch that the CUs hold at once to the push
    # kernel, small replicas too, with the moves of the kernels that each size
    # class has (small ones: per_replica, two waves above 32 agents, else one)
    import torch
    from abm_amd.vf import VFConfig
    cfgs, states = [], []
    for b, n in enumerate(sizes):
        side = 90.0 * np.sqrt(n) + 60.0
        cfgs.append(VFConfig(n_agents=n, n_rays=rays[0] if n > 64 else rays[1], width=side, height=side,
                             boundary=("infinite", "walls")[b % 2], ALP0=1.0, BET0=0.5))
        states.append(uniform_start(n, side, side, 20, seed=900 + b, v=0.7))
    pick = lambda big: [b for b, n in enumerate(sizes) if (n > 64) == big]
    a = swarm(cfgs, states, 0)
    parts = [(idx, swarm([cfgs[b] for b in idx], [states[b] for b in idx], launch))
             for idx, launch in ((pick(False), 2 if max(n for n in sizes if n <= 64) > 32 else 1), (pick(True), 32))
             if idx]
    for step in range(3):
        kw = dict(diag=True) if step == 1 else {}
        a.step(**kw)
        assert a.last_kernels() == {"push"}
        for idx, p in parts:
            p.step(**kw)
            for at, b in enumerate(idx):
                for x, y in zip(a.state_numpy(), p.state_numpy()):
                    assert np.array_equal(x[a.replica_slice(b)], y[p.replica_slice(at)]), (step, sizes[b])


@pytest.mark.parametrize("sizes, rays", [((200, 8, 9, 10), (250, 250)),                       # a few of both
                                         ((200, 8, 9, 10, 64, 65, 33, 12, 2), (1024, 250)),   # shorter sums
                                         ((200, 8, 9, 10, 64, 65, 33, 12, 2), (250, 1024))])
def test_batches_that_keep_a_kernel_for_each_class(gpu, sizes, rays):
    from abm_amd.vf import VFConfig
    cfgs = [VFConfig(n_agents=n, n_rays=rays[0] if n > 64 else rays[1], width=900.0, height=900.0, boundary="walls")
            for n in sizes]
    a = swarm(cfgs, [uniform_start(n, 900.0, 900.0, 20, seed=n, v=0.7) for n in sizes], 0)
    a.step()
    assert a.last_kernels() == {"per_replica", "push"}

"""The chain step's segments in the order in which agents come free: a flock
spread wider than an agent sees, with dependences in a segment few, many or
none, a segment of one agent, agents that jump beyond the margin (the segment
is then taken again in id order) and a torus too small for it.  Fields,
diagnostics, poses and speeds equal the push kernel's bit for bit, in the step
with outputs and in the plain one."""
import numpy as np
import pytest

from test_gpu_push import swarm
from test_gpu_vf_f32 import uniform_start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, side, n_rays, boundary, v, alp0", [
    (257, 20000.0, 250, "infinite", 0.5, 1.0),     # nobody sees anybody
    (600, 3000.0, 512, "infinite", 0.5, 1.0),      # a few in sight
    (600, 3000.0, 512, "walls", 2.0, 1.0),
    (400, 6000.0, 2048, "infinite", 1.0, 1.0),     # a third in sight: either order
    (500, 4000.0, 1024, "infinite", 0.5, 200.0),   # jumps beyond the margin
    (300, 420.0, 1024, "infinite", 0.5, 1.0),      # everybody sees everybody
])
def test_segments_in_any_order(gpu, n, side, n_rays, boundary, v, alp0):
    import torch
    from abm_amd.vf import VFConfig
    cfg = VFConfig(n_agents=n, n_rays=n_rays, width=side, height=side, boundary=boundary, ALP0=alp0, BET0=0.5)
    st = uniform_start(n, side, side, 30, seed=n + n_rays, v=v)
    st[0][n // 2:n // 2 + 2] = st[0][:2]           # two on others' places
    st[1][n // 2:n // 2 + 2] = st[1][:2]
    a, b, c, d = (swarm([cfg], [st], launch) for launch in (64, 32, 64, 32))
    for step in range(3):
        print(f"  chain flow n={n} side={side} R={n_rays} {boundary} step {step}", flush=True)
        a.step(fields=True, diag=True)
        b.step(fields=True, diag=True)
        c.step()
        d.step()
        assert a.last_kernels() == c.last_kernels() == {"chain"}
        assert b.last_kernels() == d.last_kernels() == {"push"}
        torch.cuda.synchronize()
        assert torch.equal(a.fields, b.fields) and torch.equal(a.diag, b.diag), step
        for x, y in ((a, b), (c, d)):
            for p, q in zip(x.state_numpy(), y.state_numpy()):
                assert np.array_equal(p, q), step

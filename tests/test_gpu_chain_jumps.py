"""The chain step where agents jump beyond the margin of the dependences: a
segment with a jump is taken again in id order at once, and a step in which that
is the rule stops trying.  All agents, some in every segment, a few, one and none
jump, over nine segments, the last of four agents: poses, fields and diagnostics
equal those of steps that count (which go in id order) bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jumpers", ["all", "a fiftieth", "a few", "the last", "none", "all but the last segments'"])
@pytest.mark.parametrize("boundary, side, R", [("infinite", 6000.0, 512), ("walls", 4500.0, 2048)])
def test_jumps_over_segments(gpu, jumpers, boundary, side, R):
    from abm_amd.vf import VFConfig, VFSwarm
    n = 8 * 256 + 4
    rng = np.random.RandomState(R)
    far = {"all": np.ones(n, bool), "a fiftieth": rng.rand(n) < 0.02, "a few": np.isin(np.arange(n), [3, 300, 301, 1500]),
           "the last": np.arange(n) == n - 1, "none": np.zeros(n, bool),
           "all but the last segments'": np.arange(n) < 4 * 256}[jumpers]
    cfg = VFConfig(n_agents=n, n_rays=R, width=side, height=side, boundary=boundary, BET0=0.5)
    st = [30 + rng.uniform(0, side, n), 30 + rng.uniform(0, side, n), rng.uniform(0, 2 * np.pi, n)]
    a, b = (VFSwarm([cfg], *st, 0.5, radius=5, precision="f32", alp0=np.where(far, 3000.0, 1.0)) for _ in range(2))
    plain = VFSwarm([cfg], *st, 0.5, radius=5, precision="f32", alp0=np.where(far, 3000.0, 1.0))
    for sw in (a, b, plain):
        sw.set_launch(64)
    for step in range(3):
        a.step(fields=True, diag=True)
        b.step(fields=True, diag=True, count=True)
        plain.step()
        assert a.last_kernels() == b.last_kernels() == plain.last_kernels() == {"chain"}
        assert np.array_equal(a.fields.cpu().numpy(), b.fields.cpu().numpy()), step
        assert np.array_equal(a.diag_numpy(), b.diag_numpy()), step
        for p, q in zip(a.state_numpy(), b.state_numpy()):
            assert np.array_equal(p, q), step
        want = VFSwarm([cfg], *st, 0.5, radius=5, precision="f32", alp0=np.where(far, 3000.0, 1.0))
        want.set_launch(64)
        for _ in range(step + 1):
            want.step(count=True)
        for p, q in zip(plain.state_numpy(), want.state_numpy()):
            assert np.array_equal(p, q), step

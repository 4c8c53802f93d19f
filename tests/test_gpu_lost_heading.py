"""Focal agents whose heading the reference loses: it takes the heading from two
positions a radius apart, so a radius of 0 gives none (every object falls into
bin 0), a negative one the opposite and a position far beyond the radius a
rounded one.  The float32 decisions of the float64 flocking step and of the
cooperative-signalling projections must leave these to float64: fields and
projections identical to the plain float64 kernel's and to the oracle's."""
import numpy as np
import pytest

from oracle import cs_oracle as co

pytestmark = pytest.mark.gpu
PI = np.pi


@pytest.mark.parametrize("radii, offset", [((0, 3, 8), 0.0), ((-4, 3, 8), 0.0), ((1, 2), 1e13)])
@pytest.mark.parametrize("N, R", [(40, 512), (70, 1000)])
def test_float64_step(gpu, radii, offset, N, R):
    from abm_amd.vf import VFConfig, VFSwarm
    rng = np.random.RandomState(N + R + len(radii))
    side = 300.0
    x, y = (30.0 + offset + rng.uniform(0, side, N) for _ in range(2))
    th, v = rng.uniform(0, 2 * PI, N), rng.uniform(0, 2, N)
    cfg = VFConfig(n_agents=N, n_rays=R, width=side + 10 * offset, height=side + 10 * offset, boundary="infinite")
    rad = rng.choice(radii, N)
    a, b = (VFSwarm([cfg], x, y, th, v, radius=rad, precision="f64") for _ in range(2))
    for step in range(2):
        a.step(fields=True)
        b.step(fields=True, count=True)   # the plain kernel
        assert np.array_equal(a.fields.cpu().numpy(), b.fields.cpu().numpy()), step
        for name in ("x", "y", "theta", "v"):   # the next step from identical poses
            p, q = getattr(a, name).cpu().numpy(), getattr(b, name).cpu().numpy()
            assert np.max(np.abs(p - q) / np.maximum(np.abs(q), 1.0)) <= 1e-12, (step, name)
            getattr(a, name).copy_(getattr(b, name))


@pytest.mark.parametrize("radius, spread", [(0.0, 80.0), (1e-12, 1e-10)])
def test_signalling_projections(gpu, radius, spread):
    import torch
    from abm_amd.cs import CSProjection
    rng = np.random.RandomState(11)
    R, n, fov = 1200, 40, (-0.8 * PI, 0.8 * PI)
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")
    focal = np.array([(100.0, 90.0, radius, rng.uniform(0, 2 * PI)) for _ in range(20)])
    objs = [focal[k, :2] + rng.uniform(-spread, spread, (n, 2)) for k in range(len(focal))]
    off = np.arange(0, n * len(focal) + 1, n).astype(np.int64)
    mets = rng.uniform(0, 1, n * len(focal))
    args = (T(focal), T(off), T(np.concatenate(objs)))
    proj = CSProjection(R, fov, None)
    rows = proj.rows(*args, T(mets)).cpu().numpy()
    peak = proj.max(*args, T(mets)).cpu().numpy()
    count = proj.sum(*args, T(np.full(len(focal), 7.0))).cpu().numpy()
    for k, (x, y, r, th) in enumerate(focal):
        with np.errstate(all="ignore"):
            want = co.projection_field(fov, R, np.array([x, y]), r, th, list(objs[k]), list(mets[off[k]:off[k + 1]]), None)
            ones = co.projection_field(fov, R, np.array([x, y]), r, th, list(objs[k]), [1.0] * n, None)
        assert np.array_equal(rows[off[k]:off[k + 1]], want), (k, "rows")
        assert np.array_equal(peak[k], want.max(axis=0)), (k, "max")
        assert np.array_equal(count[k], ones.sum(axis=0) / 7.0), (k, "sum")

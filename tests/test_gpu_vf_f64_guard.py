"""The float64 step with guarded float32 decisions against the plain float64
kernel (which a step that counts near ties takes): fields and every decision
identical; poses and diagnostics, whose sums run in another order, within the
float64 path's 1e-12 relative bar."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
PI = np.pi


def _pair(cfgs, x, y, th, v, radius):
    from abm_amd.vf import VFSwarm
    return [VFSwarm(cfgs, x, y, th, v, radius=radius, precision="f64") for _ in range(2)]


def _check(a, b, order, steps):
    for step in range(steps):
        a.step(order=order, fields=True, diag=True)
        b.step(order=order, fields=True, diag=True, count=True)
        assert np.array_equal(a.fields.cpu().numpy(), b.fields.cpu().numpy()), step
        for p, q in zip(a.state_numpy() + (a.diag_numpy(),), b.state_numpy() + (b.diag_numpy(),)):
            assert np.max(np.abs(p - q) / np.maximum(np.abs(q), 1.0)) <= 1e-12, step
        for name in ("x", "y", "theta", "v"):   # the next step from identical poses
            getattr(a, name).copy_(getattr(b, name))


# rays: a part of one lane's span, one and several waves' spans full, one ray
# more and less, the largest the guarded kernel takes and one beyond it (plain);
# agents: one, a wavefront less one, full, one more
@pytest.mark.parametrize("N, R", [(1, 33), (2, 255), (63, 256), (64, 257), (65, 512), (20, 513), (130, 1025),
                                  (33, 2049), (9, 4096), (9, 4097)])
@pytest.mark.parametrize("boundary, fov, order", [("infinite", 1.0, "sequential"), ("walls", 0.6, "sequential"),
                                                  ("infinite", 1.0, "synchronous")])
def test_guarded_equals_plain(gpu, N, R, boundary, fov, order):
    from abm_amd.vf import VFConfig
    rng = np.random.RandomState(N * 10000 + R)
    cfgs, x, y, th, v, rad = [], [], [], [], [], []
    for b in range(3):   # three replicas of several sizes, mixed radii, movement limits in one
        n, side = max(1, N - 5 * b), 40.0 * np.sqrt(N) + 60.0
        cfgs.append(VFConfig(n_agents=n, n_rays=R, width=side, height=side * 1.3, boundary=boundary,
                             fov=VFConfig.fov_from_ratio(fov), ALP0=0.5 + b, BET0=0.3 + b, LIMIT_MOVEMENT=b == 1))
        x.append(rng.uniform(30, 30 + side, n))
        y.append(rng.uniform(30, 30 + 1.3 * side, n))
        th.append(rng.uniform(0, 2 * PI, n))
        v.append(rng.uniform(0, 2, n))
        rad.append(rng.choice([2, 5, 9], n))
    cat = np.concatenate
    a, b = _pair(cfgs, cat(x), cat(y), cat(th), cat(v), cat(rad))
    _check(a, b, order, 2)


@pytest.mark.parametrize("R", [8, 64, 100, 512, 1000])
def test_guarded_equals_plain_on_a_lattice(gpu, R):
    # integer positions and headings in eighths of a turn: pairs on bin ties,
    # dead ahead and behind, exactly half an arena apart, overlapping, touching
    # and coincident, where only the float64 replica may decide
    from abm_amd.vf import VFConfig
    rng = np.random.RandomState(R)
    cfgs, x, y, th = [], [], [], []
    for b in range(40):
        n = 48
        cfgs.append(VFConfig(n_agents=n, n_rays=R, width=64, height=64, boundary=("infinite", "walls")[b % 2]))
        x.append(30.0 + 4.0 * rng.randint(0, 16, n))
        y.append(30.0 + 4.0 * rng.randint(0, 16, n))
        th.append(PI / 4 * rng.randint(0, 8, n))
    cat = np.concatenate
    a, b = _pair(cfgs, cat(x), cat(y), cat(th), np.zeros(40 * 48), 4)
    _check(a, b, "synchronous", 1)

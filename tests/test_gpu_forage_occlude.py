"""GPU parity of the foraging update with visual exclusion
(forage_occlude_kernel: each field prepared ahead of its agent's turn, the
agent before it added last) against the oracle's id-order update.

Bar: as test_gpu_forage.compare (fields, modes and generator positions
identical, continuous state within 1e-12 relative)."""
import numpy as np
import pytest

from oracle import forage_oracle as fo
from test_gpu_forage import compare, make_world
from test_gpu_forage_update import _swarm

pytestmark = pytest.mark.gpu


def _steps(ags, kw, R, steps, rng_seed=5):
    rng, orng = np.random.RandomState(rng_seed), np.random.RandomState(rng_seed)
    sw = _swarm([(ags, R, kw)], [rng])
    for step in range(steps):
        used = sw.step(fields=True)
        np.random.set_state(orng.get_state())
        fo.group_update(ags)
        orng.set_state(np.random.get_state())
        assert orng.get_state()[2] == rng.get_state()[2], (step, used)
        compare(sw, 0, ags)


# as many agents as one preparing wave and as all seven of them, one more and
# one less; one, two and four records per lane; words fewer and more than
# lanes; few and many in range
@pytest.mark.parametrize("N, R, fov, vision", [
    (1, 33, 1.0, 2000.0), (2, 64, 1.0, 2000.0), (6, 100, 1.0, 2000.0), (7, 600, 0.6, 2000.0),
    (8, 2081, 1.0, 2000.0), (15, 40000, 1.0, 2000.0), (63, 600, 1.0, 150.0), (64, 1000, 0.7, 2000.0),
    (65, 300, 1.0, 200.0), (129, 500, 1.0, 120.0), (257, 200, 1.0, 60.0)])
def test_occluded_update_matches_oracle(gpu, N, R, fov, vision):
    W = int(45 * np.sqrt(N)) + 80
    ags, kw = make_world(6000 + N, N=N, R=R, W=W, vis_ex=True, vision=vision)
    kw["fov"] = (-fov * np.pi, fov * np.pi)
    for a in ags:
        a.FOV = kw["fov"]
    print(f"occluded N={N} R={R}", flush=True)
    _steps(ags, kw, R, 2 if N <= 65 else 1)


@pytest.mark.parametrize("pitch", [20.0, 31.0])
def test_equal_distances_and_shared_places(gpu, pitch):
    # a lattice: many records at one distance, which the obstacle list's order
    # ranks, overlapping end to end; some agents on one place
    ags, kw = make_world(6500, N=40, R=720, W=300, vis_ex=True)
    for i, a in enumerate(ags):
        a.position = np.array([60.0 + pitch * (i % 6), 60.0 + pitch * (i // 6)], dtype=np.float64)
        if i % 9 == 4:
            a.position = ags[i - 1].position.copy()
        if i % 3 == 0:
            a.set_mode("exploit")
            a.exploited_patch_id = i % 4
    _steps(ags, kw, 720, 3)

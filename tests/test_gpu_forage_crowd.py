"""The foraging update with visual exclusion for more agents than the occlusion
kernel holds in registers, with dozens to hundreds in range of each (their ranks
and the walk over the nearer ones), against the oracle: the smallest such
replica, ties of distance on a lattice, and more agents than threads."""
import numpy as np
import pytest

from test_gpu_forage import make_world
from test_gpu_forage_occlude import _steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N, R, vision, lattice", [
    (257, 600, 200.0, False), (261, 333, 120.0, True), (520, 500, 80.0, False)])
def test_crowded_occlusion_matches_oracle(gpu, N, R, vision, lattice):
    W = int(45 * np.sqrt(N)) + 80
    ags, kw = make_world(6800 + N, N=N, R=R, W=W, vis_ex=True, vision=vision)
    if lattice:
        for i, a in enumerate(ags):
            a.position = np.array([60.0 + 31.0 * (i % 17), 60.0 + 31.0 * (i // 17)], dtype=np.float64)
            if i % 3 == 0:
                a.set_mode("exploit")
                a.exploited_patch_id = i % 4
    print(f"crowd N={N} R={R}", flush=True)
    _steps(ags, kw, R, 1)

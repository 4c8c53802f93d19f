"""GPU parity of the resource loop at the line between one workgroup per
replica (a thread per agent, up to 1024) and launches over the replica's agents
(above it), against the oracle's ForageWorld.  Bar: as test_gpu_world.compare."""
import numpy as np
import pytest

from oracle import forage_oracle as fo
from test_gpu_world import compare, forage_config, load_agents, make_agents, same_stream

pytestmark = pytest.mark.gpu

APART = [(1, (150, 150)), (2, (700, 300)), (3, (300, 800))]
OVERLAP = [(1, (150, 150)), (2, (190, 150)), (3, (300, 800))]   # 1 and 2 share agents: the serial walk


# a full workgroup; one agent more, patches apart and overlapping: a patch
# with more exploiting agents than units (destroyed), several 64-agent words of
# them, and agents of many words on one patch
@pytest.mark.parametrize("N, layout, teleport, device_rng", [
    (1024, APART, True, False), (1025, APART, True, True), (1025, OVERLAP, False, False)])
def test_world_around_a_full_workgroup(gpu, N, layout, teleport, device_rng):
    from abm_amd.forage import ForageSwarm, ResourceWorld, WorldConfig
    W, R = 1000, 64
    ags, p = make_agents(2500 + N, N, W, R, True, 0)
    r0 = np.random.RandomState(9)
    for i, a in enumerate(ags):   # every third agent near a patch, in id order across all words
        if i % 3 == 0:
            cx, cy = layout[(i // 3) % 3][1]
            a.position = np.array([r0.randint(cx + 5, cx + 55), r0.randint(cy + 5, cy + 55)], dtype=np.float64)
    world = fo.ForageWorld(ags, W, W, 30, 0, 40, 3, 9, 0.5, 1.0, teleport_exploit=teleport)
    # the second patch outlasts its exploiting agents, the others do not
    world.patches = [fo.Patch(i, 40, pos, 400 if i == 2 else 20, 0.75) for i, pos in layout]
    rngs, orng = [np.random.RandomState(77)], np.random.RandomState(77)
    sw = ForageSwarm([forage_config(N, W, R, p)], [a.position[0] for a in ags], [a.position[1] for a in ags],
                     [a.orientation for a in ags], radius=10, rngs=rngs)
    rw = ResourceWorld(sw, [WorldConfig(N_resc=3, patch_radius=40, min_resc_perpatch=3, max_resc_perpatch=9,
                                        min_resc_quality=0.5, max_resc_quality=1.0,
                                        teleport_exploit=teleport)], device_rng=device_rng)
    load_agents(sw, rw, ags, 0)
    pt = world.patches
    rw.set_patches(0, [q.id for q in pt], [q.position[0] for q in pt], [q.position[1] for q in pt],
                   [q.radius for q in pt], [q.resc_units for q in pt], [q.resc_left for q in pt],
                   [q.unit_per_timestep for q in pt])
    start = [q.position[0] for q in pt]
    for step in range(2):
        print(f"  N={N} step {step}", flush=True)
        rw.step()
        rw.sync_rng()
        np.random.set_state(orng.get_state())
        world.step()
        orng.set_state(np.random.get_state())
        assert same_stream(rngs[0], orng), step
        compare(sw, rw, world, 0, step)
        load_agents(sw, rw, world.agents, 0)
    assert [q.position[0] for q in world.patches] != start   # some patch was destroyed

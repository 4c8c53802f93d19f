"""GPU parity of the foraging update without visual exclusion
(forage_update_kernel: every field of a replica at once) at the edges of its
wavefronts, words and blocks, against the oracle's id-order update.

Bar: as test_gpu_forage.compare (fields, modes and generator positions
identical, continuous state within 1e-12 relative)."""
import numpy as np
import pytest

from oracle import forage_oracle as fo
from test_gpu_forage import compare, load_swarm, make_world

pytestmark = pytest.mark.gpu


def _swarm(worlds, rngs):
    from abm_amd.forage import ForageConfig, ForageSwarm
    ags = [a for w, _, _ in worlds for a in w]
    sw = ForageSwarm([ForageConfig(n_agents=len(w), n_rays=R, **kw) for w, R, kw in worlds],
                     [a.position[0] for a in ags], [a.position[1] for a in ags],
                     [a.orientation for a in ags], radius=10, rngs=rngs)
    for b, (w, _, _) in enumerate(worlds):
        load_swarm(sw, w, sw.replica_slice(b))
    return sw


# one agent, a wavefront less one, full and one more, several wavefronts of
# cues; fields of less than a word, whole words, a ragged last word, more
# words than lanes, and counts beyond 15 bits
@pytest.mark.parametrize("N, R, fov, vision", [
    (1, 31, 1.0, 2000.0), (2, 32, 1.0, 2000.0), (63, 1001, 0.5, 2000.0), (64, 2048, 1.0, 250.0),
    (65, 2081, 0.7, 2000.0), (257, 96, 1.0, 400.0), (5, 40000, 1.0, 2000.0)])
def test_update_matches_oracle_at_size_edges(gpu, N, R, fov, vision):
    W = int(60 * np.sqrt(N)) + 200
    ags, kw = make_world(7000 + N, N=N, R=R, W=W, vision=vision)
    kw["fov"] = (-fov * np.pi, fov * np.pi)
    for a in ags:
        a.FOV = kw["fov"]
    rng, orng = np.random.RandomState(5), np.random.RandomState(5)
    print(f"forage N={N} R={R}", flush=True)
    sw = _swarm([(ags, R, kw)], [rng])
    for step in range(2):
        used = sw.step(fields=True)
        np.random.set_state(orng.get_state())
        fo.group_update(ags)
        orng.set_state(np.random.get_state())
        assert orng.get_state()[2] == rng.get_state()[2], (step, used)
        compare(sw, 0, ags)


def test_many_small_replicas_equal_few(gpu):
    # a batch of many replicas takes smaller workgroups: the same bits
    worlds = []
    for b in range(530):
        n, R = 1 + b % 9, (64, 100, 300)[b % 3]
        ags, kw = make_world(8000 + b, N=n, R=R, W=300)
        worlds.append((ags, R, kw))
    many = _swarm(worlds, [np.random.RandomState(b) for b in range(530)])
    few = _swarm(worlds[-40:], [np.random.RandomState(b) for b in range(490, 530)])
    for step in range(3):
        many.step(fields=True)
        few.step(fields=True)
        gm, gf = many.get_state(), few.get_state()
        n = len(gf["x"])
        for k in ("x", "y", "theta", "v", "w", "u", "I_priv", "collected_r_before", "mode", "overriding_mode"):
            assert np.array_equal(gm[k][-n:], gf[k]), (step, k)
        fm, ff = many.fields.cpu().numpy(), few.fields.cpu().numpy()
        assert np.array_equal(fm[-len(ff):], ff), step


# a chunk of 64 agents less one, full and one more, several chunks, several
# replicas in the three launches; host words and device generators
@pytest.mark.parametrize("device_rng", [False, True])
def test_update_over_the_whole_gpu_equals_a_workgroup_each(gpu, device_rng):
    from abm_amd.forage import ResourceWorld, WorldConfig
    worlds = []
    for b, (n, R) in enumerate([(63, 100), (64, 64), (65, 1024), (1, 33), (200, 2081), (130, 512)]):
        ags, kw = make_world(9000 + b, N=n, R=R, W=500, mixed=False)
        worlds.append((ags, R, kw))
    pair = []
    for path in ("auto", "sweep"):
        rngs = [np.random.RandomState(50 + b) for b in range(len(worlds))]
        sw = _swarm(worlds, rngs)
        if path == "auto":   # enough other replicas that the batch takes a workgroup each
            extra = [make_world(9100 + b, N=80, R=96, W=400, mixed=False) for b in range(400)]
            rngs += [np.random.RandomState(1000 + b) for b in range(400)]
            sw = _swarm(worlds + [(a, 96, kw) for a, kw in extra], rngs)
        else:
            sw.set_path(path)
        rw = ResourceWorld(sw, [WorldConfig(N_resc=4, min_resc_perpatch=3, max_resc_perpatch=9)] * len(rngs),
                           device_rng=device_rng)
        rw.create_resources()
        pair.append((sw, rw, rngs))
    (a, ra, ga), (s, rs, gs) = pair
    n = len(s.get_state("x")["x"])
    for step in range(40):
        ra.step(fields=True)
        rs.step(fields=True)
        fa, fs = a.get_state(), s.get_state()
        for k in ("x", "y", "theta", "v", "w", "u", "I_priv", "collected_r_before", "mode", "overriding_mode"):
            assert np.array_equal(fa[k][:n], fs[k]), (step, k)
        bits = s.fields.cpu().numpy()
        assert np.array_equal(a.fields.cpu().numpy()[:len(bits)], bits), step
    ra.sync_rng()
    rs.sync_rng()
    for b in range(len(worlds)):
        assert ga[b].get_state()[2] == gs[b].get_state()[2], b
        assert np.array_equal(ga[b].get_state()[1], gs[b].get_state()[1]), b
    assert s.sweep_counts()[0] == 40 * len(worlds) and a.sweep_counts()[0] == 0

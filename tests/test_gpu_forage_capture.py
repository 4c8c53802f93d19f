"""Captured foraging steps: replays equal an eager twin bit for bit, whatever the
batch is asked for between capture and replay."""
import numpy as np
import pytest

from test_gpu_forage import make_world
from test_gpu_forage_update import _swarm

pytestmark = pytest.mark.gpu
KEYS = ("x", "y", "theta", "v", "w", "u", "I_priv", "collected_r", "collected_r_before", "mode", "overriding_mode")


def _world(sizes, seed):
    from abm_amd.forage import ResourceWorld, WorldConfig
    worlds = []
    for b, (n, R, vis_ex) in enumerate(sizes):
        ags, kw = make_world(seed + b, N=n, R=R, W=int(40 * np.sqrt(n)) + 300, vis_ex=vis_ex, mixed=False)
        worlds.append((ags, R, kw))
    sw = _swarm(worlds, [np.random.RandomState(seed + b) for b in range(len(worlds))])
    rw = ResourceWorld(sw, [WorldConfig(N_resc=4, min_resc_perpatch=3, max_resc_perpatch=9)] * len(worlds),
                       device_rng=True)
    rw.create_resources()
    for _ in range(5):
        rw.step(fields=True)
    return rw


def _same(a, b, where):
    sa, sb = a.swarm.get_state(), b.swarm.get_state()
    for k in KEYS:
        assert np.array_equal(sa[k], sb[k]), (where, k)
    assert np.array_equal(a.swarm.fields.cpu().numpy(), b.swarm.fields.cpu().numpy()), where
    a.sync_rng()
    b.sync_rng()
    for p, q in zip(a.swarm.rngs, b.swarm.rngs):
        assert np.array_equal(p.get_state()[1], q.get_state()[1]) and p.get_state()[2] == q.get_state()[2], where


@pytest.mark.parametrize("sizes", [
    [(30, 256, False), (12, 300, True), (50, 512, False), (20, 100, True)],   # a workgroup each
    [(300, 512, False), (12, 300, True), (70, 100, False)],                   # over the whole GPU
    [(1500, 1200, False), (40, 256, True)],                                   # beyond one workgroup's LDS
])
def test_replays_after_a_new_path(gpu, sizes):
    import torch
    g, e = _world(sizes, 400), _world(sizes, 400)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g.step(fields=True)
    junk = torch.randn(1 << 18, device="cuda")
    for rep, path in enumerate(("auto", "sweep", "auto", "sweep")):
        print(f"  capture {sizes} replay {rep} after {path}", flush=True)
        g.swarm.set_path(path)
        graph.replay()
        e.step(fields=True)
        junk = torch.sort(junk)[0]
        torch.cuda.synchronize()
        _same(g, e, rep)
        g.step(fields=True)   # and an eager step of the path chosen
        e.step(fields=True)
        _same(g, e, (rep, "eager"))

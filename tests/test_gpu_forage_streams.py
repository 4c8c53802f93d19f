"""Steps of several states through one foraging batch, on streams and threads of
their own, on paths whose launches share the batch's scratch: each state equals
its twin that stepped alone, bit for bit."""
import copy
import threading

import numpy as np
import pytest

from test_gpu_forage import make_world
from test_gpu_forage_capture import _same
from test_gpu_forage_update import _swarm

pytestmark = pytest.mark.gpu

# over the whole GPU because that is faster, and because one workgroup's LDS does not hold them
SIZES = [[(300, 512)], [(200, 256), (65, 100), (130, 1024)], [(2500, 600)]]


def _world(sizes, seed, batch_of=None):
    """A world of its own state; batch_of: on that world's batch."""
    from abm_amd.forage import ResourceWorld, WorldConfig
    worlds = []
    for b, (n, R) in enumerate(sizes):
        ags, kw = make_world(seed + b, N=n, R=R, W=int(40 * np.sqrt(n)) + 300)
        worlds.append((ags, R, kw))
    sw = _swarm(worlds, [np.random.RandomState(seed + b) for b in range(len(worlds))])
    if batch_of is not None:
        other = copy.copy(sw)   # the state above, the handle of the other's batch
        other.handle = batch_of.swarm.handle
        other.keep = sw
        sw = other
    cfg = [WorldConfig(N_resc=6, min_resc_perpatch=3, max_resc_perpatch=9)] * len(worlds)
    rw = ResourceWorld(sw, cfg, device_rng=True)
    rw.create_resources()
    for _ in range(3):
        rw.step(fields=True)
    return rw


@pytest.fixture(autouse=True)
def keep_handles(monkeypatch):
    # a copied swarm does not destroy the batch it borrows
    from abm_amd.forage import ForageSwarm
    free = ForageSwarm.__del__
    monkeypatch.setattr(ForageSwarm, "__del__", lambda self: None if hasattr(self, "keep") else free(self))


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("threads", [False, True])
def test_streams_equal_alone(gpu, sizes, threads):
    import torch
    shared = [_world(sizes, 600)]
    shared += [_world(sizes, 600 + 50 * i, shared[0]) for i in range(1, 3)]
    alone = [_world(sizes, 600 + 50 * i) for i in range(3)]
    torch.cuda.synchronize()
    streams = [None, torch.cuda.Stream(), torch.cuda.Stream()]   # None: the null stream
    steps = 40
    print(f"  streams {sizes} threads {threads}", flush=True)

    def go(i):
        for _ in range(steps):
            shared[i].step(fields=True, stream=streams[i])
    if threads:
        ts = [threading.Thread(target=go, args=(i,)) for i in range(3)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    else:
        for _ in range(steps):
            for i in range(3):
                shared[i].step(fields=True, stream=streams[i])
    torch.cuda.synchronize()
    for i in range(3):
        for _ in range(steps):
            alone[i].step(fields=True)
        _same(shared[i], alone[i], i)


@pytest.mark.parametrize("sizes", SIZES)
def test_graphs_beside_eager_steps(gpu, sizes):
    import torch
    shared = [_world(sizes, 800)]
    shared += [_world(sizes, 800 + 50 * i, shared[0]) for i in range(1, 3)]
    alone = [_world(sizes, 800 + 50 * i) for i in range(3)]
    torch.cuda.synchronize()
    graphs = []
    for i in (0, 1):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for _ in range(2):
                shared[i].step(fields=True)
        graphs.append(g)
    streams = [torch.cuda.Stream(), torch.cuda.Stream(), None]
    print(f"  graphs {sizes}", flush=True)
    for rep in range(10):
        for i in (0, 1):
            with torch.cuda.stream(streams[i]):
                graphs[i].replay()
        for _ in range(2):
            shared[2].step(fields=True, stream=streams[2])
        if rep % 3 == 2:
            torch.cuda.synchronize()
    torch.cuda.synchronize()
    for i in range(3):
        for _ in range(20):
            alone[i].step(fields=True)
        _same(shared[i], alone[i], i)

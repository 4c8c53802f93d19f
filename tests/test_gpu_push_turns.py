"""The push kernel's two loops (the next agent's field summed ahead, or each
agent's in its turn) on both sides of every size at which the launch changes
from one to the other: ray classes, up to 128 rays, agents, outputs, counters,
and small replicas that sum in two halves.  Steps equal the one-wave
per-replica kernel's (two-wave, for the halves) bit for bit."""
import numpy as np
import pytest

from test_gpu_push import swarm
from test_gpu_vf_f32 import uniform_start

pytestmark = pytest.mark.gpu


def group(sizes, n_rays, boundary, launch):
    from abm_amd.vf import VFConfig
    cfgs, states = [], []
    for n in sizes:
        side = 70.0 * np.sqrt(n) + 60.0
        cfgs.append(VFConfig(n_agents=n, n_rays=n_rays, width=side, height=side, boundary=boundary,
                             ALP0=1.0, BET0=0.5))
        states.append(uniform_start(n, side, side, 20, seed=n + n_rays, v=0.7))
    return swarm(cfgs, states, launch)


@pytest.mark.parametrize("n, n_rays, boundary", [
    (64, 128, "infinite"), (65, 128, "walls"), (65, 129, "infinite"), (512, 256, "walls"), (513, 256, "infinite"),
    (384, 257, "infinite"), (385, 512, "walls"), (512, 1024, "infinite"), (513, 700, "walls"),
    (64, 2000, "walls"), (65, 1025, "infinite"), (2, 40, "infinite"), (1, 300, "walls")])
def test_both_loops(gpu, n, n_rays, boundary):
    for kw in ({}, dict(fields=True), dict(diag=True), dict(fields=True, diag=True, count=True, verify=True)):
        print(f"  push n={n} R={n_rays} {kw}", flush=True)
        a, b = (group((n,), n_rays, boundary, launch) for launch in (32, 1))
        for step in range(2):
            for sw in (a, b):
                sw.step(**kw)
            assert a.last_kernels() == {"push"} and b.last_kernels() == {"per_replica"}
            for p, q in zip(a.state_numpy(), b.state_numpy()):
                assert np.array_equal(p, q), (kw, step)
            if "fields" in kw:
                assert np.array_equal(a.fields.cpu().numpy(), b.fields.cpu().numpy()), (kw, step)
            if "diag" in kw:
                assert np.array_equal(a.diag_numpy(), b.diag_numpy()), (kw, step)
        if "count" in kw:
            pairs, _, disagree = a.fallback_counts()
            assert pairs == 2 * n * (n - 1) and disagree == 0


@pytest.mark.parametrize("outputs", [False, True])
@pytest.mark.parametrize("n_rays", [512, 1024, 2048])
@pytest.mark.parametrize("big", [384, 385, 513])
def test_small_replicas_beside_a_large_one(gpu, big, n_rays, outputs):
    # one launch for the batch: the large replica's sums are one wave's, the small ones' two halves'
    # (513 agents at 2048 rays outgrow the LDS: the 16-wave kernel, and one launch for each class)
    held = (56 + 4 * ((n_rays + 31) // 32 + 1)) * big + 4096 <= 163840
    small = (64, 33, 9, 2, 1, 48, 17, 64)   # (a batch of more than eight replicas)
    a = group((big, *small), n_rays, "infinite", 0)
    parts = [(0, group((big,), n_rays, "infinite", 1 if held else 16))] + [
        (1 + i, group((n,), n_rays, "infinite", 2)) for i, n in enumerate(small)]
    for step in range(2):
        a.step(fields=outputs)
        assert a.last_kernels() == ({"push"} if held else {"big", "per_replica"})
        for at, p in parts:
            p.step(fields=outputs)
            for x, y in zip(a.state_numpy(), p.state_numpy()):
                assert np.array_equal(x[a.replica_slice(at)], y), (step, at)
            if outputs:
                assert np.array_equal(a.fields_numpy(at), p.fields_numpy(0)), (step, at)


def test_counters_of_a_whole_batch(gpu):
    # counted on the push kernel; verified (every pair in float64 too) on the
    # kernels of the size classes, with the same pairs and the same steps
    sizes = (64, 33, 9, 2, 1, 48, 17, 64, 5, 30)
    a, b = (group(sizes, 512, "walls", 0) for _ in range(2))
    for step in range(3):
        a.step(count=True)
        b.step(verify=True)
        assert a.last_kernels() == {"push"} and b.last_kernels() == {"per_replica"}
        for p, q in zip(a.state_numpy(), b.state_numpy()):
            assert np.array_equal(p, q), step
    pairs = 3 * sum(n * (n - 1) for n in sizes)
    got, rechecked, _ = a.fallback_counts()
    assert got == pairs and 0 <= rechecked <= pairs
    got, _, disagree = b.fallback_counts()
    assert got == pairs and disagree == 0

"""The push kernel on replicas that fill a workgroup's LDS to the last bytes (its
limit is what the fields, poses and queues of a replica take, nothing beside
them): steps equal those of the one-wave per-replica kernel, which sums in the
same order, bit for bit, in the step with outputs and in the plain one."""
import numpy as np
import pytest

from test_gpu_push import swarm
from test_gpu_vf_f32 import uniform_start

pytestmark = pytest.mark.gpu


# 163,840 bytes of LDS less these: 32, 32, 48, 32, 0
@pytest.mark.parametrize("n, n_rays", [(1736, 250), (1288, 512), (1079, 700), (644, 1500), (512, 2000)])
def test_replicas_that_fill_the_lds(gpu, n, n_rays):
    from abm_amd.vf import VFConfig
    side = 100.0 * np.sqrt(n)
    cfg = VFConfig(n_agents=n, n_rays=n_rays, width=side, height=side, boundary="infinite", ALP0=1.0, BET0=0.5)
    st = uniform_start(n, side, side, 30, seed=n, v=0.6)
    for outputs in (True, False):
        print(f"  push n={n} R={n_rays} outputs={outputs}", flush=True)
        a, b = swarm([cfg], [st], 0), swarm([cfg], [st], 1)
        for step in range(2):
            for sw in (a, b):
                sw.step(fields=outputs, diag=outputs)
            assert a.last_kernels() == {"push"} and b.last_kernels() == {"per_replica"}
            for p, q in zip(a.state_numpy(), b.state_numpy()):
                assert np.array_equal(p, q), step
            if outputs:
                assert np.array_equal(a.fields.cpu().numpy(), b.fields.cpu().numpy()), step
                assert np.array_equal(a.diag_numpy(), b.diag_numpy()), step

"""Host side of the foraging update over the whole GPU: its plan, its scratch and
the calls a step makes, followed on the CPU with a stand-in for the HIP runtime."""
import pytest

import hip_standin


@pytest.fixture(scope="module")
def standin(tmp_path_factory):
    return hip_standin.build(tmp_path_factory.mktemp("standin"))


def test_a_failed_plan_leaves_the_one_in_use(standin):
    hip_standin.run(standin, """
        h = forage_batch(replica(40), replica(30, visual_exclusion=1))
        log()
        assert forage_step(h) == 0
        before = kernels(log())
        assert before == ["forage_update_kernel", "forage_occlude_kernel"]
        fail("hipMalloc")   # the scratch of the path asked for
        assert lib.abm_forage_set_path(h, 1) == L.ABM_ERR_HIP
        log()
        assert forage_step(h) == 0
        assert kernels(log()) == before
        assert lib.abm_forage_set_path(h, 1) == 0
        assert forage_step(h) == 0
        assert "wide_field_kernel" in kernels(log())
        lib.abm_forage_batch_destroy(h)
        assert held()[0] == 0
        """)

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


def test_a_new_path_leaves_what_captured_steps_read(standin):
    # one of each class: a workgroup each, too many rays for the launches over
    # the whole GPU, exclusion below and above 256 agents, beyond one
    # workgroup's LDS
    hip_standin.run(standin, """
        h = forage_batch(replica(40), replica(20, 9000), replica(30, visual_exclusion=1),
                         replica(300, visual_exclusion=1), replica(2000), replica(25000))
        lib.abm_forage_set_path(h, 1)   # both paths' scratch is made
        log()
        before = held()
        for path in (0, 1, 1, 0):
            assert lib.abm_forage_set_path(h, path) == 0
            assert held() == before
        assert not [ln for ln in log() if "Malloc" in ln or "Free" in ln]
        lib.abm_forage_batch_destroy(h)
        assert held()[0] == 0
        """)


def test_each_replica_has_one_kernel(standin):
    hip_standin.run(standin, """
        def grids(h):
            log()
            assert forage_step(h) == 0
            return {ln.split()[1]: int(ln.split()[2]) for ln in log() if ln.startswith("launch ")}

        own = (replica(40), replica(20, 9000), replica(30, visual_exclusion=1), replica(300, visual_exclusion=1))
        h = forage_batch(*own)
        assert grids(h) == dict(forage_update_kernel=2, forage_occlude_kernel=1, forage_step_kernel=1)
        lib.abm_forage_set_path(h, 1)
        assert grids(h) == dict(forage_update_kernel=1, forage_occlude_kernel=1, forage_step_kernel=1,
                                wide_drive_kernel=1, wide_field_kernel=16, wide_move_kernel=1)
        h = forage_batch(replica(200), *own[1:])   # work for more than one CU
        assert grids(h) == dict(forage_update_kernel=1, forage_occlude_kernel=1, forage_step_kernel=1,
                                wide_drive_kernel=1, wide_field_kernel=64, wide_move_kernel=1)
        h = forage_batch(replica(2000), replica(25000), *own)   # enough of it to fill the GPU
        assert grids(h) == dict(forage_update_kernel=2, forage_occlude_kernel=1, forage_step_kernel=1,
                                wide_drive_kernel=106, wide_field_kernel=16 * 423, wide_move_kernel=106)
        """)

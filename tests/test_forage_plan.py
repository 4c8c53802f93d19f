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


def test_calls_on_several_streams(standin):
    # the null stream has scratch of its own; the others share one, each call
    # behind the launches of the one before it, also of one that failed
    hip_standin.run(standin, """
        h = forage_batch(replica(200), replica(12, visual_exclusion=1))
        log()
        bytes0 = held()[0]
        for s in (None, 64, None, 128, 128):
            assert forage_step(h, s) == 0
            on = "on " + ("(nil)" if s is None else hex(s))
            calls = [ln for ln in log() if "occlude" not in ln]
            if held()[0] > bytes0:   # (first on another stream)
                assert s == 64 and calls.pop(0) == "hipMalloc" and "wide_clear_kernel" in calls.pop(1)
                bytes0 = held()[0]
            steps = ["launch"] * 3 if s is None else ["wait", "launch", "launch", "launch", "record"]
            assert [ln.split()[0] for ln in calls] == steps and all(ln.endswith(on) for ln in calls)
        for which, launched in ((2, 0), (3, 1), (4, 2)):   # (the first is the other replica's)
            fail("hipLaunchKernel", which)
            assert forage_step(h, 64) == L.ABM_ERR_HIP
            calls = log()
            assert len(kernels(calls)) == 1 + launched and calls[-1] == "record on 0x40"
        fail("hipEventRecord")
        assert forage_step(h, 64) == L.ABM_ERR_HIP
        assert log()[-1] == "hipDeviceSynchronize"
        """)


def test_captured_steps_have_scratch_of_their_own(standin):
    hip_standin.run(standin, """
        h = forage_batch(replica(200), replica(100, 1200))
        assert forage_step(h, 256) == 0
        log()
        one = ["wide_clear_kernel", "wide_drive_kernel", "wide_field_kernel", "wide_move_kernel"]
        for s, id, steps in ((64, 1, 3), (128, 1, 1), (64, 2, 2)):   # a stream's capture; a branch of it; the next one
            sim.standin_capture(C.c_void_p(s), C.c_ulonglong(id))
            before = held()[0]
            for _ in range(steps):
                assert forage_step(h, s) == 0
            calls = log()
            assert kernels(calls) == steps * one
            assert calls.count("hipMalloc") == 1 and held()[0] > before
            assert not [ln for ln in calls if ln.split()[0] in ("wait", "record")]
            assert forage_step(h, 256) == 0   # not the stream that is captured
            assert [ln.split()[0] for ln in log()] == ["wait", "launch", "launch", "launch", "record"]
        fail("hipMalloc")
        sim.standin_capture(C.c_void_p(64), C.c_ulonglong(3))
        assert forage_step(h, 64) == L.ABM_ERR_HIP
        log()
        assert forage_step(h, 64) == 0 and kernels(log()) == one
        lib.abm_forage_batch_destroy(h)
        assert held()[0] == 0
        """)


@pytest.mark.parametrize("stream", [None, 64])
def test_a_step_cut_short_leaves_no_cues(standin, stream):
    # the cues are counted by the first launch and cleared by the last: after a
    # call that failed between them the next one clears them first
    hip_standin.run(standin, f"""
        s = {stream}
        h = forage_batch(replica(200))
        assert forage_step(h, s) == 0
        one = ["wide_drive_kernel", "wide_field_kernel", "wide_move_kernel"]
        for which in (1, 2, 3):
            fail("hipLaunchKernel", which)
            assert forage_step(h, s) == L.ABM_ERR_HIP
            fail("hipLaunchKernel", 1)
            assert forage_step(h, s) == L.ABM_ERR_HIP   # the clearing itself
            log()
            assert forage_step(h, s) == 0
            assert kernels(log()) == ["wide_clear_kernel"] + one
            assert forage_step(h, s) == 0
            assert kernels(log()) == one
        """)


def test_many_agents_take_several_launches(standin):
    # 67 million agents, beyond the 2^32 threads of one launch at a wave each
    hip_standin.run(standin, """
        h = forage_batch(*[replica(65536)] * 1025)
        log()
        assert forage_step(h) == 0
        grids = [int(ln.split()[2]) for ln in log() if "wide_field_kernel" in ln]
        assert sum(grids) == 16 * 1025 * 1024 and len(grids) > 1 and max(grids) * 256 < 1 << 32
        h = forage_batch(replica(200), *[replica(1)] * 4200000)   # 16 waves each would be beyond it
        log()
        assert forage_step(h) == 0
        assert kernels(log()) == ["forage_update_kernel"]
        """)

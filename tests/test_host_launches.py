"""What the host library launches, copies and allocates, on the CPU: its sources linked against tests/hoststub/hip_stub.cpp,
which logs the launches.  Each case runs in a process of its own.
"""
import os
import subprocess
import sys
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STUB = os.path.join(ROOT, "tests", "hoststub", "libfluidsx_stub.so")

PRELUDE = """
import ctypes as C
import sys
sys.path.insert(0, {root!r})
import numpy as np
import fluids3_amd.particles as particles
particles.LIB_PATH = {stub!r}
from fluids3_amd import Particles, abi, scenes
stub = particles.lib()
stub.stub_log.restype = C.c_char_p
for f in ("stub_captures", "stub_events", "stub_pinned_bytes", "stub_waits"):
    getattr(stub, f).restype = C.c_long
stub.stub_fail_new.argtypes = [C.c_long]

def launches(call):
    stub.stub_clear_log()
    call()
    return stub.stub_log().decode().split()
"""


def on_stub(code):
    if not os.path.exists(STUB):
        subprocess.run(["make", "-C", os.path.dirname(STUB)], check=True, capture_output=True)
    src = PRELUDE.format(root=ROOT, stub=STUB) + textwrap.dedent(code)
    r = subprocess.run([sys.executable, "-c", src], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout}{r.stderr}"


def test_long_download_without_memory_for_every_thread():
    """A worker thread that cannot be had for want of memory is left out: no thread, the first one only, two."""
    on_stub("""
        ps = Particles()
        n = 1000000  # 12 MB
        ps.Restart(scenes.scaled_dam_break(n))
        pos = np.arange(3 * n, dtype=np.float32).reshape(n, 3)
        ps.Commit(abi.FPOS, pos)
        for nth in (1, 2, 3):
            stub.stub_fail_new(nth)
            got = ps.Retrieve(abi.FPOS)
            stub.stub_fail_new(0)
            assert np.array_equal(got, pos), nth
        ps.close()
    """)


def test_no_steps_need_no_scene():
    """A run of no steps does nothing, also where there is no scene yet; one step is refused then."""
    on_stub("""
        ps = Particles()
        ps.Run(0)
        assert ps.TimeSteps(0, False) == 0.0
        for call in (lambda: ps.Run(1), lambda: ps.TimeSteps(1, False)):
            try:
                call()
            except Exception as e:
                assert "Restart" in str(e)
            else:
                raise AssertionError("a step without a scene")
        ps.Restart(scenes.scaled_dam_break(64))
        assert launches(lambda: ps.Run(0)) == []
        ps.close()
    """)


def test_download_of_no_elements_waits():
    """A download waits for the stream's work, also one that takes no element."""
    on_stub("""
        ps = Particles()
        ps.Restart(scenes.scaled_dam_break(64))
        for call in (lambda: ps.Retrieve(abi.FPOS, 0), lambda: ps.RetrieveAccel(abi.AGRIDCNT, 0)):
            ps.Run(1)
            before = stub.stub_waits()
            assert call().size == 0
            assert stub.stub_waits() > before
        ps.close()
    """)


def test_steps_are_joined_whatever_the_particles_per_thread():
    """In a run the force launch makes the advance and the next insert, also where those stages' own launches (of the
    first step and the last) take several particles a thread: in one scene, in a batch and replayed."""
    on_stub("""
        ps = Particles()
        for insert, advance in ((1, 1), (2, 1), (1, 4), (4, 2)):
            ps.SetStagePpt(abi.STAGE_INSERT, insert)
            ps.SetStagePpt(abi.STAGE_ADVANCE, advance)
            for batch in (False, True):
                sc = scenes.scaled_dam_break(300)
                ps.RestartBatch([sc, sc]) if batch else ps.Restart(sc)
                for run in (lambda: ps.Run(6), lambda: ps.LaunchGraph(3)):
                    log = launches(run)
                    count = lambda part: sum(part in k for k in log)
                    assert count("+next") == 5, (insert, advance, batch, log)
                    assert count("insertParticles") == count("advanceParticles") == 1, (insert, advance, batch, log)
        ps.close()
    """)


def test_autotune_times_what_a_run_launches():
    """The tuner times the force as a run launches it (here fastest in the smallest blocks), offers the pair stages no size
    beyond the largest they launch (here what is tried last looks fastest), and its check takes joined steps too."""
    on_stub("""
        ps = Particles()
        for n, batch, most in ((3000, False, 256), (100000, False, 512), (3000, True, 256), (60000, True, 512)):
            sc = scenes.scaled_dam_break(n)
            ps.RestartBatch([sc, sc]) if batch else ps.Restart(sc)
            res = {}
            log = launches(lambda: res.update(ps.Autotune(2)))
            got = [ps.StageBlockSize(k) for k in range(abi.NUM_STAGES)]
            assert got == [t for t, _ in res.values()]
            assert got[abi.STAGE_FORCE] == 64, (n, batch, got)
            assert got[abi.STAGE_PRESSURE] == 512, (n, batch, got)
            # the candidates' joined steps, two a profile (at most five sizes and two counts), and one a check step
            joined = sum("+next" in k for k in log)
            assert joined == 2 * 7 + 2, (n, batch, joined)
            assert most >= got[abi.STAGE_FORCE]
        ps.close()
    """)


def test_batch_runs_on_after_persistent_launches():
    """Switching a batch to persistent launches and back leaves every stage a table of its blocks."""
    on_stub("""
        ps = Particles()
        sc = scenes.scaled_dam_break(3000)
        for n in (1, 40):
            ps.SetPersistent(True)
            ps.RestartBatch([sc] * n)
            ps.Run(2)
            ps.SetPersistent(False)
            assert any("computeForceWave" in k for k in launches(lambda: ps.Run(2)))
            ps.SetPersistent(True)
            assert any("computeForceBatchP" in k for k in launches(lambda: ps.Run(2)))
        ps.close()
    """)


def test_transfers_without_pinned_memory():
    """Where no pinned memory is to be had, systems are made and arrays copied as before, directly."""
    on_stub("""
        stub.stub_no_pinned(1)
        ps = Particles()
        n = 1000000
        ps.Restart(scenes.scaled_dam_break(n))
        pos = np.arange(3 * n, dtype=np.float32).reshape(n, 3)
        ps.Commit(abi.FPOS, pos)
        for k in (2000, 200000, n):  # a slot, several, a long download
            ps.Commit(abi.FVEL, pos[:k])
            assert np.array_equal(ps.Retrieve(abi.FVEL, k), pos[:k])
            assert np.array_equal(ps.Retrieve(abi.FPOS, k), pos[:k])
        ps.Run(1)
        ps.close()
        stub.stub_no_pinned(0)
        ps = Particles()
        assert stub.stub_pinned_bytes() > 0
        ps.close()
        assert stub.stub_pinned_bytes() == 0
    """)


def test_one_replay_captures_one_pair_of_steps():
    """A replay of two steps that has to capture them first captures no pair that another would follow; a later replay
    of several does, once; a capture of its own takes both."""
    on_stub("""
        ps = Particles()
        ps.Restart(scenes.scaled_dam_break(300))
        def captures(call):
            before = stub.stub_captures()
            call()
            return stub.stub_captures() - before
        assert captures(lambda: ps.LaunchGraph(1)) == 1
        assert captures(lambda: ps.LaunchGraph(1)) == 0
        log = launches(lambda: ps.LaunchGraph(3))
        assert captures(lambda: ps.LaunchGraph(2)) == 0
        assert sum("+next" in k for k in log) == 5 and sum("advanceParticles" in k for k in log) == 1, log
        ps.Run(1)
        assert captures(lambda: ps.LaunchGraph(2)) == 2
        ps.Run(1)
        assert captures(lambda: ps.TimeSteps(3, True)) == 1
        assert captures(lambda: ps.TimeSteps(4, True)) == 2
        assert captures(lambda: ps.TimeSteps(0, True)) == 0
        ps.Run(1)
        assert captures(lambda: ps.CaptureGraph()) == 2
        assert captures(lambda: ps.LaunchGraph(2)) == 0
        ps.close()
    """)


def test_bench_names_the_kernels_that_run():
    """The kernel names of the benchmark's line are those that its timed region launches, at both sides of the counts where
    the lanes to a particle change, for stencil rows of 2 to 4 cells, batches and persistent batches."""
    on_stub("""
        sys.path.insert(0, particles._HERE + "/..")
        import bench
        ps = Particles()
        cases = [(n, 1.5) for n in (300, 81920, 81921, 262144, 262145)] + [(300, 1.0), (300, 2.5)]
        for n, density in cases:
            for batch in (0, 1, 2):  # one scene, a batch, a batch with persistent launches
                sc = scenes.scaled_dam_break(n - 100 if batch else n)
                small = scenes.scaled_dam_break(100)
                sc.grid_density = small.grid_density = density
                ps.SetPersistent(batch == 2)
                ps.RestartBatch([sc, small]) if batch else ps.Restart(sc)
                for graph in (True, False):
                    log = set(launches(lambda: ps.BenchSteps(2, use_graph=graph)))
                    names = bench.launched_kernels(ps.NumPoints(), ps.params.gridSrch, batch > 0, batch == 2, graph)
                    assert set(names) == set(bench.STAGES)
                    assert set(names.values()) <= log, (n, density, batch, graph, names, log)
        ps.close()
    """)

"""The per-wave pair stages at the sizes and densities where their paths change, bit for bit against the oracle.

Lanes per particle change with the particle count; a stencil layer goes through the wave's LDS tile whole, row by row
(dense cells), or from memory (particles of one wave spread over a sparse layer above a dense one).
"""
import numpy as np
import pytest

from fluids3_amd import Particles, abi, derive_params, scenes
from oracle import oracle
from parity import assert_int_equal, bits_equal, valid_mask

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ps():
    p = Particles()
    yield p
    p.close()


def one_step_bitexact(ps, scene, pos=None, vel=None, threads=None):
    ps.Restart(scene)
    if pos is not None:
        ps.Commit(abi.FPOS, pos)
    if vel is not None:
        ps.Commit(abi.FVEL, vel)
        ps.Commit(abi.FVEVAL, vel)
    if threads is not None:
        ps.SetStageBlockSize(abi.STAGE_PRESSURE, threads)
        ps.SetStageBlockSize(abi.STAGE_FORCE, threads)
    s0 = ps.state()
    ps.Run(1)
    g = ps.state()
    ps.SetStageBlockSize(abi.STAGE_PRESSURE, 256)
    ps.SetStageBlockSize(abi.STAGE_FORCE, 256)
    p = ps.params
    ref = oracle.make_state(p, s0["pos"], vel=s0["vel"], veval=s0["veval"], clr=s0["clr"], ids=s0["id"], time=s0["time"])
    oracle.run(p, ref, 1)
    for k in ("gcell", "gndx", "id", "cnt", "off"):
        assert_int_equal(k, g[k], ref[k])
    m = valid_mask(ref)
    for k in ("press", "force"):
        assert bits_equal(g[k][m], ref[k][m]), k
    for k in ("pos", "vel", "veval"):
        assert bits_equal(g[k], ref[k]), k


def swirl(n, seed):
    return (0.3 * np.random.default_rng(seed).standard_normal((n, 3))).astype(np.float32)


# one lane, a wave's last lane, both sides of a wave at 1, 2 and 4 lanes a
# particle, and both sides of the counts where the lanes change (256 CUs)
@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 33, 64, 255, 257, 81920, 81921, 131072, 131073, 262144, 262145])
def test_counts(ps, n):
    one_step_bitexact(ps, scenes.scaled_dam_break(n), vel=swirl(n, n))


# threads a block, over particles that fill no block
@pytest.mark.parametrize("threads", [64, 128, 512, 1024])
@pytest.mark.parametrize("n", [5003, 100003, 270001])
def test_block_sizes(ps, n, threads):
    one_step_bitexact(ps, scenes.scaled_dam_break(n), vel=swirl(n, 7), threads=threads)


def cloud(n, kind, seed):
    """Positions in the 16,384-particle dam break's box (cells of 2.5): `members` to a cell on average."""
    rng = np.random.default_rng(seed)
    if kind == "sparse":  # a thin layer far apart above a dense floor: a wave's particles span many rows
        k = n // 8
        top = np.column_stack([rng.uniform(-28, 28, k), np.full(k, 30.0), rng.uniform(-28, 28, k)])
        floor = np.column_stack([rng.uniform(-28, 28, n - k), rng.uniform(27, 29, n - k), rng.uniform(-28, 28, n - k)])
        return np.concatenate([top, floor]).astype(np.float32)
    side = 2.5 * (n / float(kind)) ** (1.0 / 3.0)
    return (rng.uniform(0, 1, (n, 3)) * side + [-side / 2, 20, -side / 2]).astype(np.float32)


# rows of about 3 x members: around the pad (64), the tile (400 entries a
# layer, then a row) and beyond the bitmask's 8,192 candidates (1,100 a cell);
# 9,000, 100,000 and 280,000 particles take 4, 2 and 1 lanes
@pytest.mark.parametrize("kind", ["sparse", "6", "15", "19", "22", "45", "120", "150", "1100"])
def test_densities_four_lanes(ps, kind):
    one_step_bitexact(ps, scenes.dambreak_16k(9000), pos=cloud(9000, kind, 3), vel=swirl(9000, 4))


@pytest.mark.parametrize("n", [100000, 280000])
@pytest.mark.parametrize("kind", ["sparse", "15", "22", "60", "140"])
def test_densities_fewer_lanes(ps, n, kind):
    sc = scenes.dambreak_4m(n)
    one_step_bitexact(ps, sc, pos=cloud(n, kind, 5), vel=swirl(n, 6))


@pytest.mark.parametrize("gd", [1.0, 1.5, 2.5])
def test_stencils_in_a_batch(ps, gd):
    """Rows of 2, 3 and 4 cells beside rows of 3, each scene as it is alone."""
    a, b = scenes.scaled_dam_break(3001, seed=5), scenes.scaled_dam_break(1030, seed=6)
    a.grid_density = gd
    ps.RestartBatch([a, b])
    ps.Run(2)
    got = ps.state()
    for s, sc in enumerate((a, b)):
        p0, n, _, _ = ps.SceneRange(s)
        with Particles() as one:
            one.Restart(sc)
            one.Run(2)
            want = one.state()
        for k in ("press", "force", "pos", "vel", "veval"):
            assert bits_equal(got[k][p0:p0 + n], want[k]), (s, k)


# In steps that run straight through the force launch also advances and makes
# the next step's insert (one or four lanes to a particle): the same state,
# tables and ranks as single steps, in one scene (with particles that leave the
# grid), in a batch and replayed.
@pytest.mark.parametrize("n", [1, 63, 65, 257, 5003, 60001])
@pytest.mark.parametrize("batch", [False, True])
def test_joined_steps(ps, n, batch):
    def restart():
        if batch:
            ps.RestartBatch([scenes.scaled_dam_break(n), scenes.scaled_dam_break(64), scenes.scaled_dam_break(n + 7)])
        else:
            ps.Restart(scenes.scaled_dam_break(n))
        total = ps.NumPoints()
        pos = ps.state()["pos"]
        pos[:: 9] += 500.0
        ps.Commit(abi.FPOS, pos)
        ps.Commit(abi.FVEL, swirl(total, total))

    states = []
    for steps in ([1] * 5, [5], [2, 3], "graph", "graphs"):
        restart()
        if steps == "graph":
            ps.LaunchGraph(2)
            ps.Run(1)
        elif steps == "graphs":
            ps.Run(1)
            ps.LaunchGraph(1)
            ps.state()
            ps.LaunchGraph(1)
        else:
            for k in steps:
                ps.Run(k)
        states.append(ps.state())
    for s in states[1:]:
        for k in ("gcell", "gndx", "id", "cnt", "off"):
            assert_int_equal(k, s[k], states[0][k])
        m = valid_mask(states[0])
        for k in ("press", "force"):
            assert bits_equal(s[k][m], states[0][k][m]), k
        for k in ("pos", "vel", "veval"):
            assert bits_equal(s[k], states[0][k]), k


# particles and cell tables on both sides of the block counts (24 blocks of
# 2,048 entries) up to which one launch scans them
@pytest.mark.parametrize("n,half", [(2047, 30), (2049, 30), (49152, 30), (49153, 30), (2047, 67), (2047, 68)])
def test_scan_launches(ps, n, half):
    sc = scenes.dambreak_16k(n)
    sc.bound_min.x, sc.bound_max.x = -half, half
    one_step_bitexact(ps, sc, vel=swirl(n, 9))


@pytest.mark.parametrize("threads", [64, 512, 1024])
@pytest.mark.parametrize("n,gd", [(5003, 1.5), (5003, 1.0), (90001, 1.5), (90001, 1.0)])
def test_joined_steps_block_sizes(ps, n, gd, threads):
    sc = scenes.scaled_dam_break(n)
    sc.grid_density = gd
    states = []
    for steps in ([1, 1, 1], [3]):
        ps.Restart(sc)
        pos = ps.state()["pos"]
        pos[:: 7] += 500.0
        ps.Commit(abi.FPOS, pos)
        ps.Commit(abi.FVEL, swirl(n, 8))
        ps.SetStageBlockSize(abi.STAGE_PRESSURE, threads)
        ps.SetStageBlockSize(abi.STAGE_FORCE, threads)
        for k in steps:
            ps.Run(k)
        states.append(ps.state())
        ps.SetStageBlockSize(abi.STAGE_PRESSURE, 256)
        ps.SetStageBlockSize(abi.STAGE_FORCE, 256)
    a, b = states
    for k in ("gcell", "gndx", "id", "cnt", "off"):
        assert_int_equal(k, b[k], a[k])
    m = valid_mask(a)
    for k in ("press", "force"):
        assert bits_equal(b[k][m], a[k][m]), k
    for k in ("pos", "vel", "veval"):
        assert bits_equal(b[k], a[k]), k


# A slot whose particle leaves the grid keeps the force it last held, whichever
# buffer set and launch wrote it: joined steps against single ones in every
# slot, with particles going out through the top in the steps between (one and
# four lanes to a particle, one scene and a batch, eager and replayed).
@pytest.mark.parametrize("n", [5003, 100003])
@pytest.mark.parametrize("batch", [False, True])
def test_force_of_particles_that_leave(ps, n, batch):
    sc = scenes.scaled_dam_break(n)
    P = derive_params(sc)
    top = P.gridMin.tolist()[1] + (P.gridScanMax.tolist()[1] + 1) / P.gridDelta.tolist()[1]

    def restart():
        ps.RestartBatch([sc, sc]) if batch else ps.Restart(sc)
        pos = ps.Retrieve(abi.FPOS)
        vel = np.zeros_like(pos)
        for k in range(5):  # group k leaves in about step k of a run
            pos[k::50, 1] = top - 0.9 * (k + 1)
            vel[k::50, 1] = 0.99 * P.VL
        for b, a in ((abi.FPOS, pos), (abi.FVEL, vel), (abi.FVEVAL, vel)):
            ps.Commit(b, a)

    states, out = [], []
    for steps in ([1] * 6, [6], [2, 4], "graph"):
        restart()
        if steps == "graph":
            ps.LaunchGraph(3)
        else:
            for k in steps:
                ps.Run(k)
                out.append(int(np.count_nonzero(ps.Retrieve(abi.FGCELL) == abi.GRID_UNDEF)))
        states.append(ps.state())
    assert len(set(out[:6])) >= 4  # they leave in several of the steps
    for s in states[1:]:
        assert_int_equal("gcell", s["gcell"], states[0]["gcell"])
        for k in ("force", "press"):
            assert bits_equal(s[k], states[0][k]), k


def test_joined_steps_over_a_large_grid():
    """A cell table beyond the blocks that the two-launch scan takes (8,192 of 2,048 cells): the three-level scan, and the
    set exchange as a launch of its own, in joined steps, eager and replayed."""
    sc = scenes.dambreak_16k(5003)
    sc.bound_min.x, sc.bound_min.z = -330.0, -330.0
    sc.bound_max.x, sc.bound_max.y, sc.bound_max.z = 330.0, 660.0, 330.0
    P = derive_params(sc)
    assert P.gridTotal > 8192 * 2048
    states = []
    with Particles() as ps:
        for steps in ([1] * 5, [5], "graph"):
            ps.Restart(sc)
            ps.Commit(abi.FVEL, swirl(5003, 3))
            if steps == "graph":
                ps.LaunchGraph(2)
                ps.Run(1)
            else:
                for k in steps:
                    ps.Run(k)
            states.append(ps.state())
    for s in states[1:]:
        for k in ("gcell", "gndx", "id", "cnt", "off"):
            assert_int_equal(k, s[k], states[0][k])
        for k in ("press", "force", "pos", "vel", "veval"):
            assert bits_equal(s[k], states[0][k]), k

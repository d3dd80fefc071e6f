"""The ranked path of a host that loads the code object by kernel name (FHostCaps set, tables of gridTotal + 1 entries,
an id buffer, countingSortIndex then countingSortFullRanked with the particle count alone), bit for bit against the
oracle, through the HIP module API.
"""
import ctypes as C

import numpy as np
import pytest

from fluids3_amd import abi, derive_params, fill_points, scenes
from fluids3_amd.particles import CODE_OBJECT
from oracle import oracle
from parity import assert_int_equal, bits_equal, rel_err

pytestmark = pytest.mark.gpu

STRIDE = {abi.FPOS: 12, abi.FVEL: 12, abi.FCLR: 4, abi.FVEVAL: 12, abi.FFORCE: 12, abi.FPRESS: 4, abi.FGCELL: 4,
          abi.FGNDX: 4, abi.FID: 4}
THREADS = 256


class ModuleHost:
    """Buffers, tables and launches of such a host; every buffer has the size that include/fluidsx_params.h states."""

    def __init__(self, P, n):
        self.hip = C.CDLL("/opt/rocm/lib/libamdhip64.so")
        self.P, self.n, self.mem = P, n, []
        self.cells = P.gridTotal + 1
        self.mod = C.c_void_p()
        self.ok(self.hip.hipModuleLoad(C.byref(self.mod), CODE_OBJECT.encode()))
        self.sets = [{b: self.alloc(s * n) for b, s in STRIDE.items()} for _ in range(2)]
        e2 = self.cells // 1024 + 1
        e3 = e2 // 1024 + 1
        assert e3 == 1  # two scan levels
        self.elem = (self.cells, e2, e3)
        sizes = {abi.AGRID: 4 * n, abi.AGRIDCNT: 4 * self.cells, abi.AGRIDOFF: 4 * self.cells, abi.AAUXARRAY1: 4 * e2,
                 abi.AAUXSCAN1: 4 * e2, abi.AAUXARRAY2: 4 * e3, abi.AAUXSCAN2: 4 * e3, abi.ANBRBITS: 4 * 256 * n,
                 abi.AFREC: 32 * n, 15: 4 * 16 * self.cells}
        self.accel = {b: self.alloc(s) for b, s in sizes.items()}
        for name, tab in (("FPnts", self.sets[0]), ("FPntTmp", self.sets[1]), ("FAccel", self.accel)):
            mbuf = (C.c_uint64 * 16)(*[tab.get(b, 0) for b in range(16)])
            self.set_global(name, mbuf)
        self.set_global("FHostCaps", C.c_int(3))  # FX_CAP_TAIL | FX_CAP_RANKED
        self.set_global("FParams", P)

    def ok(self, e):
        assert e == 0, f"HIP error {e}"

    def alloc(self, nbytes):
        p = C.c_void_p()
        self.ok(self.hip.hipMalloc(C.byref(p), C.c_size_t(nbytes)))
        self.mem.append(p)
        self.ok(self.hip.hipMemset(p, 0, C.c_size_t(nbytes)))
        return p.value

    def set_global(self, name, value):
        p, size = C.c_void_p(), C.c_size_t()
        self.ok(self.hip.hipModuleGetGlobal(C.byref(p), C.byref(size), self.mod, name.encode()))
        assert size.value == C.sizeof(value), name
        self.ok(self.hip.hipMemcpy(p, C.byref(value), size, 1))

    def put(self, b, a):
        self.ok(self.hip.hipMemcpy(C.c_void_p(self.sets[0][b]), a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes), 1))

    def get(self, dev, shape, dtype):
        a = np.empty(shape, dtype)
        self.ok(self.hip.hipMemcpy(a.ctypes.data_as(C.c_void_p), C.c_void_p(dev), C.c_size_t(a.nbytes), 2))
        return a

    def launch(self, name, grid, block, *args):
        f = C.c_void_p()
        self.ok(self.hip.hipModuleGetFunction(C.byref(f), self.mod, name.encode()))
        argv = (C.c_void_p * len(args))(*[C.addressof(a) for a in args])
        self.ok(self.hip.hipModuleLaunchKernel(f, *grid, *block, 0, None, argv, None))

    def per_particle(self, name, *args):
        self.launch(name, ((self.n + THREADS - 1) // THREADS, 1, 1), (THREADS, 1, 1), *args)

    def step(self):
        pnum = C.c_int(self.n)
        ptr = lambda b: C.c_uint64(self.accel[b])
        self.ok(self.hip.hipMemset(C.c_void_p(self.accel[abi.AGRIDCNT]), 0, C.c_size_t(4 * self.cells)))
        self.per_particle("insertParticles", pnum)
        e1, e2, e3 = (C.c_int(e) for e in self.elem)
        one = C.c_int(1)
        self.launch("prefixSum", (e2.value, 1, 1), (512, 1, 1), ptr(abi.AGRIDCNT), ptr(abi.AGRIDOFF),
                    ptr(abi.AAUXARRAY1), e1, one)
        self.launch("prefixSum", (e3.value, 1, 1), (512, 1, 1), ptr(abi.AAUXARRAY1), ptr(abi.AAUXSCAN1),
                    ptr(abi.AAUXARRAY2), e2, one)
        self.launch("prefixFixup", (e2.value, 1, 1), (512, 1, 1), ptr(abi.AGRIDOFF), ptr(abi.AAUXSCAN1), e1)
        for b, s in STRIDE.items():  # CopyAllToTemp
            self.ok(self.hip.hipMemcpy(C.c_void_p(self.sets[1][b]), C.c_void_p(self.sets[0][b]),
                                       C.c_size_t(s * self.n), 3))
        self.per_particle("countingSortIndex", pnum)
        self.per_particle("countingSortFullRanked", pnum)
        self.per_particle("computePressure", pnum)
        self.per_particle("computeForce", pnum)
        P = self.P
        self.per_particle("advanceParticles", C.c_float(P.time), C.c_float(P.dt), C.c_float(P.sim_scale), pnum)
        self.ok(self.hip.hipDeviceSynchronize())

    def close(self):
        for p in self.mem:
            self.hip.hipFree(p)
        self.hip.hipModuleUnload(self.mod)


@pytest.fixture()
def stepped():
    """A host after one step of a block that leaves part of a launch block empty, and the oracle's state after it."""
    sc = scenes.dambreak_16k(10007)
    P = derive_params(sc)
    pos, clr = fill_points(sc)
    ids = np.arange(pos.shape[0], dtype=np.uint32)
    h = ModuleHost(P, pos.shape[0])
    for b, a in ((abi.FPOS, pos), (abi.FCLR, clr), (abi.FID, ids)):
        h.put(b, np.ascontiguousarray(a))
    h.step()
    ref = oracle.run(P, oracle.make_state(P, pos, clr=clr, ids=ids), 1)
    yield h, P, ref
    h.close()


def test_ranked_host(stepped):
    h, P, ref = stepped
    got = {"cnt": h.get(h.accel[abi.AGRIDCNT], h.cells, np.uint32), "off": h.get(h.accel[abi.AGRIDOFF], h.cells, np.uint32),
           "gcell": h.get(h.sets[0][abi.FGCELL], h.n, np.int32), "id": h.get(h.sets[0][abi.FID], h.n, np.uint32)}
    for k, v in got.items():
        assert_int_equal(k, v, ref[k])
    for k, b in (("pos", abi.FPOS), ("vel", abi.FVEL), ("veval", abi.FVEVAL), ("force", abi.FFORCE)):
        assert bits_equal(h.get(h.sets[0][b], (h.n, 3), np.float32), ref[k]), k
    assert bits_equal(h.get(h.sets[0][abi.FPRESS], h.n, np.float32), ref["press"])


# the brick kernel under the reference's name: blocks of any shape, some of their voxels beyond the brick
@pytest.mark.parametrize("block", [(8, 8, 4), (64, 1, 1), (3, 5, 7)])
def test_brick_by_the_reference_name(stepped, block):
    h, P, _ = stepped
    res, lo, hi, scalar = (19, 13, 11), (-25.0, 0.0, -25.0), (25.0, 30.0, 25.0), 0.5
    brick = h.alloc(4 * res[0] * res[1] * res[2])
    grid = tuple((r + b - 1) // b for r, b in zip(res, block))
    h.launch("sampleParticles", grid, block, C.c_uint64(brick), (C.c_int * 3)(*res), (C.c_float * 3)(*lo),
             (C.c_float * 3)(*hi), C.c_int(h.n), C.c_float(scalar))
    h.ok(h.hip.hipDeviceSynchronize())
    got = h.get(brick, (res[2], res[1], res[0]), np.float32)
    st = {"pos": h.get(h.sets[0][abi.FPOS], (h.n, 3), np.float32),
          "cnt": h.get(h.accel[abi.AGRIDCNT], h.cells, np.uint32),
          "off": h.get(h.accel[abi.AGRIDOFF], h.cells, np.uint32)}
    want = oracle.sample(P, st, res, lo, hi, scalar)
    assert np.count_nonzero(want) > 100
    assert np.array_equal(got == 0, want == 0)
    assert rel_err(got, want) <= 1e-5  # powers in 32 bits on both sides

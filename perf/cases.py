"""The work that is timed: what a program that uses this library has it do, through its public entry points
(`fluids3_amd.Particles`), from single calls on a few thousand particles to runs of four million.

A case is a dict of plain values; its "kind" says which of these passes it is:

  step      host state in, one step, the whole new state and its forces out (a solver coupled to the caller's own code,
            step by step): latency of small transfers and launches
  evaluate  host state in, the five stages insert .. force called one by one, density and force out in sorted order
  run       host state in, a run of steps (eager, or replays of the captured graph), positions and velocities out:
            frames of an animation, samples of a data set
  batch     the same for many independent scenes in one system
  adjoint   host state in, rollout with loss, gradients with respect to the whole initial state and the scalars
  sample    the particles splatted onto a voxel brick, brick out

Each pass starts from the same host state, so that repeated passes do the same work.  Scenes are this repository's own:
"rest" is the dam break at rest density, "block" the dam break whose block holds its particles compressed, "beach" the
reference's beach with its moving wall and sloped floor.
"""
import math

import numpy as np
import torch

from fluids3_amd import Particles, abi, scenes
from fluids3_amd.particles import fill_points

# steps that a run's or a batch's state has behind it when the pass begins: past the lattice, in motion
EVOLVE = {"rest": 40, "block": 5, "beach": 20}
# pairs within the radius per particle, roughly, over the steps of a pass (for work())
PAIRS = {"rest": 25.0, "block": 180.0, "beach": 36.0}


def listed():
    return [
        # the smallest calls: one step of a few thousand particles between the caller's own code
        {"name": "step_2k", "kind": "step", "scene": "rest", "n": 2000},
        # density and force of a given cloud, stage by stage; an odd size
        {"name": "evaluate_100k", "kind": "evaluate", "scene": "rest", "n": 100003},
        # the 16,384-particle dam break of the reference CPU path's configuration, its 100 steps
        {"name": "run_16k", "kind": "run", "scene": "block", "n": 16384, "steps": 100, "graph": False},
        # a mid-sized scene replayed as a graph, one particle more than a power of two
        {"name": "run_65k_graph", "kind": "run", "scene": "rest", "n": 65537, "steps": 50, "graph": True},
        # the size of the differentiable scene, stepped eagerly
        {"name": "run_262k", "kind": "run", "scene": "rest", "n": 262144, "steps": 50, "graph": False},
        # the headline size: the compressed 4M dam break, as a graph
        {"name": "dam_4m", "kind": "run", "scene": "block", "n": 4000000, "steps": 40, "graph": True},
        # the reference's own 4M scene
        {"name": "beach_4m", "kind": "run", "scene": "beach", "n": 4000000, "steps": 100, "graph": False},
        # 64 uneven scenes in one system
        {"name": "batch_64", "kind": "batch", "scenes": 64, "lo": 8192, "hi": 262144, "steps": 50},
        # the smallest rollout whose gradients are taken
        {"name": "adjoint_2k", "kind": "adjoint", "scenes": 1, "lo": 2000, "hi": 2000, "steps": 3, "every": 2},
        # fitting a 262,144-particle scene: 50 steps, checkpoints every 10
        {"name": "adjoint_262k", "kind": "adjoint", "scenes": 1, "lo": 262144, "hi": 262144, "steps": 50, "every": 10},
        # fitting many uneven scenes at once: 40 steps, checkpoints every 8
        {"name": "adjoint_batch12", "kind": "adjoint", "scenes": 12, "lo": 16384, "hi": 262144, "steps": 40, "every": 8},
        # a brick for a surface or volume renderer
        {"name": "sample_131k", "kind": "sample", "scene": "rest", "n": 131072, "res": 80},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "evaluate", "run", "run", "run", "run", "batch", "adjoint", "adjoint", "sample"])
    if kind in ("step", "evaluate"):
        return {"kind": kind, "scene": "rest", "n": _log(rng, 2000, 200000 if kind == "evaluate" else 20000)}
    if kind == "sample":
        return {"kind": kind, "scene": "rest", "n": _log(rng, 8192, 262144), "res": rng.randint(20, 96)}
    if kind == "batch":
        lo = _log(rng, 4096, 16384)
        return {"kind": kind, "scenes": rng.randint(2, 64), "lo": lo, "hi": _log(rng, 32768, 262144),
                "steps": rng.randint(5, 50)}
    if kind == "adjoint":
        count = rng.choice([1, 1, rng.randint(2, 12)])
        n = _log(rng, 2000, 262144)
        every = rng.randint(2, 12)
        return {"kind": kind, "scenes": count, "lo": n if count == 1 else max(2000, n // 8), "hi": n,
                "steps": rng.randint(3, 40), "every": every}
    scene = rng.choice(["rest", "rest", "block", "beach"])
    n = _log(rng, *{"rest": (2000, 4000000), "block": (8192, 4000000), "beach": (500000, 4000000)}[scene])
    steps = 2 * rng.randint(1, max(1, min(50, 80000000 // n)))
    return {"kind": kind, "scene": scene, "n": n, "steps": steps, "graph": scene != "beach" and rng.random() < 0.5}


# ------------------------------------------------------------------ inputs


def _scene(case, seed):
    n = case["n"]
    if case["scene"] == "beach":
        return scenes.ref_beach(n, seed=seed)
    if case["scene"] == "rest":
        return scenes.scaled_dam_break(n, seed=seed)
    return scenes.dambreak_16k(n, seed=seed) if n <= 32768 else scenes.dambreak_4m(n, seed=seed)


def _scenes(case, seed):
    """The scenes of a batch or of a rollout: uneven sizes and their own viscosities; the same sizes for every seed, so that
    the work is."""
    sizes = scenes.batch_scenes(case["scenes"], case["lo"], case["hi"])
    rng = np.random.default_rng(seed)
    if case["scenes"] == 1:
        return [scenes.scaled_dam_break(case["lo"], seed=seed, visc=float(rng.uniform(0.2, 0.5)))]
    return [scenes.scaled_dam_break(s.num_points, seed=seed + 1 + k, visc=float(rng.uniform(0.2, 0.5)))
            for k, s in enumerate(sizes)]


def _cloud(scene, seed):
    """A scene's jittered lattice, falling and swirling, as host arrays: positions, velocities, evaluation velocities."""
    pos, _ = fill_points(scene)
    rng = np.random.default_rng(seed)
    vel = (0.15 * rng.standard_normal(pos.shape) + [0.4, -0.3, 0.1]).astype(np.float32)
    veval = (vel + np.float32([0.0, 0.0147, 0.0]) * rng.random((pos.shape[0], 1))).astype(np.float32)
    return pos, vel, veval


def _held(ps):
    return [(b, ps.Retrieve(b)) for b in (abi.FPOS, abi.FVEL, abi.FVEVAL)]


def prepare(case, seed):
    kind = case["kind"]
    ps = Particles()
    st = {"kind": kind, "ps": ps, "case": case}
    if kind == "batch":
        ps.RestartBatch(_scenes(case, seed))
        ps.Run(EVOLVE["rest"])
        st["held"] = _held(ps)
        ps.CaptureGraph()
        return st
    if kind == "adjoint":
        every = _scenes(case, seed)
        if len(every) == 1:
            ps.Restart(every[0])
        else:
            ps.RestartBatch(every)
        clouds = [_cloud(s, seed + k) for k, s in enumerate(every)]
        pos, vel, veval = (np.concatenate(c) for c in zip(*clouds))
        st["held"] = [(abi.FPOS, pos), (abi.FVEL, vel), (abi.FVEVAL, veval),
                      (abi.FID, np.arange(pos.shape[0], dtype=np.uint32))]
        for buf, a in st["held"]:
            ps.Commit(buf, a)
        ps.AdjointConfigure(case["steps"], case["every"])
        ps.AdjointSetTarget(_target(pos, seed))
        return st
    scene = _scene(case, seed)
    ps.Restart(scene)
    if kind == "run":
        ps.Run(EVOLVE[case["scene"]])
        st["held"] = _held(ps)
        st["params"] = ps.params
        if case["graph"]:
            ps.CaptureGraph()
        return st
    pos, vel, veval = _cloud(scene, seed)
    st["held"] = [(abi.FPOS, pos), (abi.FVEL, vel), (abi.FVEVAL, veval),
                  (abi.FID, np.arange(pos.shape[0], dtype=np.uint32))]
    if kind == "sample":
        for buf, a in st["held"]:
            ps.Commit(buf, a)
        for stage in range(abi.STAGE_INSERT, abi.STAGE_SORT + 1):
            ps.Stage(stage)
        p = ps.params
        st["res"] = _res(case)
        st["lo"] = [p.bound_min.x, p.bound_min.y, p.bound_min.z]
        st["hi"] = [p.bound_max.x, p.bound_max.y, p.bound_max.z]
    return st


def _target(pos, seed):
    """Where the particles of a rollout should be: a little below where they are."""
    rng = np.random.default_rng(seed + 77)
    return (pos + np.float32([0.3, -0.4, 0.05]) + 0.1 * rng.standard_normal(pos.shape)).astype(np.float32)


def _res(case):
    return [2 * case["res"], case["res"], case["res"]]  # cubes: the box is twice as long as high and deep


# -------------------------------------------------------------------- pass


def _by_id(ids, a):
    out = np.empty_like(a)
    out[ids] = a
    return out


def run(st):
    ps, kind, case = st["ps"], st["kind"], st["case"]
    if kind == "sample":
        return ps.SampleParticles(st["res"], st["lo"], st["hi"])
    for buf, a in st["held"]:
        ps.Commit(buf, a)
    if kind == "step":
        ps.Run(1)
        ids = ps.Retrieve(abi.FID)
        return {name: _by_id(ids, ps.Retrieve(b)) for name, b in
                (("pos", abi.FPOS), ("vel", abi.FVEL), ("veval", abi.FVEVAL), ("press", abi.FPRESS),
                 ("force", abi.FFORCE))}
    if kind == "evaluate":
        ps.InsertParticles()
        ps.PrefixScanParticles()
        ps.CountingSort()
        ps.ComputePressure()
        ps.ComputeForce()
        return {"id": ps.Retrieve(abi.FID), "press": ps.Retrieve(abi.FPRESS), "force": ps.Retrieve(abi.FFORCE)}
    if kind == "adjoint":
        loss, _ = ps.AdjointForward()
        g = ps.AdjointBackward()
        g.pop("ms")
        return {"loss": loss, **g}
    if kind == "batch":
        ps.LaunchGraph(case["steps"] // 2)
    elif case["graph"]:
        ps.LaunchGraph(case["steps"] // 2)
    else:
        if case["scene"] == "beach":
            ps.UpdateParams(st["params"])  # the wall's phase: the clock goes back with the state
        ps.Run(case["steps"])
    return {"pos": ps.Retrieve(abi.FPOS), "vel": ps.Retrieve(abi.FVEL)}


# ------------------------------------------------------------ work of a pass


def work(case):
    """Bytes and operations of one pass.  A step reads and writes each particle's state (position, two velocities, colour,
    id: 44 bytes) and writes density and force (16); 36 operations a pair and 70 a particle.  The host state goes in once
    and the results come out once."""
    kind = case["kind"]
    if kind == "sample":
        nv = 2.0 * case["res"] ** 3
        return {"bytes": 4 * nv + 12.0 * case["n"], "flops": nv * 12.0 * 14}
    if kind in ("batch", "adjoint"):
        n = float(sum(s.num_points for s in _scenes(case, 1)))
    else:
        n = float(case["n"])
    pairs = PAIRS[case.get("scene", "rest")]
    if kind == "adjoint":
        # a step forward and a step back, whose pair terms cost about three times as much
        return {"bytes": case["steps"] * n * (104 + 140) + n * 76, "flops": case["steps"] * n * 4 * (36 * pairs + 70)}
    steps = 1 if kind in ("step", "evaluate") else case["steps"]
    return {"bytes": steps * n * 104 + n * 60, "flops": steps * n * (36 * pairs + 70)}


# ------------------------------------------------- the same in 64 bits, plain

DT, SS, H, MASS, REST, K, STIFF, DAMP, AL, VL = (float(np.float32(v)) for v in (
    0.003, 0.004, 0.01, 0.00020543, 600.0, 1.0, 10000.0, 256.0, 150.0, 3.0))
PI = 3.141592
POLY6 = 315.0 / (64.0 * PI * H ** 9)
SPIKY = -45.0 / (PI * H ** 6)
LAP = 45.0 / (PI * H ** 6)
GAUSS = 1.0 / (PI * 2.0 * H * H) ** 1.5
D2 = SS * SS
RD2 = H * H / D2


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _rows(n, pairs=1 << 27):
    """Slices of n rows of n pairs, about `pairs` of them at a time."""
    step = max(1, pairs // n)
    return [slice(a, min(n, a + step)) for a in range(0, n, step)]


def _density(x):
    out = []
    for s in _rows(x.shape[0]):
        dsq = (x[s, None, :] - x[None]).square().sum(-1)
        t = torch.where((dsq < RD2) & (dsq > 0), (RD2 - dsq) * D2, torch.zeros_like(dsq))
        out.append(MASS * POLY6 * (t ** 3).sum(1))
    rho = torch.cat(out)
    return torch.where(rho == 0, torch.ones_like(rho), rho)


def _force(x, ve, rho, visc, k):
    p = (rho - REST) * k
    out = []
    for s in _rows(x.shape[0], 1 << 25):
        d = x[s, None, :] - x[None]
        dsq = d.square().sum(-1)
        pair = (dsq < RD2) & (dsq > 0)
        r = torch.sqrt(torch.where(pair, dsq, torch.ones_like(dsq)) * D2)
        c = torch.where(pair, H - r, torch.zeros_like(r))
        w = c / (rho[s, None] * rho[None])
        a = SS * -0.5 * c * SPIKY * (p[s, None] + p[None]) / r * w
        b = LAP * visc * w
        out.append(torch.stack([(a * d[..., q] + b * (ve[None, :, q] - ve[s, None, q])).sum(1) for q in range(3)], 1))
    return torch.cat(out)


def _advance(x, v, ve, f, lo, hi):
    a = f * MASS
    push = []
    for q, (face, sign) in ((1, (lo, 1.0)), (1, (hi, -1.0)), (0, (None, 1.0)), (0, (hi, -1.0)), (2, (lo, 1.0)),
                            (2, (hi, -1.0))):
        at = lo[q] if face is None else face[q]
        diff = H - sign * (x[:, q] - at) * SS  # the contact radius is the smoothing radius
        stiff = 0.0 if face is None else STIFF  # the X-min wall's stiffness is scaled by its motion, none here
        adj = torch.where(diff > 0.00001, stiff * diff - DAMP * sign * ve[:, q], torch.zeros_like(diff))
        e = torch.zeros(3, dtype=x.dtype, device=x.device)
        e[q] = sign
        push.append(adj[:, None] * e)
    a = a + sum(push) + torch.tensor([0.0, -float(np.float32(9.8)), 0.0], dtype=x.dtype, device=x.device)
    s = a.square().sum(1, keepdim=True)
    a = torch.where(s > AL * AL, a * (AL / torch.sqrt(torch.clamp(s, min=1e-300))), a)
    s = v.square().sum(1, keepdim=True)
    v = torch.where(s > VL * VL, v * (VL / torch.sqrt(torch.clamp(s, min=1e-300))), v)
    vn = a * DT + v
    return x + vn * (DT / SS), vn, (v + vn) * 0.5


def _sorted(scene, pos):
    """The order that a step's sort puts the particles in: by cell, by sixteenth of the cell along x, by index; the cell is
    found in 32 bits, whose rounding decides it."""
    f = np.float32
    size = f(1.5 * float(f(scene.smooth_radius)) / float(f(scene.grid_density)))
    wc = size / f(scene.sim_scale)
    off = f(2.0 * float(wc))
    lo = [f(f(getattr(scene.bound_min, q)) - off) for q in "xyz"]
    hi = [f(f(getattr(scene.bound_max, q)) + off) for q in "xyz"]
    res = [int(math.ceil(f(b - a) / wc)) for a, b in zip(lo, hi)]
    delta = [f(r) / f(f(r) * wc) for r in res]
    g = [(pos[:, q] - lo[q]) * delta[q] for q in range(3)]
    c = [a.astype(np.int64) for a in g]
    cell = (c[1] * res[2] + c[2]) * res[0] + c[0]
    slab = np.minimum(((g[0] - c[0].astype(f)) * f(16)).astype(np.int64), 15)
    return np.lexsort((np.arange(pos.shape[0]), slab, cell))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("run", "batch"):
        return None  # after dozens of steps two roundings of the same flow are two flows
    dev = _device()
    if kind == "adjoint":
        if case["hi"] * case["hi"] * case["steps"] > 5e7 or case["scenes"] > 1 or case["steps"] > 5:
            return None
        scene = _scenes(case, seed)[0]
        pos, vel, veval = _cloud(scene, seed)
        x0, v0, e0 = (torch.tensor(a, dtype=torch.float64, device=dev, requires_grad=True) for a in (pos, vel, veval))
        visc = torch.tensor(float(scene.visc), dtype=torch.float64, device=dev, requires_grad=True)
        k = torch.tensor(K, dtype=torch.float64, device=dev, requires_grad=True)
        lo, hi = _box(scene)
        x, v, e = x0, v0, e0
        for _ in range(case["steps"]):
            x, v, e = _advance(x, v, e, _force(x, e, _density(x), visc, k), lo, hi)
        t = torch.tensor(_target(pos, seed), dtype=torch.float64, device=dev)
        loss = (x - t).square().sum() / pos.shape[0]
        loss.backward()
        one = [float(loss.detach()), float(visc.grad), float(k.grad)]
        return {"loss": np.array(one[:1]), "gpos": x0.grad.cpu().numpy(), "gvel": v0.grad.cpu().numpy(),
                "gveval": e0.grad.cpu().numpy(), "gvisc": np.array(one[1:2]), "gk": np.array(one[2:])}
    scene = _scene(case, seed)
    pos, vel, veval = _cloud(scene, seed)
    if kind == "sample":
        if case["n"] * 2 * case["res"] ** 3 > 2e11 or dev == "cpu":
            return None
        return _brick(case, scene, pos, dev)
    if case["n"] > 300000 or (dev == "cpu" and case["n"] > 5000):
        return None
    x, v, e = (torch.tensor(a, dtype=torch.float64, device=dev) for a in (pos, vel, veval))
    rho = _density(x)
    f = _force(x, e, rho, float(scene.visc), K)
    if kind == "evaluate":
        order = _sorted(scene, pos)
        return {"id": None, "press": rho.cpu().numpy()[order], "force": f.cpu().numpy()[order]}
    lo, hi = _box(scene)
    xn, vn, en = _advance(x, v, e, f, lo, hi)
    return {"pos": xn.cpu().numpy(), "vel": vn.cpu().numpy(), "veval": en.cpu().numpy(), "press": rho.cpu().numpy(),
            "force": f.cpu().numpy()}


def _box(scene):
    return ([scene.bound_min.x, scene.bound_min.y, scene.bound_min.z],
            [scene.bound_max.x, scene.bound_max.y, scene.bound_max.z])


def _brick(case, scene, pos, dev):
    res = _res(case)
    lo, hi = _box(scene)
    axes = [torch.tensor(np.float32(a) + np.arange(r, dtype=np.float32) / np.float32(r) * (np.float32(b) - np.float32(a)),
                         dtype=torch.float64, device=dev) for a, b, r in zip(lo, hi, res)]
    z, y, x = torch.meshgrid(axes[2], axes[1], axes[0], indexing="ij")
    at = torch.stack([x.reshape(-1), y.reshape(-1), z.reshape(-1)], 1)
    q = torch.tensor(pos, dtype=torch.float64, device=dev)
    h2 = 2.0 * H * H / 8.0
    out = torch.empty(at.shape[0], dtype=torch.float64, device=dev)
    step = max(1, (1 << 27) // q.shape[0])
    for s in (slice(a, a + step) for a in range(0, at.shape[0], step)):
        dsq = sum((at[s, None, k] - q[None, :, k]).square_() for k in range(3))
        out[s] = torch.where((dsq < RD2) & (dsq > 0), GAUSS * torch.exp(dsq * (-D2 / h2)), torch.zeros_like(dsq)).sum(1)
    return out.reshape(res[2], res[1], res[0]).cpu().numpy()

"""The work that users of this library have it do, as cases that a timing program can prepare
and run.

Kinds of case:
- "clip": a scene in hand (particles with velocities, pre-sampled walls) is loaded and advanced
  some frames. Each frame's positions, radii and colours are read back for display while the next
  one is computed; the velocities are read at the end, as a program that saves its state does.
  The scene is loaded again in every pass, so every pass does the same work.
    "dam":     a block of fluid in one corner of a longer tank (the benchmark's workload);
    "pool":    fluid that fills its tank from wall to wall near rest density, sloshing: twice as
               many neighbours per particle as a dam break that has just been let go;
    "drops":   the reference's surface-tension scene, two small cubes (poly6/spiky kernels);
    "column":  the reference's viscosity scene, a tall thin column (poly6/spiky kernels).
- "batch": several independent scenes advanced together in one context; "fluids": two coupled
  fluid objects of one world.
- "gradient": torch.autograd through a rollout of one or several falling droplets: the positions
  after the observed steps, and the gradients with respect to the initial velocities and each
  scene's viscosity and surface tension (one iteration of a parameter recovery).
- "query": SPH density and DFSPH factor of a point set, through the phases of the step.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mps_cuda_amd import KERNEL_CUBIC, HipSim
from mps_cuda_amd import scenes as S
from mps_cuda_amd.autograd import DifferentiableRollout

#: Particle volume over r^3 (R^3/48 * 3.141592 with R = 4 r): the lattice spacing that gives the
#: density `fill` (in units of the rest density) is (VOLUME / fill)^(1/3) r.
VOLUME = 64.0 / 48.0 * 3.141592


def listed() -> list[dict]:
    return [
        # The reference's own test scenes, as a viewer runs them: a few hundred particles, where
        # every launch and every wait of the host counts.
        dict(name="drops_250", kind="clip", scene="drops", size=5, frames=20),
        dict(name="column_2k", kind="clip", scene="column", size=7, height=41, frames=20),
        # The 32^3 dam break that a CPU can still run, from its lattice (half the rest density).
        dict(name="dam_33k", kind="clip", scene="dam", nx=32, ny=32, nz=32, h=0.04, fill=0.5236, frames=16),
        # A settled tank of odd sizes: full neighbour lists, many wall neighbours.
        dict(name="pool_45k", kind="clip", scene="pool", nx=41, ny=27, nz=41, h=0.04, fill=0.97, frames=10),
        # A dam break on its way, of a size between the droplets and the full tank.
        dict(name="dam_257k", kind="clip", scene="dam", nx=61, ny=67, nz=63, h=0.02, fill=0.62, frames=10),
        # The benchmark's size: a million particles, collapsed a little (35 neighbours each).
        dict(name="dam_1m", kind="clip", scene="dam", nx=100, ny=100, nz=100, h=0.02, fill=0.6, frames=10),
        # A large tank long after the dam broke: near rest density everywhere.
        dict(name="pool_525k", kind="clip", scene="pool", nx=105, ny=50, nz=100, h=0.02, fill=0.95, frames=6),
        # Scenes for training data: a dozen at once, of uneven sizes, in one context.
        dict(name="batch_12", kind="batch", scenes=12, n_min=3000, n_max=60000, frames=8),
        # Two fluids of different rest density and viscosity, one above the other.
        dict(name="fluids_2x14k", kind="fluids", nx=37, ny=10, nz=38, frames=8),
        # The differentiable droplet at its full size (64k particles): a few steps and back.
        dict(name="gradient_64k", kind="gradient", scenes=1, n_min=65536, n_max=65536, steps=4, observed=1),
        # One recovery iteration over a small batch of droplets observed twice.
        dict(name="gradient_4x9k", kind="gradient", scenes=4, n_min=4100, n_max=16000, steps=6, observed=2),
        # Densities of a cloud of points.
        dict(name="query_300k", kind="query", n=300007, fill=0.8),
    ]


def draw(rng) -> dict:
    """A case of the same ranges: 250 to 700,000 particles, half to full rest density."""
    kind = rng.choice(["clip"] * 6 + ["batch", "fluids", "gradient", "query"])
    if kind == "clip":
        scene = rng.choice(["dam", "dam", "pool", "pool", "drops", "column"])
        if scene == "drops":
            return dict(kind=kind, scene=scene, size=rng.randint(5, 13), frames=rng.randint(10, 20))
        if scene == "column":
            return dict(kind=kind, scene=scene, size=rng.randint(4, 11), height=rng.randint(20, 60), frames=rng.randint(10, 20))
        n = math.exp(rng.uniform(math.log(2000), math.log(450000 if scene == "pool" else 700000)))
        edge = n ** (1.0 / 3.0)
        nx, nz = (max(6, round(edge * rng.uniform(0.75, 1.35))) for _ in range(2))
        ny = max(6, round(n / (nx * nz)))
        fill = rng.uniform(0.9, 1.0) if scene == "pool" else rng.uniform(0.52, 0.75)
        return dict(kind=kind, scene=scene, nx=nx, ny=ny, nz=nz, h=0.02 if n > 1e5 else 0.04, fill=fill,
                    frames=rng.randint(3, 6) if n > 1e5 else rng.randint(6, 12))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(2, 16), n_min=rng.randint(300, 5000), n_max=rng.randint(6000, 60000),
                    frames=rng.randint(4, 8))
    if kind == "fluids":
        return dict(kind=kind, nx=rng.randint(12, 45), ny=rng.randint(6, 14), nz=rng.randint(12, 45), frames=rng.randint(4, 10))
    if kind == "gradient":
        k = rng.choice([1, 1, 2, 3, 5])
        n = rng.randint(2000, 40000 // k)
        return dict(kind=kind, scenes=k, n_min=n, n_max=round(n * rng.uniform(1.0, 2.0)), steps=rng.randint(2, 6),
                    observed=rng.choice([1, 2]))
    return dict(kind="query", n=round(math.exp(rng.uniform(math.log(500), math.log(600000)))), fill=rng.uniform(0.5, 1.0))


# ---------------------------------------------------------------------------- scenes
def _swirl(pos: np.ndarray, rng: np.random.Generator, speed: float) -> np.ndarray:
    """A smooth divergence-free velocity field: three plane shear waves of one to two periods over
    the fluid's largest extent, largest speed `speed`."""
    extent = float(np.ptp(pos, axis=0).max()) or 1.0
    v = np.zeros_like(pos)
    for _ in range(3):
        k = rng.normal(size=3)
        k /= np.linalg.norm(k)
        a = np.cross(k, rng.normal(size=3))
        a /= max(np.linalg.norm(a), 1e-12)
        v += np.sin(2.0 * math.pi * rng.uniform(1.0, 2.0) / extent * (pos @ k) + rng.uniform(0.0, 2.0 * math.pi))[:, None] * a
    return (v * (speed / max(np.linalg.norm(v, axis=1).max(), 1e-12))).astype(np.float32)


def _lattice(nx: int, ny: int, nz: int, spacing: float, rng: np.random.Generator, jitter: float) -> np.ndarray:
    y, z, x = np.meshgrid(np.arange(ny), np.arange(nz), np.arange(nx), indexing="ij")  # layer by layer
    p = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1).astype(np.float32) * np.float32(spacing)
    return p + rng.uniform(-jitter * spacing, jitter * spacing, size=p.shape).astype(np.float32)


def _tank(pos, size, h, dt, rng, speed, viscosity=0.01, surface_tension=0.05, density=1000.0, **config) -> S.Scene:
    """Fluid in a walled tank with a corner at the origin, as scenes.dam_break sets it up."""
    size = [float(v) for v in size]
    hash_size = [max(64, 1 << math.ceil(math.log2(v / h))) for v in size]
    return S.Scene(
        name="tank", pos=pos, radius=np.full(len(pos), h / 4, np.float32), vel=_swirl(pos, rng, speed),
        physics=dict(dt=dt, gravity=(0.0, -9.81, 0.0), box_min=[0.0, 0.0, 0.0], box_max=size),
        material=dict(radius=h, density=density, viscosity=viscosity, xsph=0.1, surface_tension=surface_tension),
        config=dict(kernel=KERNEL_CUBIC, hash_size=tuple(hash_size), cell_size=h, df_tol=1.0e-2, cd_tol=1.0e-3, **config),
        boundary_mesh=dict(verts=S.CUBE_VERTS, tris=S.CUBE_TRIS, center=[v / 2 for v in size], size=size, radius=h, density=1.0))


def _spacing(h: float, fill: float) -> float:
    return h / 4 * (VOLUME / fill) ** (1.0 / 3.0)


def _clip_scene(case: dict, rng: np.random.Generator) -> S.Scene:
    if case["scene"] in ("drops", "column"):
        sc = (S.surface_tension_test_scene(case["size"]) if case["scene"] == "drops"
              else S.viscosity_test_scene(case["size"], case["height"]))
        sc.pos = (sc.pos + rng.uniform(-0.002, 0.002, size=sc.pos.shape)).astype(np.float32)
        sc.vel = _swirl(sc.pos, rng, 0.2)
        return sc
    h, nx, ny, nz = case["h"], case["nx"], case["ny"], case["nz"]
    s = _spacing(h, case["fill"])
    wall = h / 2  # a particle stays one wall-particle spacing away from the walls
    pool = case["scene"] == "pool"
    pos = _lattice(nx, ny, nz, s, rng, 0.02 if pool else 0.1) + np.float32(wall)
    block = [s * (n - 1) + 2 * wall for n in (nx, ny, nz)]
    grow = (1.0, 1.5, 1.0) if pool else (2.0, 1.25, 1.25)
    return _tank(pos, [b * g for b, g in zip(block, grow)], h, 5.0e-4 if h < 0.03 else 1.0e-3, rng, 0.5)


def _sizes(case: dict) -> list[int]:
    k = case["scenes"]
    lo, hi = math.log(case["n_min"]), math.log(case["n_max"])
    return [round(math.exp(lo + (hi - lo) * q / max(k - 1, 1))) for q in range(k)]


def _batch_scenes(case: dict, rng: np.random.Generator) -> list[S.Scene]:
    """Blocks in the corner of their boxes, of uneven sizes, materials and densities."""
    h = 0.04
    out = []
    for q, n in enumerate(_sizes(case)):
        s = _spacing(h, 0.52 + 0.1 * (q % 4))
        a = math.ceil(n ** (1.0 / 3.0))
        pos = _lattice(a, a, a, s, rng, 0.05)[:n] + np.float32(h / 2)
        edge = max(1.0, 1.3 * s * (a + 2))
        out.append(_tank(pos, (edge, edge, edge), h, 1.0e-3, rng, 0.5, viscosity=0.005 + 0.04 * (q % 5) / 4,
                         surface_tension=0.05 + 0.4 * (q % 3) / 2))
        out[-1].config["hash_size"] = (64, 64, 64)
    return out


def _fluid_scenes(case: dict, rng: np.random.Generator) -> list[S.Scene]:
    """A light fluid above a heavy one in one tank; the walls belong to both."""
    h = 0.04
    s = _spacing(h, 0.9)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    size = [s * (nx - 1) + h, 3.2 * s * ny + h, s * (nz - 1) + h]
    out = []
    for q, density in enumerate((1000.0, 600.0)):
        pos = _lattice(nx, ny, nz, s, rng, 0.02) + np.float32(h / 2)
        pos[:, 1] += np.float32(q * ny * s)
        out.append(_tank(pos, size, h, 1.0e-3, rng, 0.2, viscosity=(0.01, 0.03)[q], density=density))
    for sc in out:
        sc.config.update(hash_size=(64, 64, 64), couple_scenes=1)
    return out


def _droplets(case: dict, seed: int) -> list[S.Scene]:
    return [S.diff_droplet(n=n, radius=0.25 * (n / 65536) ** (1.0 / 3.0), seed=seed + q, viscosity=0.02 + 0.01 * q,
                           surface_tension=0.3 - 0.04 * q, steps=case["steps"]) for q, n in enumerate(_sizes(case))]


def _points(case: dict, seed: int) -> tuple[np.ndarray, float]:
    """Jittered lattice points in a cube, in shuffled order, and their support radius."""
    rng = np.random.default_rng(seed)
    h = 0.02
    a = math.ceil(case["n"] ** (1.0 / 3.0))
    pos = _lattice(a, a, a, _spacing(h, case["fill"]), rng, 0.2)[:case["n"]]
    return pos[rng.permutation(len(pos))], h


# ---------------------------------------------------------------------------- prepare and run
def _display(n: int) -> list[tuple]:
    """Two sets of pinned host buffers (positions, radii, colours): two frames in flight."""
    pin = torch.cuda.is_available()
    return [(torch.empty(n, 3, pin_memory=pin), torch.empty(n, pin_memory=pin), torch.empty(n, 4, pin_memory=pin))
            for _ in range(2)]


def prepare(case: dict, seed: int) -> dict:
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "clip":
        sc = _clip_scene(case, rng)
        return dict(kind=kind, frames=case["frames"], scenes=[sc], walls=[S.sample_walls(HipSim, sc)],
                    sim=HipSim(S.make_config(sc)), display=_display(sc.n))
    if kind in ("batch", "fluids"):
        scs = _batch_scenes(case, rng) if kind == "batch" else _fluid_scenes(case, rng)
        return dict(kind=kind, frames=case["frames"], scenes=scs, walls=[S.sample_walls(HipSim, sc) for sc in scs],
                    sim=HipSim(S.make_config(scs[0])), display=_display(sum(sc.n for sc in scs)))
    if kind == "gradient":
        scs = _droplets(case, seed)
        roll = DifferentiableRollout(scs, steps=case["steps"], checkpoint_every=10)
        v0 = np.concatenate([sc.extra["v0"] for sc in scs]).astype(np.float32)
        leaf = lambda a, t: torch.tensor(a, dtype=t, device="cuda", requires_grad=True)  # noqa: E731
        observed = [case["steps"]] if case["observed"] == 1 else [(case["steps"] + 1) // 2, case["steps"]]
        target = torch.tensor(np.concatenate([sc.pos for sc in scs]), dtype=torch.float32, device="cuda")
        return dict(kind=kind, roll=roll, observed=observed, v0=leaf(v0, torch.float32), target=target,
                    mu=leaf([sc.material["viscosity"] for sc in scs], torch.float64),
                    sigma=leaf([sc.material["surface_tension"] for sc in scs], torch.float64))
    pos, h = _points(case, seed)
    cfg = S.make_config(S.Scene("points", pos, np.full(len(pos), h / 4), None, {}, {},
                                dict(kernel=KERNEL_CUBIC, hash_size=(128, 128, 128), cell_size=h)))
    sim = HipSim(cfg)
    sim.set_physics(5.0e-4, (0.0, -9.81, 0.0), (-1.0, -1.0, -1.0), (4.0, 4.0, 4.0))
    sim.set_fluid_material(h, 1000.0, 0.01, 0.1, 0.05)
    return dict(kind=kind, sim=sim, pos=pos, radius=np.full(len(pos), h / 4, np.float32))


def run(state: dict):
    kind = state["kind"]
    if kind == "gradient":
        return _run_gradient(state)
    sim = state["sim"]
    if kind == "query":
        sim.upload_fluid(state["pos"], state["radius"])
        for phase in ("HASH", "NEIGHBORS", "DENSITY", "ALPHA"):
            sim.run_phase(phase)
        return dict(density=sim.get("FLUID_DENSITY"), alpha=sim.get("FLUID_ALPHA"))
    if kind == "clip":
        S.load_plain(sim, state["scenes"][0], state["walls"][0])
    else:
        S.load_batch(sim, state["scenes"], state["walls"])
    loops, fences = [], [None, None]
    for t in range(state["frames"]):
        st = sim.step()
        loops.append((st.l_df, st.l_cg, st.l_cd))
        if fences[t & 1] is not None:
            sim.fence_wait(fences[t & 1])
        fences[t & 1] = sim.readback_async(*(b.numpy() for b in state["display"][t & 1]))
    for f in fences:
        if f is not None:
            sim.fence_wait(f)
    pos, radius, rgba = state["display"][(state["frames"] - 1) & 1]
    return dict(pos=pos, radius=radius, rgba=rgba, vel=sim.get("FLUID_VEL"), loops=np.array(loops, np.int64))


def _run_gradient(state: dict):
    x = state["roll"].trajectory(state["v0"], state["mu"], state["sigma"], state["observed"])
    loss = (x - state["target"]).square().sum()
    gv, gmu, gsigma = torch.autograd.grad(loss, (state["v0"], state["mu"], state["sigma"]))
    return dict(pos=x.detach(), grad_v0=gv, grad_mu=gmu, grad_sigma=gsigma)


# ---------------------------------------------------------------------------- the work of a pass
def _particles(case: dict) -> int:
    kind = case["kind"]
    if kind == "query":
        return case["n"]
    if kind in ("batch", "gradient"):
        return sum(_sizes(case))
    if kind == "fluids":
        return 2 * case["nx"] * case["ny"] * case["nz"]
    if case["scene"] == "drops":
        return 2 * case["size"] ** 3
    if case["scene"] == "column":
        return case["size"] ** 2 * case["height"]
    return case["nx"] * case["ny"] * case["nz"]


#: Flops per pair: density and factor with their kernels, one pressure iteration (rate of change
#: of the density, then the force), one iteration of the viscosity solve.
DENSITY_PAIR, PRESSURE_PAIR, VISCOSITY_PAIR = 45, 25, 22


def work(case: dict) -> dict:
    """The state read and written once a frame, and the pair terms of the fewest solver iterations
    that such scenes take: two of each pressure solve, and of the viscosity solve 15 (100 at the
    gradients' tolerance, and as many again in their transposed solve)."""
    n = _particles(case)
    pairs = n * (64.0 * case.get("fill", 0.55) - 1.0)
    if case["kind"] == "query":
        return dict(bytes=24.0 * n, flops=pairs * DENSITY_PAIR)
    if case["kind"] == "gradient":
        step = DENSITY_PAIR + 4 * PRESSURE_PAIR + 100 * VISCOSITY_PAIR
        return dict(bytes=case["steps"] * 128.0 * n, flops=case["steps"] * 3.0 * pairs * step)
    step = DENSITY_PAIR + 4 * PRESSURE_PAIR + 15 * VISCOSITY_PAIR
    return dict(bytes=case["frames"] * 88.0 * n, flops=case["frames"] * pairs * step)


# ---------------------------------------------------------------------------- 64-bit values
def exact(case: dict, seed: int):
    """Density and factor of the "query" kind. The other kinds are whole runs of an iterated
    time step, which have no value in 64 bits that a few lines give."""
    if case["kind"] != "query":
        return None
    pos, h = _points(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x = torch.tensor(pos, device=dev, dtype=torch.float64)
    n = len(x)
    vol, cw, cg = VOLUME * (h / 4) ** 3, 8.0 / math.pi, 48.0 / math.pi
    # particles by cell, in a table of the fullest cell's width
    cell = torch.floor(x / h).long()
    cell -= cell.min(0).values - 1
    ext = cell.max(0).values + 2
    key = (cell[:, 0] * ext[1] + cell[:, 1]) * ext[2] + cell[:, 2]
    order = torch.argsort(key)
    count = torch.bincount(key, minlength=int(ext.prod()))
    first = torch.cumsum(count, 0) - count
    width = torch.arange(int(count.max()), device=dev)
    density = torch.full((n,), cw / h ** 3, device=dev, dtype=torch.float64)
    grad, square = torch.zeros_like(x), torch.zeros_like(density)
    for i in torch.arange(n, device=dev).split(65536):
        for o in range(27):
            k = key[i] + ((o // 9 - 1) * ext[1] + (o // 3 % 3 - 1)) * ext[2] + (o % 3 - 1)
            there = width < count[k][:, None]
            j = order[(first[k][:, None] + width).clamp(max=n - 1)]
            d = x[i][:, None] - x[j]
            q = d.norm(dim=2) / h
            there &= (j != i[:, None]) & (q < 1.0)
            near = q <= 0.5
            w = torch.where(near, (6.0 * q - 6.0) * q * q + 1.0, 2.0 * (1.0 - q) ** 3) * (cw / h ** 3)
            g = torch.where(near, 3.0 * q - 2.0, -((1.0 - q) ** 2) / q.clamp(min=1e-30)) * (cg / h ** 5)
            density[i] += torch.where(there, w, 0.0).sum(1)
            term = vol * torch.where(there, g, 0.0)[:, :, None] * d
            grad[i] += term.sum(1)
            square[i] += term.square().sum((1, 2))
    alpha = 1.0 / (square + grad.square().sum(1))
    return dict(density=(density * vol * 1000.0).cpu(), alpha=alpha.cpu())

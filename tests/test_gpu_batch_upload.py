"""A batch laid out on the device from the scenes' own arrays: with and without velocities, masses, walls
and wall masses, sizes around a workgroup's; the arrays read back equal what each scene was given, and
the memory of a larger batch before does not show. Copies: equal, not close.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes

pytestmark = pytest.mark.gpu


def _add(g, n: int, nb: int, given, rng):
    sc = scenes.dam_break(2, 2, 2, 0.02, 0.0, 1, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), 1.0e-3, 1, (64, 64, 64))
    sc.pos, sc.radius = rng.random((n, 3), np.float32), rng.random(n, np.float32)
    sc.vel = rng.standard_normal((n, 3), np.float32) if "vel" in given else None
    mass = rng.random(n, np.float32) if "mass" in given else None
    walls = (rng.random((nb, 3), np.float32), rng.random(nb, np.float32), rng.random(nb, np.float32) if "bmass" in given else None)
    g.batch_add_scene(sc.physics, sc.material, sc.pos, sc.radius, vel=sc.vel, mass=mass, bpos=walls[0] if nb else None,
                      bradius=walls[1] if nb else None, bmass=walls[2] if nb else None)
    h = sc.material["radius"]
    own = sc.material["density"] * (h * h * h / 48.0 * 3.141592)
    return dict(FLUID_POS=sc.pos, FLUID_RADIUS=sc.radius, FLUID_VEL=sc.vel if sc.vel is not None else np.zeros((n, 3), np.float32),
                FLUID_MASS=mass if mass is not None else np.full(n, own, np.float32),
                FLUID_COLOR=np.tile(np.float32([0, 0, 1, 1]), (n, 1)), FLUID_DENSITY=np.zeros(n, np.float32),
                BND_POS=walls[0], BND_RADIUS=walls[1], BND_MASS=walls[2] if walls[2] is not None else np.zeros(nb, np.float32),
                BND_VOLUME=np.zeros(nb, np.float32))


@pytest.mark.parametrize("given", [(), ("vel", "bmass"), ("mass",), ("vel", "mass", "bmass")])
@pytest.mark.parametrize("sizes", [[(1, 0)], [(256, 3), (257, 0), (1, 700)], [(300, 0), (255, 0)], [(5, 1), (512, 0), (511, 0), (40, 257)]])
def test_arrays_of_a_batch(sizes, given):
    rng = np.random.default_rng(len(sizes))
    sc = scenes.dam_break(2, 2, 2, 0.02, 0.0, 1, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), 1.0e-3, 1, (64, 64, 64))
    g = HipSim(scenes.make_config(sc))
    for some in ([(3000, 900), (2000, 10)], sizes, sizes):
        parts = [_add(g, n, nb, given, rng) for n, nb in some]
        g.batch_commit()
        want = {k: np.concatenate([p[k] for p in parts]) for k in parts[0]}
        for t in range(2):
            for name, v in want.items():
                assert np.array_equal(g.get(name), v), (some, t, name)
            g.run_phase("HASH")

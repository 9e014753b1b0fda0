"""The fluid search in hash grids of one or two cells along an axis, where a particle's 27 cells are the
same few over and over and its own cell comes up several times, against the FP32 oracle entry for entry:
one radius and several, with walls (three times the candidates) and without, one pass and two.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes
from oracle.binding import OracleSim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,hash_size", [(1, (1, 1, 1)), (300, (1, 1, 1)), (300, (2, 2, 2)), (2500, (1, 8, 16)), (2500, (2, 1, 8)),
                                         (2500, (8, 16, 1)), (2500, (16, 1, 1)), (133000, (1, 64, 64)), (133000, (2, 64, 64))])
@pytest.mark.parametrize("kind", ["one_radius", "radii", "no_walls", "wide_cells"])
def test_lists_equal_the_oracle(kind, n, hash_size):
    a, h = int(np.ceil(n ** (1.0 / 3.0))), 0.04
    edge = 0.02 * (a + 2)
    sc = scenes.dam_break(max(a, 2), max(a, 2), max(a, 2), 0.02, 0.002, 7, (0.0, 0.0, 0.0), (edge,) * 3, 1.0e-3, 2, hash_size)
    sc.pos, sc.radius = sc.pos[:n], np.full(n, h / 4)
    if kind == "radii":
        sc.radius[np.random.default_rng(n).random(n) < 0.3] *= 0.8
    if kind == "wide_cells":
        sc.config["cell_size"] = 3 * h
    if n > 100000 and kind == "wide_cells":
        sc.config["hash_size"] = (hash_size[0], 16, 16)
    walls = scenes.sample_walls(HipSim, sc)
    if kind == "no_walls":
        walls = tuple(w[:0] for w in walls)
    print(f"[narrow] {kind} n={n} {hash_size}", flush=True)
    g, o = HipSim(scenes.make_config(sc)), OracleSim(scenes.make_config(sc), 32)
    for s in (g, o):
        scenes.load_plain(s, sc, walls)
        s.run_phase("HASH"), s.run_phase("NEIGHBORS")
    for name in ("NEI_FF_IDX", "NEI_FF", "NEI_FB_IDX", "NEI_FB"):
        assert np.array_equal(g.get(name), o.get(name)), name

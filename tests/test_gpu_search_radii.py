"""The fluid search over unequal radii, against the FP32 oracle entry for entry, and two steps on those
lists: radii of two and of many values, one particle of three times the usual radius among the others
(its support is wider than a cell), a radius of zero, walls of two radii, and the same where cells are so
wide that blocks search the global tables. One pass of quads (36 workgroups) and two passes (520).
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes
from oracle.binding import OracleSim

pytestmark = pytest.mark.gpu

SMALL, LARGE = 9000, 133000


@pytest.mark.parametrize("n", [SMALL, LARGE])
@pytest.mark.parametrize("kind,cells,spacing", [("two", 1, 0.02), ("many", 1, 0.02), ("many", 1, 0.0165), ("many", 3, 0.02),
                                                ("one_wide", 1, 0.02), ("zero", 1, 0.02), ("walls", 1, 0.02),
                                                ("walls", 3, 0.02), ("both", 1, 0.0165)])
def test_lists_and_step_equal_the_oracle(kind, cells, spacing, n):
    a, h = int(np.ceil(n ** (1.0 / 3.0))), 0.04
    edge = spacing * (a + 2)
    sc = scenes.dam_break(a, a, a, spacing, 0.1 * spacing, 7, (0.0, 0.0, 0.0), (edge, edge, edge), 1.0e-3, 2, (64, 64, 64))
    rng = np.random.default_rng(n)
    sc.pos, sc.radius = sc.pos[:n], np.full(n, h / 4)
    sc.material["radius"] = sc.boundary_mesh["radius"] = h
    sc.config["cell_size"] = cells * h
    if kind in ("two", "both"):
        sc.radius[rng.random(n) < 0.3] *= 0.8
    if kind == "many":
        sc.radius = (rng.uniform(0.5, 1.0, n) * h / 4).astype(np.float32).astype(np.float64)
    if kind == "one_wide":
        sc.radius[n // 2] *= 3.0
    if kind == "zero":
        sc.pos = np.concatenate([sc.pos, [[0.5 * edge, 0.98 * edge, 0.5 * edge]]]).astype(np.float32)
        sc.radius = np.append(sc.radius, 0.0)
    walls = scenes.sample_walls(HipSim, sc)
    if kind in ("walls", "both"):
        walls = (walls[0], np.where(rng.random(len(walls[1])) < 0.3, 0.8, 1.0).astype(np.float32) * walls[1], walls[2])
    print(f"[radii] {kind} n={n} cells={cells} spacing={spacing}", flush=True)
    g, o = HipSim(scenes.make_config(sc)), OracleSim(scenes.make_config(sc), 32)
    for s in (g, o):
        scenes.load_plain(s, sc, walls)
        s.run_phase("HASH"), s.run_phase("NEIGHBORS")
    lists = ("NEI_FF_IDX", "NEI_FF", "NEI_FB_IDX", "NEI_FB")
    for name in lists:
        assert np.array_equal(g.get(name), o.get(name)), name
    if kind == "zero":  # (its own support is empty: a step divides by it)
        return
    for t in range(2):
        sg, so = g.step(), o.step()
        assert (sg.l_df, sg.l_cg, sg.l_cd) == (so.l_df, so.l_cg, so.l_cd), t
        assert sg.nnz_ff == so.nnz_ff
        for name in ("FLUID_DENSITY", "FLUID_CG_B", "FLUID_VEL", "FLUID_POS"):
            assert np.array_equal(g.get(name), o.get(name)), (t, name)
    for name in lists:
        assert np.array_equal(g.get(name), o.get(name)), name

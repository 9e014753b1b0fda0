"""The fluid search over scattered particles, against the FP32 oracle entry for entry, and steps on those
lists: clouds of less than a particle per cell (every block has more rows and cells than LDS holds), alone
and beside a block of fluid (few such blocks: the second pass takes them from the second search on), in
a grid of one pass of quads and of the two passes.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes
from oracle.binding import OracleSim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_block,n_cloud,per_cell", [(0, 9000, 0.05), (0, 9000, 1.0), (0, 133000, 0.05), (0, 133000, 1.0),
                                                      (9000, 500, 0.3), (140000, 900, 0.3)])
def test_lists_and_step_equal_the_oracle(n_block, n_cloud, per_cell):
    h, spacing, a = 0.04, 0.02, int(np.ceil(n_block ** (1.0 / 3.0)))
    size = max(h * (n_cloud / per_cell) ** (1.0 / 3.0), spacing * (a + 2))
    sc = scenes.dam_break(max(a, 2), max(a, 2), max(a, 2), spacing, 0.1 * spacing, 7, (0.0, 0.0, 0.0), (size, size + spacing * a, size),
                          1.0e-3, 2, (128, 128, 128))
    cloud = np.random.default_rng(n_cloud).uniform(0.0, size, (n_cloud, 3)) + [0.0, spacing * (a + 2) if a else 0.0, 0.0]
    sc.pos = np.concatenate([sc.pos[:n_block], cloud]).astype(np.float32)
    sc.radius = np.full(len(sc.pos), h / 4)
    print(f"[scattered] {n_block} + {n_cloud} particles, {per_cell} per cell", flush=True)
    g, o = HipSim(scenes.make_config(sc)), OracleSim(scenes.make_config(sc), 32)
    walls = (np.zeros((0, 3), np.float32), np.zeros(0, np.float32), np.zeros(0, np.float32))
    for s in (g, o):
        scenes.load_plain(s, sc, walls)
    for t in range(3):
        sg, so = g.step(), o.step()
        assert (sg.l_df, sg.l_cg, sg.l_cd) == (so.l_df, so.l_cg, so.l_cd), t
        for name in ("NEI_FF_IDX", "NEI_FF", "FLUID_DENSITY", "FLUID_CG_B", "FLUID_VEL", "FLUID_POS"):
            assert np.array_equal(g.get(name), o.get(name)), (t, name)

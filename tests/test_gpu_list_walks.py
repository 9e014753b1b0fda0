"""The forms of the list walks (one lane per slot or a quad; shallow or deep halo staging, or
gathers from global memory) at the sizes where they change, against the FP32 oracle.

A sum over a list has the same bits in every form, so the whole step has the oracle's bits: the
tolerance is zero. Sizes: single particles and lists shorter than a group of four; the edges of a
workgroup (256 slots); the workgroup counts where the quad form ends (256 and 512 workgroups); a
lattice near rest density, whose halos are deeper than the shallow staging depth.
"""
import numpy as np
import pytest

from mps_cuda_amd import scenes
from tests.parity import make_pair

pytestmark = pytest.mark.gpu


def _block(n: int, spacing: float, seed: int = 3):
    """n particles of a jittered lattice in the corner of a walled tank, h = 0.04."""
    a = int(np.ceil(n ** (1.0 / 3.0)))
    edge = max(0.5, 1.5 * spacing * (a + 1))
    sc = scenes.dam_break(a, a, a, spacing, 0.1 * spacing, seed, (0.0, 0.0, 0.0), (edge, edge, edge), 1.0e-3, 2,
                          (64, 64, 64))
    # dam_break sets the radius from the spacing; here the radius stays and the spacing varies
    h = 0.04
    sc.pos, sc.radius = sc.pos[:n], np.full(n, h / 4)
    sc.material["radius"] = h
    sc.config["cell_size"] = h
    sc.boundary_mesh["radius"] = h
    return sc


@pytest.mark.parametrize("n,spacing", [(1, 0.02), (2, 0.02), (5, 0.02), (63, 0.02), (255, 0.0165), (257, 0.02),
                                       (4097, 0.0165), (65536, 0.02), (65537, 0.0165), (131072, 0.02), (131073, 0.0165)])
def test_steps_equal_the_oracle_bit_for_bit(n, spacing):
    sc = _block(n, spacing)
    g, o = make_pair(sc)
    print(f"[walks] n={n} spacing={spacing}", flush=True)
    for t in range(2):
        sg, so = g.step(), o.step()
        assert (sg.l_df, sg.l_cg, sg.l_cd) == (so.l_df, so.l_cg, so.l_cd), t
        for name in ("FLUID_DENSITY", "FLUID_ALPHA", "FLUID_FACTOR_ST", "FLUID_CG_B", "FLUID_VEL", "FLUID_POS"):
            assert np.array_equal(g.get(name), o.get(name)), (t, name)
    print(f"[walks] largest halo {sg.halo_max}, lists of {sg.nnz_ff / n:.1f}", flush=True)


@pytest.mark.parametrize("n", [30000, 90000, 150000])
@pytest.mark.parametrize("depth", [0, 1, 2])
def test_deep_and_shallow_staging_equal(n, depth):
    """Halos over 1264 records (compressed lattice): every staging depth, against halos that are not
    staged at all (limit 1), for a quad grid, one between the two quad limits, and a one-lane grid."""
    from mps_cuda_amd import HipSim
    sims = []
    for kw in (dict(halo_limit=1), dict(cg_halo_depth=depth)):
        sc = _block(n, 0.0158)
        cfg = scenes.make_config(sc)
        for k, v in kw.items():
            setattr(cfg, k, v)
        g = HipSim(cfg)
        scenes.load_into(g, sc)
        sims.append(g)
    a, b = sims
    for t in range(3):
        sa, sb = a.step(), b.step()
        assert (sa.l_df, sa.l_cg, sa.l_cd) == (sb.l_df, sb.l_cg, sb.l_cd), t
        for name in ("FLUID_DENSITY", "FLUID_CG_B", "FLUID_VEL", "FLUID_POS"):
            assert np.array_equal(a.get(name), b.get(name)), (t, name)
    assert sb.halo_max > 1264

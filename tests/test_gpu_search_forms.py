"""The forms of the fluid search (one pass with a quad per slot; the one-lane pass, its dense form, the
second pass over the blocks it left; the global tables and k_halo_build for what fits nowhere)
against the FP32 oracle: lists equal entry for entry, the step that uses the block halos bit for bit.

Cases on both sides of 512 workgroups: a lattice near rest density with walls (more candidates than
the usual form holds), two radii in one fluid (staged copies of unequal radius), cells three supports
wide (runs longer than a hit mask), a hash so small that rows wrap around onto themselves, particles
strung out in sheets (many rows and cells per block), a halo limit below every halo, and NaN and
infinite positions.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes
from tests.parity import make_pair

pytestmark = pytest.mark.gpu

SMALL, LARGE = 9000, 133000  # 36 and 520 workgroups


def _scene(kind: str, n: int):
    spacing = 0.0165 if kind in ("dense", "long_runs") else 0.02
    a = int(np.ceil(n ** (1.0 / 3.0)))
    if kind == "sheets":
        a = int(np.ceil((n / 3) ** 0.5))
    h, ny = 0.04, 3 if kind == "sheets" else a
    edge = spacing * (a + 2)
    sc = scenes.dam_break(a, ny, a, spacing, 0.1 * spacing, 7, (0.0, 0.0, 0.0), (edge, max(edge, 0.2), edge), 1.0e-3, 2,
                          (64, 64, 64) if kind != "sheets" else (256, 64, 256))
    sc.pos, sc.radius = sc.pos[:n], np.full(min(n, len(sc.pos)), h / 4)
    sc.material["radius"] = h
    sc.config["cell_size"] = h
    sc.boundary_mesh["radius"] = h
    if kind == "two_radii":
        sc.radius[::3] = 0.8 * h / 4
    if kind == "long_runs":
        sc.config["cell_size"] = 3 * h
    if kind == "wrapped":
        sc.config["hash_size"] = (8, 4, 16) if n == SMALL else (8, 64, 64)
    return sc


@pytest.mark.parametrize("n", [SMALL, LARGE])
@pytest.mark.parametrize("kind", ["dense", "two_radii", "long_runs", "wrapped", "sheets"])
def test_lists_and_step_equal_the_oracle(kind, n):
    sc = _scene(kind, n)
    print(f"[search] {kind} n={sc.n}", flush=True)
    g, o = make_pair(sc)
    for ph in ("HASH", "NEIGHBORS"):
        g.run_phase(ph), o.run_phase(ph)
    for name in ("NEI_FF_IDX", "NEI_FF", "NEI_FB_IDX", "NEI_FB"):
        assert np.array_equal(g.get(name), o.get(name)), name
    for t in range(2):  # the second search knows what the first one left
        sg, so = g.step(), o.step()
        assert (sg.l_df, sg.l_cg, sg.l_cd) == (so.l_df, so.l_cg, so.l_cd), t
        for name in ("FLUID_DENSITY", "FLUID_CG_B", "FLUID_VEL", "FLUID_POS"):
            assert np.array_equal(g.get(name), o.get(name)), (t, name)
    for name in ("NEI_FF_IDX", "NEI_FF", "NEI_FB_IDX", "NEI_FB"):
        assert np.array_equal(g.get(name), o.get(name)), name


@pytest.mark.parametrize("n", [SMALL, LARGE])
def test_halo_limit_below_every_halo(n):
    sims = []
    for limit in (0, 3):
        sc = _scene("dense", n)
        cfg = scenes.make_config(sc)
        cfg.halo_limit = limit
        g = HipSim(cfg)
        scenes.load_into(g, sc)
        sims.append(g)
    for t in range(2):
        s = [g.step() for g in sims]
        assert s[1].halo_spill > 0 and s[0].halo_spill == 0
        for name in ("FLUID_VEL", "FLUID_POS"):
            assert np.array_equal(sims[0].get(name), sims[1].get(name)), (t, name)


@pytest.mark.parametrize("n", [SMALL, LARGE])
def test_nonfinite_positions_are_nobodys_neighbours(n):
    """NaN (of either sign) and infinite positions: the other particles' lists are those of the scene
    without them."""
    sc = _scene("dense", n)
    bad = np.array([3, n // 2, n - 1])
    lists = []
    for spoil in (False, True):
        pos = sc.pos.astype(np.float32).copy()
        # the spoiled particles lie far outside in the reference run, in a cell of their own
        pos[bad] = [[50.0, 50.0, 50.0]] * 3
        if spoil:
            pos[bad] = [[np.nan, 0.1, 0.1], [-np.nan, 0.1, 0.1], [np.inf, 0.1, 0.1]]
            pos[bad[1]].view(np.uint32)[0] |= np.uint32(0x80000000)
        s2 = _scene("dense", n)
        s2.pos = pos
        g = HipSim(scenes.make_config(s2))
        scenes.load_into(g, s2)
        g.run_phase("HASH"), g.run_phase("NEIGHBORS")
        idx, nei = g.get("NEI_FF_IDX"), g.get("NEI_FF")
        lists.append([np.sort(nei[idx[q]:idx[q + 1]]) for q in range(0, n, 97) if q not in bad])
        for q in bad:
            got = nei[idx[q]:idx[q + 1]]
            assert spoil is False or len(got) == 0, (q, got)
    for a, b in zip(*lists):
        assert np.array_equal(a, b)

"""Sums folded by the workgroups that need them (grids of up to 1536 workgroups per scene) against
the fold launches of larger grids and the folds in the last workgroup: the same partial sums added
in the same order, so r.r logs, loop counts and states are equal bit for bit. Sizes: one workgroup,
a remainder, and both sides of the limit.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [200, 65537, 393216, 393217])
def test_folds_in_consumers_match_folds_in_last_workgroup(n):
    a = int(np.ceil(n ** (1.0 / 3.0)))
    edge = 0.02 * (a + 3)
    sims = []
    for fold_in in (0, 1):
        sc = scenes.dam_break(a, a, a, 0.02, 0.002, 4, (0.0, 0.0, 0.0), (edge, edge, edge), 1.0e-3, 2, (128, 128, 128))
        sc.pos, sc.radius = sc.pos[:n], sc.radius[:n]
        cfg = scenes.make_config(sc)
        cfg.cg_fold_in_kernel = fold_in
        g = HipSim(cfg)
        scenes.load_into(g, sc)
        sims.append(g)
    a, b = sims
    print(f"[folds] n={n}", flush=True)
    for t in range(3):
        sa, sb = a.step(), b.step()
        assert (sa.l_df, sa.l_cg, sa.l_cd) == (sb.l_df, sb.l_cg, sb.l_cd), t
        k = min(sa.l_cg + 1, 128)
        assert list(sa.rr_cg[:k]) == list(sb.rr_cg[:k]), t
        for name in ("FLUID_POS", "FLUID_VEL"):
            assert np.array_equal(a.get(name), b.get(name)), (t, name)


@pytest.mark.parametrize("n", [200, 5000, 70001])
def test_pressure_decision_in_the_apply_matches_the_oracle(n):
    """A compressed block: the pressure loops run several iterations, each ended by the apply's own
    fold; loop counts equal, per-iteration errors within FP64 rounding of the oracle's sums (n terms
    added in another order: n * 2^-53 relative)."""
    from tests.parity import make_pair
    a = int(np.ceil(n ** (1.0 / 3.0)))
    edge = max(0.4, 0.015 * (a + 3))
    sc = scenes.dam_break(a, a, a, 0.0148, 0.0007, 4, (0.0, 0.0, 0.0), (edge, edge, edge), 1.0e-3, 2, (64, 64, 64))
    h = 0.04
    sc.pos, sc.radius = sc.pos[:n], np.full(n, h / 4)
    sc.material["radius"] = h
    sc.config["cell_size"] = h
    sc.boundary_mesh["radius"] = h
    g, o = make_pair(sc)
    most = 0
    for t in range(3):
        sg, so = g.step(), o.step()
        assert (sg.l_df, sg.l_cg, sg.l_cd) == (so.l_df, so.l_cg, so.l_cd), t
        for ga, oa, l in ((sg.err_df, so.err_df, sg.l_df), (sg.err_cd, so.err_cd, sg.l_cd)):
            k = min(l, 100)
            np.testing.assert_allclose(ga[:k], oa[:k], rtol=n * 2.0 ** -53, atol=0.0)
        assert np.array_equal(g.get("FLUID_VEL"), o.get("FLUID_VEL")), t
        most = max(most, sg.l_cd)
    print(f"[folds] n={n}: at most {most} constant-density iterations", flush=True)
    assert most > 3

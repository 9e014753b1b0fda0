"""Coupled scenes over 512 workgroups whose first search pass leaves blocks to the second: lists, their
total and the step, with a list capacity below the longest list, which belongs to a block that the
first pass has finished. (The counts of all passes and the ref search go through the same records.)
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes
from oracle.binding import OracleWorld
from tests.parity import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5  # of a coupled step against the oracle world (tests/test_gpu_phases.py)


def _lattice(shape, spacing, at, rng):
    x = np.stack(np.meshgrid(*[np.arange(k) for k in shape], indexing="ij"), -1).reshape(-1, 3) * spacing + at
    return (x + rng.uniform(-0.05 * spacing, 0.05 * spacing, x.shape)).astype(np.float32)


def test_counts_of_a_search_in_two_passes():
    rng = np.random.default_rng(3)
    sc = scenes.dam_break(2, 2, 2, 0.02, 0.002, 0, (0.0, 0.0, 0.0), (1.64, 1.5, 0.9), 1.0e-3, 2, (64, 64, 64))
    r = float(sc.radius[0])
    # a usual fluid with one tight cluster far above it (the longest lists, few candidates), and one near
    # rest density, whose blocks hold more candidates than the first pass stages
    usual = np.concatenate([_lattice((41, 41, 41), 0.02, (0.02, 0.02, 0.02), rng),
                            _lattice((5, 5, 5), 0.006, (0.4, 1.2, 0.4), rng)])
    dense = _lattice((41, 41, 41), 0.0165, (0.842, 0.02, 0.02), rng)
    parts = [usual, dense]
    mats = [dict(sc.material), dict(sc.material, density=600.0)]
    walls = scenes.sample_walls(HipSim, sc)
    cfg = scenes.make_config(sc)
    cfg.couple_scenes, cfg.nei_capacity = 1, 8
    g = HipSim(cfg)
    g.batch_clear()
    for p, m in zip(parts, mats):
        g.batch_add_scene(sc.physics, m, p, r, bpos=walls[0], bradius=walls[1], bmass=walls[2])
    g.batch_commit()
    assert sum((len(p) + 255) // 256 for p in parts) > 512
    print("[coupled search] lists", flush=True)
    g.run_phase("HASH"), g.run_phase("NEIGHBORS")
    idx, nei = g.get("NEI_FF_IDX").astype(np.int64), g.get("NEI_FF").astype(np.int64)
    counts = np.diff(idx)
    assert counts[:len(usual)].max() > 100 > counts[len(usual):].max()
    off = 0
    for p, m in zip(parts, mats):  # each fluid alone takes one pass
        s1 = scenes.dam_break(2, 2, 2, 0.02, 0.002, 0, (0.0, 0.0, 0.0), (1.64, 1.5, 0.9), 1.0e-3, 2, (64, 64, 64))
        s1.pos, s1.radius, s1.material = p, np.full(len(p), r), m
        a = HipSim(scenes.make_config(s1))
        scenes.load_plain(a, s1, walls)
        a.run_phase("HASH"), a.run_phase("NEIGHBORS")
        i0 = a.get("NEI_FF_IDX").astype(np.int64)
        assert np.array_equal(idx[off:off + len(p) + 1] - idx[off], i0)
        assert np.array_equal(nei[idx[off]:idx[off + len(p)]] - off, a.get("NEI_FF"))
        off += len(p)
    print("[coupled search] steps", flush=True)
    w = OracleWorld(scenes.make_config(sc), 2, 32)
    for k in range(2):
        o, ph, m = w.phase(k), sc.physics, mats[k]
        o.set_physics(ph["dt"], ph["gravity"], ph["box_min"], ph["box_max"])
        o.set_fluid_material(m["radius"], m["density"], m["viscosity"], m["xsph"], m["surface_tension"])
        o.upload_boundary(*walls)
        o.upload_fluid(parts[k], r, None)
    for t in range(2):  # the second search runs both passes at once
        st, so = g.step(), w.step()
        assert st.nnz_ff == g.get("NEI_FF_IDX")[-1], t
        x = g.get("FLUID_POS")
        for q, lo, hi in ((0, 0, len(usual)), (1, len(usual), len(x))):
            sg = g.scene_stats(q)
            assert (sg.l_df, sg.l_cd, sg.l_cg) == (so[q].l_df, so[q].l_cd, so[q].l_cg), (t, q)
            assert rel_err(x[lo:hi], w.phase(q).get("FLUID_POS")) <= TOL, (t, q)

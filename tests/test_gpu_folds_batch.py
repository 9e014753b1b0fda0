"""Batches on both sides of the limit up to which sums are folded by the workgroups that need them. The
limit is on the whole grid (1536 workgroups), while each workgroup folds its own scene's sums: a batch
just over it takes fold launches, its scenes alone (384 workgroups each) never do. Equal bit for bit,
also with the CG's sums folded by the last workgroup.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes

pytestmark = pytest.mark.gpu


def _scene(n: int, seed: int):
    a = int(np.ceil(n ** (1.0 / 3.0)))
    edge = 0.02 * (a + 3)
    sc = scenes.dam_break(a, a, a, 0.02, 0.002, seed, (0.0, 0.0, 0.0), (edge, edge, edge), 1.0e-3, 2, (64, 64, 64))
    sc.pos, sc.radius = sc.pos[:n], sc.radius[:n]
    sc.vel = np.random.default_rng(seed).normal(0.0, 0.1 * seed, (n, 3)).astype(np.float32)  # other counts per scene
    return sc


@pytest.mark.parametrize("fold_in", [0, 1])
@pytest.mark.parametrize("last", [98304, 98305])
def test_batch_around_the_limit_equals_scenes_alone(last, fold_in):
    scs = [_scene(98304, 1), _scene(98304, 2), _scene(98304, 5), _scene(last, 9)]
    assert (sum((s.n + 255) // 256 for s in scs) > 1536) == (last == 98305)
    walls = [scenes.sample_walls(HipSim, s) for s in scs]
    cfg = scenes.make_config(scs[0])
    cfg.cg_fold_in_kernel = fold_in
    bat = HipSim(cfg)
    scenes.load_batch(bat, scs, walls)
    print(f"[folds] batch of {sum(s.n for s in scs)}, fold_in={fold_in}", flush=True)
    sb = [bat.step() and [bat.scene_stats(q) for q in range(4)] for _ in range(2)]
    counts, at = set(), 0
    for q, (s, w) in enumerate(zip(scs, walls)):
        g = HipSim(scenes.make_config(s))
        scenes.load_plain(g, s, w)
        for t in range(2):
            a, b = g.step(), sb[t][q]
            assert (a.l_df, a.l_cg, a.l_cd) == (b.l_df, b.l_cg, b.l_cd), (t, q)
            assert list(a.rr_cg[:a.l_cg]) == list(b.rr_cg[:a.l_cg]) and list(a.err_cd[:a.l_cd]) == list(b.err_cd[:a.l_cd])
            counts.add((t, a.l_df, a.l_cg, a.l_cd))
        for name in ("FLUID_POS", "FLUID_VEL"):
            assert np.array_equal(bat.get(name)[at:at + s.n], g.get(name)), (name, q)
        at += s.n
        g.close()
    assert len(counts) > 2  # the scenes' loops end apart

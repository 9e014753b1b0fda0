"""The adjoint's walks with a quad per slot, at scene sizes around a wave's and a workgroup's slots: a scene
has the same gradients, bit for bit, alone and at any place of a batch, and a lone particle has those of
free flight.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes

pytestmark = pytest.mark.gpu


def _scene(n, two_radii):
    sc = scenes.diff_droplet(n=600, radius=0.055, seed=3, steps=2)
    keep = np.argsort(np.linalg.norm(sc.pos - sc.pos.mean(0), axis=1), kind="stable")[:n]
    sc.pos, sc.radius, sc.extra["v0"] = sc.pos[keep], sc.radius[keep].copy(), sc.extra["v0"][keep]
    if two_radii:
        sc.radius[::2] *= 0.8
    return sc


def _grads(scs, kernel=None):
    cfg = scenes.make_config(scs[0])
    if kernel is not None:
        cfg.kernel = kernel
    g = HipSim(cfg)
    scenes.load_batch(g, scs, [scenes.sample_walls(HipSim, s) for s in scs])
    g.set("FLUID_VEL", np.concatenate([s.extra["v0"] for s in scs]))
    g.adj_rollout(2, 2)
    w = np.concatenate([np.random.default_rng(len(s.pos)).normal(size=(len(s.pos), 3)) for s in scs]).astype(np.float32)
    gv, gmu, gsig = g.adj_backward(w)
    at = np.cumsum([0] + [len(s.pos) for s in scs])
    return [(gv[a:b], gmu[q], gsig[q]) for q, (a, b) in enumerate(zip(at, at[1:]))]


@pytest.mark.parametrize("two_radii", [False, True])
@pytest.mark.parametrize("sizes", [(63, 64, 65), (255, 1, 256, 257), (2, 3, 4, 5, 321)])
def test_alone_equals_batched(sizes, two_radii):
    scs = [_scene(n, two_radii) for n in sizes]
    for order in (list(range(len(sizes))), list(range(len(sizes)))[::-1]):
        together = _grads([scs[q] for q in order])
        for q, got in zip(order, together):
            alone = _grads([scs[q]])[0]
            assert np.array_equal(got[0], alone[0]) and got[1] == alone[1] and got[2] == alone[2], sizes[q]
            assert np.isfinite(alone[0]).all() and np.abs(alone[0]).max() > 0


def test_a_lone_particle():
    (gv, gmu, gsig), = _grads([_scene(1, False)])
    w = np.random.default_rng(1).normal(size=(1, 3)).astype(np.float32)
    dt = scenes.diff_droplet(n=600, radius=0.055, seed=3, steps=2).physics["dt"]
    # x_2 = x_0 + 2 dt v_0 + ..., exactly linear in v_0 without neighbours: two FP32 additions of dt w
    assert np.allclose(gv, 2 * dt * w, rtol=4 * 2.0 ** -23, atol=0) and gmu == 0 and gsig == 0

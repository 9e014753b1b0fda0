"""The transposed solve of the adjoint on its staged and gathering paths, with a quad per slot (12 and
256 workgroups) and with one lane (257 and more): the same sums in the same order, so gradients are
equal bit for bit between halos staged in LDS and gathered from global memory, and a scene has the
same gradients alone (quad) and in a batch whose size asks for one lane.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes

pytestmark = pytest.mark.gpu


def _grad(sc, steps=3, **cfgkw):
    cfg = scenes.make_config(sc)
    for k, v in cfgkw.items():
        setattr(cfg, k, v)
    g = HipSim(cfg)
    scenes.load_into(g, sc)
    g.set("FLUID_VEL", sc.extra["v0"])
    g.adj_rollout(steps, 2)
    w = np.random.default_rng(5).normal(size=(sc.n, 3)).astype(np.float32)
    return g.adj_backward(w)


@pytest.mark.parametrize("n", [3000, 65536, 65600])
@pytest.mark.parametrize("two_radii", [False, True])
def test_staged_and_gathered_gradients_equal(n, two_radii):
    sc = scenes.diff_droplet(n=n, radius=0.25 * (n / 65536) ** (1.0 / 3.0), seed=3, steps=3)
    if two_radii:
        sc.radius[::2] *= 0.8
    a, b = _grad(sc), _grad(sc, halo_limit=1)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    assert np.all(np.isfinite(a[0])) and np.abs(a[0]).max() > 0


def test_gradients_alone_equal_those_in_a_large_batch():
    scs = [scenes.diff_droplet(n=n, radius=0.25 * (n / 65536) ** (1.0 / 3.0), seed=7 + n % 5, steps=2) for n in (5000, 70000)]
    alone = _grad(scs[0], 2)
    cfg = scenes.make_config(scs[0])
    g = HipSim(cfg)
    walls = [scenes.sample_walls(HipSim, s) for s in scs]
    scenes.load_batch(g, scs, walls)
    g.set("FLUID_VEL", np.concatenate([s.extra["v0"] for s in scs]))
    g.adj_rollout(2, 2)
    w = np.random.default_rng(5).normal(size=(scs[0].n, 3)).astype(np.float32)
    full = np.zeros((sum(s.n for s in scs), 3), np.float32)
    full[:scs[0].n] = w
    gv, gmu, gsig = g.adj_backward(full)
    assert np.array_equal(gv[:scs[0].n], alone[0])
    assert gmu[0] == alone[1][0] and gsig[0] == alone[2][0]

"""The backward of a rollout whose last segment was recorded as it ran, against the backward that runs it
again: bit for bit, with one segment and several, with the context stepped on or written to between the
two, and for a second backward of the same rollout.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, MPSError, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("between", ["nothing", "step", "write"])
@pytest.mark.parametrize("steps,every", [(1, 1), (4, 10), (5, 2), (4, 2)])
def test_recorded_equals_run_again(steps, every, between):
    sc = scenes.diff_droplet(n=3000, radius=0.09, seed=3, steps=steps)
    obs = sorted({(steps + 1) // 2, steps})
    w = np.random.default_rng(5).normal(size=(len(obs), sc.n, 3)).astype(np.float32)

    def forward(g):
        scenes.load_into(g, sc)
        g.set("FLUID_VEL", sc.extra["v0"])
        return g.adj_rollout_traj(steps, obs, every)[0]

    g = HipSim(scenes.make_config(sc))
    x = forward(g)
    want = g.adj_backward_traj(obs, w)  # nothing differentiated before: runs every segment again
    end = g.get("FLUID_POS"), g.get("FLUID_VEL")
    for t in range(2):
        assert np.array_equal(forward(g), x)
        if between == "step":
            g.step()
        if between == "write":
            g.set("FLUID_VEL", np.zeros((sc.n, 3), np.float32))
        for k in range(2):  # the second backward finds the first segment on the tape
            got = g.adj_backward_traj(obs, w)
            for a, b in zip(got, want):
                assert np.array_equal(a, b), (t, k)
            assert np.array_equal(g.get("FLUID_POS"), end[0]) and np.array_equal(g.get("FLUID_VEL"), end[1])


def test_a_dropped_rollout_stays_refused():
    sc = scenes.diff_droplet(n=600, radius=0.05, seed=3, steps=2)
    g = HipSim(scenes.make_config(sc))
    w = np.ones((sc.n, 3), np.float32)
    for t in range(2):
        scenes.load_into(g, sc)
        g.adj_rollout(2, 2)
        g.adj_backward(w)
    g.adj_rollout(2, 2)
    scenes.load_into(g, sc)
    with pytest.raises(MPSError):
        g.adj_backward(w)

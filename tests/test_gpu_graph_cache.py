"""The cache of captured solver chunks at its limit (256): it is emptied in the middle of a step whose
earlier chunks are still enqueued. Fluids of ever other sizes in one context give three new entries a
step, so the limit is met with each of the three solves. Equal to steps without graphs, bit for bit.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes

pytestmark = pytest.mark.gpu


def test_steps_while_the_cache_is_emptied():
    sc = scenes.dam_break(24, 24, 24, 0.02, 0.002, 4, (0.0, 0.0, 0.0), (0.6, 0.6, 0.6), 1.0e-3, 2, (64, 64, 64))
    out = []
    for graphs in (0, 1):
        cfg = scenes.make_config(sc)
        cfg.use_graphs = graphs
        g = HipSim(cfg)
        scenes.load_into(g, sc)
        g.step()  # sizes every buffer
        res = []
        for k in range(270):  # >= 810 entries: the limit three times
            n = sc.n - 1 - k
            g.upload_fluid(sc.pos[:n], sc.radius[:n])
            st = g.step()
            res.append((st.l_df, st.l_cg, st.l_cd, g.get("FLUID_VEL").tobytes(), g.get("FLUID_POS").tobytes()))
            if k % 90 == 0:
                print(f"[graph cache] graphs={graphs} size {k}", flush=True)
        out.append(res)
    for k, (a, b) in enumerate(zip(*out)):
        assert a == b, k

"""A step enqueued whole (solves and advection gated on the solve before them) against the same step
with a host wait after every chunk of iterations (host_sync_every): bit for bit, where the predicted
counts are too low, too high or met, and where a loop ends at its cap.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes

pytestmark = pytest.mark.gpu


def _scene(n_side: int, seed: int):
    return scenes.dam_break(n_side, n_side + 1, n_side, 0.02, 0.004, seed, (0.0, 0.0, 0.0), (0.5, 0.5, 0.5), 1.0e-3, 6, (64, 64, 64))


def _run(scs, wait: bool, steps: int, **config):
    sc = scs[0]
    cfg = scenes.make_config(sc)
    for k, v in config.items():
        setattr(cfg, k, v)
    if wait:
        cfg.host_sync_every = 3
    g = HipSim(cfg)
    if len(scs) == 1:
        scenes.load_into(g, sc)
    else:
        scenes.load_batch(g, scs, [scenes.sample_walls(HipSim, s) for s in scs])
    out = []
    for t in range(steps):
        if t == 3:  # a kick: the counts jump above the prediction, then fall below it
            v = g.get("FLUID_VEL")
            v += np.random.default_rng(5).normal(0.0, 2.0, v.shape).astype(np.float32)
            g.set("FLUID_VEL", v)
        st = g.step()
        out.append((st.l_df, st.l_cg, st.l_cd, st.hit_cap_df, st.hit_cap_cg, st.hit_cap_cd, st.nonfinite,
                    list(st.err_df)[: st.l_df], list(st.rr_cg)[: st.l_cg], list(st.err_cd)[: st.l_cd],
                    *(g.get(k).tobytes() for k in ("FLUID_POS", "FLUID_VEL", "FLUID_CG_B", "FLUID_FACTOR_ST", "FLUID_KAPPA"))))
    return out


@pytest.mark.parametrize("config", [{}, {"max_iter": 2}, {"cg_max_iter": 3}, {"max_iter": 1, "cg_max_iter": 1},
                                    {"df_tol": 1.0e-7, "max_iter": 9}, {"cd_tol": 1.0e-12, "max_iter": 4},
                                    {"cg_stream_coeffs": 0}, {"use_graphs": 0}, {"cg_fold_in_kernel": 1}],
                         ids=lambda c: ",".join(f"{k}={v}" for k, v in c.items()) or "default")
@pytest.mark.parametrize("scs", [[5], [12], [6, 11, 9]], ids=["one_block", "one_scene", "batch"])
def test_equals_the_step_that_waits(scs, config):
    scs = [_scene(n, 3 + n) for n in scs]
    ahead, waits = _run(scs, False, 6, **config), _run(scs, True, 6, **config)
    for t, (a, b) in enumerate(zip(ahead, waits)):
        assert a == b, (t, a[:7], b[:7])
    if not config:  # the counts did change both ways
        counts = [a[:3] for a in ahead]
        assert any(y[q] > x[q] for x, y in zip(counts, counts[1:]) for q in range(3)), counts
        assert any(y[q] < x[q] for x, y in zip(counts, counts[1:]) for q in range(3)), counts

"""A.p with and without the non-temporal hint on its coefficients: one lane per slot below and above the
memory-side cache, shallow and deep halos, against the operator that recomputes one of the two
coefficients (the same bits). Equal, not close.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,spacing", [(53, 0.01), (53, 0.0084), (94, 0.01), (76, 0.0084)],
                         ids=["fits", "fits_deep", "streams", "streams_deep"])
def test_streamed_equals_recomputed(side, spacing):
    out = []
    for stream in (1, 0):
        edge = spacing * (side + 3)
        sc = scenes.dam_break(side, side, side, spacing, 0.1 * spacing, 3, (0.0, 0.0, 0.0), (edge, edge, edge), 5.0e-4, 2,
                              (128, 128, 128))
        sc.radius = np.full(sc.n, 0.005)
        sc.material["radius"] = sc.config["cell_size"] = sc.boundary_mesh["radius"] = 0.02
        cfg = scenes.make_config(sc)
        cfg.cg_stream_coeffs = stream
        g = HipSim(cfg)
        scenes.load_into(g, sc)
        print(f"[streams] {sc.n} particles, stream={stream}", flush=True)
        st = [g.step() for _ in range(2)]
        out.append(([(s.l_df, s.l_cg, s.l_cd, s.nnz_ff) for s in st], g.get("FLUID_VEL"), g.get("FLUID_POS")))
    assert out[0][0] == out[1][0]
    assert (out[0][0][0][3] * 10 <= 210e6) == (side == 53)
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])

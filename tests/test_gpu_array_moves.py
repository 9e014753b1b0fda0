"""Fluid arrays to and from the host in reference order, moved on the device a part (2^20 particles) at a
time: uploads with and without velocities and masses, reads and writes of every width and of part of
a record, before and after a hash has moved the slots. Copies: equal, not close.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes

pytestmark = pytest.mark.gpu
ARRAYS = {"FLUID_POS": 3, "FLUID_VEL": 3, "FLUID_RADIUS": 1, "FLUID_MASS": 1, "FLUID_COLOR": 4, "FLUID_DENSITY": 1,
          "FLUID_KAPPA": 1, "FLUID_CG_B": 3}


@pytest.mark.parametrize("given", [(), ("vel",), ("mass",), ("vel", "mass")])
@pytest.mark.parametrize("n", [1, 255, 257, 1 << 20, (1 << 20) + 3, (1 << 21) + 1])
def test_upload_write_and_read_back(n, given):
    rng = np.random.default_rng(n)
    sc = scenes.dam_break(2, 2, 2, 0.02, 0.0, 1, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), 1.0e-3, 1, (64, 64, 64))
    g = HipSim(scenes.make_config(sc))
    g.set_fluid_material(0.04, 1000.0, 0.01, 0.1, 0.05)
    put = dict(vel=rng.standard_normal((n, 3), np.float32), mass=rng.random(n, np.float32))
    want = {"FLUID_POS": rng.random((n, 3), np.float32), "FLUID_RADIUS": rng.random(n, np.float32)}
    g.upload_fluid(want["FLUID_POS"], want["FLUID_RADIUS"], **{k: put[k] for k in given})
    want["FLUID_VEL"] = put["vel"] if "vel" in given else np.zeros((n, 3), np.float32)
    if "mass" in given:
        want["FLUID_MASS"] = put["mass"]
    want["FLUID_COLOR"] = np.tile(np.float32([0, 0, 1, 1]), (n, 1))
    for name in ("FLUID_DENSITY", "FLUID_KAPPA"):
        want[name] = np.zeros(n, np.float32)
    mass = g.get("FLUID_MASS")
    assert "mass" in given or (mass == mass[0]).all()
    for t in range(2):
        for name, v in want.items():
            assert np.array_equal(g.get(name), v), (t, name)
        g.run_phase("HASH")
    for name, w in ARRAYS.items():  # every array with values of its own; a write leaves the others alone
        want[name] = rng.random((n, w) if w > 1 else n, np.float32)
        g.set(name, want[name])
    for t in range(2):
        for name, v in want.items():
            assert np.array_equal(g.get(name), v), (t, name)
        g.run_phase("HASH")

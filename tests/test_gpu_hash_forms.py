"""The fluid hash at the sizes where its sort changes form, against a stable NumPy sort: one workgroup
(up to 8192 items), tiles of 2048 whose scatter sums the histograms itself (up to 32 tiles), tiles with a
scan in between; digits of 4 to 11 bits, one pass or several. Integers: equal, not close.
"""
import numpy as np
import pytest

from mps_cuda_amd import HipSim, scenes

pytestmark = pytest.mark.gpu


def _sim(n: int, hash_size, cell: float, seed: int):
    sc = scenes.dam_break(2, 2, 2, 0.02, 0.0, 1, (0.0, 0.0, 0.0), (0.2, 0.2, 0.2), 1.0e-3, 1, hash_size)
    rng = np.random.default_rng(seed)
    sc.pos = rng.uniform(-0.3, 1.9, (n, 3)).astype(np.float32)
    sc.radius = np.full(n, 0.01)
    sc.config["cell_size"] = cell
    g = HipSim(scenes.make_config(sc))
    scenes.load_into(g, sc)
    return g


def _linear_keys(pos, hash_size, cell):
    c = np.trunc(pos.astype(np.float64) * (1.0 / float(np.float32(cell)))).astype(np.int64) + np.array(hash_size) // 2
    c &= np.array(hash_size) - 1
    return (c[:, 2] * hash_size[1] + c[:, 1]) * hash_size[0] + c[:, 0]


@pytest.mark.parametrize("n", [1, 64, 1023, 1025, 8191, 8192, 8193, 65536, 65537, 70001])
@pytest.mark.parametrize("hash_size", [(4, 2, 4), (16, 16, 16), (64, 64, 64), (128, 32, 64), (256, 8, 8), (1024, 8, 8)])
def test_hash_equals_a_stable_sort(n, hash_size):
    cell = 0.25
    g = _sim(n, hash_size, cell, n)
    print(f"[hash] n={n} {hash_size}", flush=True)
    pos = g.get("FLUID_POS")  # in reference order
    want = _linear_keys(pos, hash_size, cell)
    order = np.argsort(want, kind="stable")
    for t in range(2):  # the second hash starts from moved slots and a used table
        g.run_phase("HASH")
        key, ids = g.get("FHASH_KEY"), g.get("FHASH_ID")
        assert np.array_equal(key, want[order]) and np.array_equal(ids, order), t
        first = np.flatnonzero(np.r_[True, key[1:] != key[:-1]])
        start, end = g.get("FHASH_START"), g.get("FHASH_END")
        used = np.zeros(start.size, bool)
        used[key] = True
        assert np.array_equal(start[key[first]], first) and np.array_equal(end[key[first]], np.r_[first[1:], n]), t
        assert (start[~used] == 0xFFFFFFFF).all() and (end[~used] == 0xFFFFFFFF).all(), t
        assert np.array_equal(g.get("FLUID_POS"), pos), t

"""GPU check of the ids of generated particles: they count the particles through the cells of tiles that
divide the grid (the largest edge up to 8, or the given ones), whatever tiles the context works with."""
import numpy as np
import pytest

import allscale_ipic3d_amd as G

pytestmark = pytest.mark.gpu


def _first_ids(n, tile, ppc):
    """The id of each cell's first particle, row-major."""
    T = [t or max(d for d in range(1, 9) if k % d == 0) for k, t in zip(n, tile)]
    x, y, z = np.indices(n).reshape(3, -1)
    order = np.lexsort((z % T[2], y % T[1], x % T[0], z // T[2], y // T[1], x // T[0]))
    first = np.empty(ppc.size, dtype=np.int64)
    first[order] = np.concatenate([[0], np.cumsum(ppc[order])[:-1]])
    return first


@pytest.mark.parametrize("n, tile", [((9, 7, 11), (0, 0, 0)), ((17, 8, 3), (0, 0, 0)), ((12, 10, 8), (0, 0, 0)),
                                     ((47, 5, 9), (1, 5, 3)), ((9, 11, 10), (3, 0, 5))], ids=str)
def test_ids_of_generated_particles(n, tile):
    ppc = np.random.default_rng(3).integers(0, 7, size=n[0] * n[1] * n[2]).astype(np.int32)
    sim = G.Simulation(n, dt=0.1, species=((-0.01, -1.0),), tile=tile, track_ids=True)
    sim.init_particles(0, ppc, (0.1, 0.1, 0.1), seed=4)
    p = sim.download_particles(0)
    order = np.lexsort((p["ids"], p["cell"]))
    cell, ids = p["cell"][order], p["ids"][order].astype(np.int64)
    np.testing.assert_array_equal(np.bincount(cell, minlength=ppc.size), ppc)
    within = np.arange(len(cell)) - np.concatenate([[0], np.cumsum(ppc)[:-1]])[cell]
    np.testing.assert_array_equal(ids, _first_ids(n, tile, ppc.astype(np.int64))[cell] + within)
    # the accumulator that the numbers passed through is clean: the counts stay right
    sim.step(3)
    assert sim.num_particles() == ppc.sum() == sim.cell_counts().sum()
    sim.close()

"""GPU checks of grids whose sides have no divisor of 5 to 8, against the oracle: the last tile of an axis
is shorter (by 1 to 7 cells, down to a single layer), so cell numbers, tile partials of J, counters and the
paths over tile faces and the periodic seam all see tiles of different shapes.  Most particles change
cell every step.  FP32 rounding of 3 steps stays below 1e-5 (20 roundings a step of 6e-8)."""
import numpy as np
import pytest

from oracle.compare import particle_errors
from tests._helpers import gpu_sim_for, make_case, rel_err

pytestmark = pytest.mark.gpu

GRIDS = [(9, 11, 13), (17, 8, 22), (41, 9, 10), (57, 13, 4), (9, 33, 26)]


@pytest.mark.parametrize("n", GRIDS, ids=str)
@pytest.mark.parametrize("kind", ["box", "ids", "sink"])
def test_short_last_tiles(n, kind):
    sink = {"sink_center": tuple(0.5 * v for v in n), "sink_radius": 2.0} if kind == "sink" else {}
    case = make_case(n=n, ppc=12, species=((-1.0, 4.0), (0.25, 1.5)), dt=0.1, B=(0, 0.2, 1.0), E_sigma=1e-3, seed=5,
                     drift=(0.5, 0.0, -0.5), **sink)
    u, sim = case[0], gpu_sim_for(case, track_ids=kind == "ids")
    for s in range(2 if kind == "box" else 0):  # the device generator numbers cells itself: the same particles
        sim.init_particles(s, 12, ((4.0,) * 3, (1.5,) * 3)[s], (0.5, 0.0, -0.5), seed=5)
    for _ in range(3):
        u.step(1)
        sim.step(1)
    got, ref = sim.download_fields(), u.fields()
    for k in ("E", "Bc", "Bn", "J"):
        assert rel_err(got[k], ref[k]) < 1e-5, k
    for e in particle_errors(u, sim, case[1]):
        assert abs(e["particles"] - e["particles_ref"]) <= (4 if sink else 0)  # rounding on the sink's face
        assert e["flip_cells"] <= 40  # FP32 and FP64 on different sides of a face
        assert e["offset_max"] < 1e-5 and e["velocity_max"] < 1e-5
    for s in range(2):
        p = sim.download_particles(s)
        assert np.array_equal(np.bincount(p["cell"], minlength=sim.ncell), sim.cell_counts(s))
    sim.close()
    u.close()


def test_many_tiles_are_scanned_in_groups():
    """One cell a tile, more tiles than the scan reads one by one."""
    n = (32, 31, 30)
    case = make_case(n=n, ppc=3, species=((-1.0, 1.0), (0.5, 0.4)), dt=0.1, B=(0, 0.2, 1.0), seed=8)
    u, sim = case[0], gpu_sim_for(case, track_ids=False, tile=(1, 1, 1))
    for _ in range(3):
        u.step(1)
        sim.step(1)
    assert rel_err(sim.download_fields()["J"], u.fields()["J"]) < 1e-5
    for e in particle_errors(u, sim, case[1]):
        assert e["particles"] == e["particles_ref"] and e["flip_cells"] <= 40
    sim.close()
    u.close()

"""GPU check of the field arrays that a caller holds through the field-state view: what it writes there
moves the particles of the next step, with one and two substeps and with the static field, whose
steps update nothing.  The tolerance is that of the other comparisons with the FP64 oracle: a
push and a field update round each component some twenty times (20 * 6e-8, below 1e-5)."""
import numpy as np
import pytest

from oracle.compare import particle_errors
from tests._helpers import gpu_sim_for, make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("substeps", [0, 1, 2])
def test_written_fields_move_the_particles(substeps):
    from allscale_ipic3d_amd import field_operator as FO
    n = (9, 7, 6)
    case = make_case(n=n, ppc=8, species=((-1.0, 0.2), (0.5, 0.3)), dt=0.1, B=(0, 0.25, 1.0), seed=5,
                     field_substeps=substeps)
    u, sim = case[0], gpu_sim_for(case, track_ids=False)
    rng = np.random.default_rng(6)
    for _ in range(2):
        u.step(1)
        sim.step(1)
        view = sim.field_state()
        new = {}
        for name, mean in (("E", view["E0"]), ("Bc", view["B0"])):
            rows = np.zeros((sim.ncell, 4), dtype=np.float32)
            rows[:, :3] = rng.normal(0.0, 0.5, size=(sim.ncell, 3))
            FO.dev_copy(view[name], rows.ctypes.data, rows.nbytes)
            new[name] = rows[:, :3].astype(np.float64) + mean
        u.set_fields(new["E"], new["Bc"])
    u.step(1)
    sim.step(1)
    for e in particle_errors(u, sim, case[1]):
        assert e["flip_particles"] <= 1
        assert e["velocity_max"] < 1e-5 and e["offset_max"] < 1e-5, e
    sim.close()
    u.close()

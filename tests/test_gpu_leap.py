"""GPU checks of the fused field substeps against the oracle: every split of the substeps into launches of
two and of one, boxes cut off by the grid, grids smaller than a box and its surrounding layers, the
static sources of a non-uniform background, and the gather fields that the next push reads.

The tolerance: a substep rounds each component about six times (2^-24 of terms no larger than the
field), so 3 steps of at most 9 substeps stay below 3 * 9 * 6 * 6e-8 = 1e-5 of the field."""
import pytest

from tests._helpers import gpu_sim_for, make_case, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(8, 8, 8), (9, 7, 5), (16, 24, 17), (3, 2, 1), (1, 40, 2)], ids=str)
@pytest.mark.parametrize("substeps", [1, 2, 3, 4, 5, 6, 7, 9])
def test_substeps(n, substeps):
    case = make_case(n=n, ppc=6, species=((-1.0, 0.05), (0.25, 0.1)), w=(0.5, 1.0, 2.0), dt=0.1, B=(0, 0.2, 1.0),
                     E_sigma=0.05, seed=substeps, field_substeps=substeps)
    u, sim = case[0], gpu_sim_for(case, track_ids=False)
    before = sim.field_state()
    for _ in range(3):
        u.step(1)
        sim.step(1)
    got, ref = sim.download_fields(), u.fields()  # ahead of field_state(), which forms the J after the push
    for k in ("E", "Bc", "Bn", "J"):
        assert rel_err(got[k], ref[k]) < 1e-5, k
    after = sim.field_state()
    assert (before["E"], before["Bc"]) == (after["E"], after["Bc"])  # the arrays handed out stay the live ones
    sim.close()
    u.close()

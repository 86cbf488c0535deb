"""GPU checks of the push kernel at the edges of its queues and counters, against the oracle: blocks
on both sides of 2^16 particles of a species and cells on both sides of 2^15 (half-word counters in
LDS), an odd number of species (two share a word), particle arrays that end in runs of one to five
(16-byte loads past the end), and steps in which most particles change cell."""
import numpy as np
import pytest

from tests._helpers import gpu_sim_for, make_case, rel_err

pytestmark = pytest.mark.gpu


def _check(case, steps, flips=4):
    u, sim = case[0], gpu_sim_for(case, track_ids=False)
    ncell = sim.ncell
    for _ in range(steps):
        u.step(1)
        sim.step(1)
    parts, cell = u.particles()
    for s, (_, qom) in enumerate(case[1]):
        ref = np.bincount(cell[parts["qom"] == qom], minlength=ncell)
        got = sim.cell_counts(s)
        assert got.sum() == ref.sum()
        # FP32 and FP64 may put a particle on different sides of a face
        assert np.abs(got - ref).sum() <= flips
    assert rel_err(sim.download_fields()["J"], u.fields()["J"]) < 1e-5
    assert abs(sim.conservation()["kinetic_energy"] / u.kinetic_energy() - 1) < 1e-5
    sim.close()
    u.close()


@pytest.mark.parametrize("crowd", [32767, 32768, 65535, 65536, 70001])
def test_crowded_cell(crowd):
    ppc = np.full(512, 3)
    ppc[100] = crowd
    _check(make_case(n=8, ppc=16, species=((-1.0, 0.05), (0.25, 0.3)), dt=0.1, B=(0, 0.2, 1.0), seed=2,
                     ppc_per_cell=ppc), 2, flips=20)


@pytest.mark.parametrize("species", [1, 3])
@pytest.mark.parametrize("last", [1, 2, 3, 4, 5])
def test_runs_at_the_array_end(species, last):
    n = (6, 5, 16)
    ppc = np.random.default_rng(last).integers(0, 12, size=480)
    ppc[-1] = last
    kinds = ((-1.0, 0.2), (0.5, 0.4), (0.125, 0.1))[:species]
    _check(make_case(n=n, ppc=8, species=kinds, dt=0.1, B=(0, 0.2, 1.0), E_sigma=1e-3, seed=7, ppc_per_cell=ppc), 3)


@pytest.mark.parametrize("vth", [4.0, 30.0], ids=["most change cell", "beyond the grid"])
def test_fast_particles(vth):
    _check(make_case(n=(16, 8, 24), ppc=24, species=((-1.0, vth), (0.5, vth / 3)), dt=0.1, B=(0, 0.2, 1.0), seed=4), 3,
           flips=40)

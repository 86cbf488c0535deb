"""GPU checks of the fused field substeps on fields that vary in space: the static sources of a
non-uniform background and the gather fields formed in the last launch (the device node B with its
background, E with its background), which the particles' velocities show; and the same fields
evolving, without a static part.

The tolerance is that of the other comparisons with the FP64 oracle: three steps round each component
some 3 * 9 * 6 times in the field update and 3 * 20 times in the push, below 1e-5."""
import numpy as np
import pytest

import allscale_ipic3d_amd as G
from oracle.compare import particle_errors
from tests._helpers import gpu_sim_for, make_case, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [0, G.FLAG_UNIFORM_BACKGROUND], ids=["static part", "evolving"])
@pytest.mark.parametrize("substeps", [2, 3])
@pytest.mark.parametrize("n", [(8, 16, 8), (9, 7, 13)], ids=str)
def test_varying_fields(n, substeps, flags):
    u, sp, parts, E, Bc = make_case(n=n, ppc=12, species=((-1.0, 0.2), (0.5, 0.3)), w=(0.5, 1.0, 2.0), dt=0.1,
                                    B=(0.1, 0.2, 0.7), seed=3, field_substeps=substeps)
    rng = np.random.default_rng(4)
    E = E + rng.normal(0.0, 0.3, size=E.shape)
    Bc = Bc + rng.normal(0.0, 0.5, size=Bc.shape)
    u.set_fields(E, Bc)
    sim = gpu_sim_for((u, sp, parts, E, Bc), track_ids=False, flags=flags)
    for _ in range(3):
        u.step(1)
        sim.step(1)
    got, ref = sim.download_fields(), u.fields()
    for k in ("E", "Bc", "J"):
        assert rel_err(got[k], ref[k]) < 1e-5, k
    for e in particle_errors(u, sim, sp):
        assert e["flip_particles"] <= 2
        assert e["velocity_max"] < 1e-5 and e["offset_max"] < 1e-5, e
    sim.close()
    u.close()

"""Semi-implicit sweeps average over neighbours of mass above 1e-9 only: cells
of negative mass (a user's own mass field) are none, as in the oracle."""
import numpy as np
import pytest

import oracle as orc
from molla_amd import Implicit, MpmConfig
from tests.gpu_util import oracle_state, rel_err, run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sweeps", [1, 2, 4])
def test_cells_of_negative_mass_are_no_neighbours(sweeps):
    G, dx, dt = 32, 1.0 / 32, 1e-3
    rng = np.random.default_rng(sweeps)
    cfg = MpmConfig.sand().copy(grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx, youngs=1.5e6, gravity_y=0.0,
                                time_step=Implicit(sweeps))
    # 64 particles of positive mass reach nodes 10 to 12 of the x axis, 64 of
    # negative mass nodes 13 to 15: no cell has terms of both
    x = (dx * (12.6 + 0.8 * rng.random((128, 3)))).astype(np.float32)
    x[:64, 0] += dx * (10.55 - 12.6)
    x[64:, 0] += dx * (13.55 - 12.6)
    v = (1.0 + 0.1 * rng.standard_normal((128, 3))).astype(np.float32)
    mass = np.full(128, cfg.particle_mass, np.float32)
    mass[64:] *= -1
    sim, got = run_gpu(cfg, x, v, dt, 1, mode="global_atomic", fields={"mass": mass})
    sim.close()
    ref = oracle_state(cfg, x, v, mass=mass.astype(np.float64))
    orc.step(cfg, ref, dt, 1)
    # one transfer and the sweeps in f32: some 10 sums of 64 terms a cell
    assert rel_err(got["v"], ref.v) <= 2e-5
    assert rel_err(got["x"], ref.x) <= 1e-6

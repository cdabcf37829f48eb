"""Blocks that count themselves out (the grid clear and the last of the
semi-implicit sweeps), for fewer blocks than there are groups of counters, one
more, and more tiles than blocks: every step starts with no dynamic tile, so a
handle that has stepped other particles agrees with a fresh one."""
import numpy as np
import pytest

from molla_amd import Implicit, MpmConfig, MpmSimulation
from tests.gpu_util import log, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,G,sweeps", [(1, 16, 3), (3, 24, 1), (40, 24, 4), (400, 40, 3), (3000, 96, 3),
                                        (40000, 128, 5)])
def test_implicit_steps_with_dynamic_tiles_start_over(n, G, sweeps):
    dx = 1.0 / G
    cfg = MpmConfig.sand().copy(grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx, max_particles=n,
                                time_step=Implicit(sweeps))
    rng = np.random.default_rng(n)
    xs = [(dx * (3.0 + (G - 7.0) * rng.random((n, 3)))).astype(np.float32) for _ in range(3)]
    v = (0.1 * rng.standard_normal((n, 3))).astype(np.float32)

    def run(states):
        sim = MpmSimulation(cfg)
        sim.set_p2g_mode("global_atomic")
        for x in states:
            sim.set_particles(x, v)
            sim.step_n(1e-5, 3)
        m, _ = sim.read_grid_mass_momentum()
        tiles, vel = sim.read_status()["active_tiles"], sim.read_velocities()
        sim.close()
        return tiles, m, vel

    used, fresh = run(xs), run(xs[2:])
    log(f"{n} particles, {used[0]} tiles")
    # mass and velocity sums of float atomics, in any order
    assert used[0] == fresh[0] and rel_err(used[1], fresh[1]) <= 1e-5 and rel_err(used[2], fresh[2]) <= 1e-4

"""The grid clear between steps resets the dynamic tile list in its own launch:
a handle that has stepped other particles reports the tiles of a fresh handle,
for no tile to spare, a few blocks, and more tiles than one round of blocks
takes (four per block, 2,048 blocks).  Counts are whole numbers and equal; the
atomic mode's mass sums agree to f32 rounding in any order, 1e-5."""
import numpy as np
import pytest

from molla_amd import MpmConfig, MpmSimulation

from gpu_util import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,G", [(1, 16), (300, 32), (40000, 128)])
def test_dynamic_tiles_start_over_each_step(n, G):
    dx = 1.0 / G
    cfg = MpmConfig.sand().copy(grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx, max_particles=n)
    rng = np.random.default_rng(n)
    xs = [(dx * (3.0 + (G - 7.0) * rng.random((n, 3)))).astype(np.float32) for _ in range(3)]
    v = np.zeros((n, 3), np.float32)

    def run(states):
        sim = MpmSimulation(cfg)
        sim.set_p2g_mode("legacy")
        for k, x in enumerate(states):
            if k == 0:
                sim.set_particles(x, v)
            else:
                sim.write_field("position", x)
            sim.step_n(1e-5, 1)
        m, _ = sim.read_grid_mass_momentum()
        tiles = sim.read_status()["active_tiles"]
        sim.close()
        return tiles, m

    used, fresh = run(xs), run(xs[2:])
    assert used[0] == fresh[0] and (n < 40000 or used[0] > 4 * 2048)
    assert rel_err(used[1], fresh[1]) <= 1e-5

"""Tile marks of a chunk whose box, grown by one cell, touches more than 128
tiles: one aligned chunk over eight tiles of a row, with one particle drifting
along x and one along y, apart from all others.  The active tiles are those of
the marking rule at the scattered positions, and the particles a dense grid's."""
import numpy as np
import pytest

import oracle as orc
from molla_amd import MpmConfig, MpmSimulation, Viscous
from tests.gpu_util import log

pytestmark = pytest.mark.gpu


def test_a_chunk_that_touches_more_than_128_tiles():
    G, dx, tx, ty, tz = 96, 1.0 / 64, 8, 9, 11
    rng = np.random.default_rng(8)
    rows = np.zeros((512, 3))
    # at rest: bases 0 in y and 0 or 1 in z of the tile row, over tiles 8 to 14
    rows[:254, 0] = np.linspace(0.6, 27.4, 254)
    rows[:254, 1] = 0.7 + 0.2 * rng.random(254)
    rows[:254, 2] = np.where(np.arange(254) % 2, 0.7, 1.7)
    rows[254] = 14.6, 3.7, 0.7  # drifts along y; nodes 3 to 5: no particle at rest reaches them
    rows[255] = 31.4, 3.7, 0.7  # drifts along x, in the last tile
    rows[256:] = 0.7  # the chunk after it
    rows[256:, 0] = 28.7 + 0.2 * rng.random(256)
    x = (dx * (rows + 4.0 * np.array([tx, ty, tz]))).astype(np.float32)
    v = np.zeros_like(x)
    dt, speed = 1e-4, 0.1 * dx / 1e-4  # a tenth of a cell per substep
    v[254, 1] = v[255, 0] = speed
    cfg = MpmConfig.sand().copy(gravity_y=0.0, rheology=Viscous(0, 0), grid_size=G, cell_size=dx,
                                grid_origin=(0.0, 0.0, 0.0), max_particles=512)
    dense, sparse = MpmSimulation(cfg), MpmSimulation.new_sparse(cfg, 1024)
    for sim in (dense, sparse):
        sim.set_particles(x, v)
        sim.set_launch_config(particles_per_thread=1, segment_tiles=8, sort_every=100)
        sim.step_n(dt, 25)
    at = sparse.read_positions()  # where the last substep scatters
    # the first chunk's box, from its base cells
    base = orc.base_cells(cfg, at[:256])
    lo, hi = base.min(0), base.max(0) + 2
    tiles = (hi + 1) // 4 - (lo - 1) // 4 + 1
    log(f"box {hi - lo + 1}, {tiles} tiles")
    assert np.prod(tiles) > 128 and np.prod(hi - lo + 1) <= 1600
    for sim in (dense, sparse):
        sim.step_n(dt, 1)
        st = sim.read_status()
        assert st["sorts"] == 1 and st["escapes"] == 0 and st["fallback_chunks"] == 0 and st["fault_bits"] == 0, st
        assert st["chunks"] == 2
    assert np.array_equal(np.sort(sparse.read_active_tile_ids()), orc.marked_tiles(cfg, at))
    for name in ("position", "velocity", "F"):
        assert np.abs(dense.read_field(name) - sparse.read_field(name)).max() <= 2e-5 * max(1.0, speed), name
    dense.close()
    sparse.close()

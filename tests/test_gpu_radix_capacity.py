"""Sorts of fewer keys than a handle's capacity, at counts whose digits are
wider than the capacity's own: the order equals the oracle's after a larger
set was there before, and a step is that of a handle of just that capacity."""
import numpy as np
import pytest

import oracle as orc
from molla_amd import MpmConfig, MpmSimulation
from tests.gpu_util import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap,n,G", [(300000, 262144, 64), (262145, 262144, 64), (524289, 524288, 48),
                                     (1048577, 1048576, 40)])
def test_a_smaller_set_in_a_larger_handle(cap, n, G):
    log(f"capacity {cap}, {n} particles, grid {G}")
    dx = 1.0 / G
    cfg = MpmConfig.sand().copy(grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx, max_particles=cap)
    x = (dx * (3.0 + (G - 7.0) * np.random.default_rng(n).random((cap, 3)))).astype(np.float32)
    sim = MpmSimulation(cfg)
    sim.set_particles(x)
    sim.step_n(1e-5, 1)
    x = x[:n]
    sim.set_particles(x)
    keys, ids = sim.sort_keys_debug()
    want_k, want_i = orc.sorted_tile_keys(cfg, x)
    assert np.array_equal(keys, want_k) and np.array_equal(ids, want_i)
    ref = MpmSimulation(cfg.copy(max_particles=n))
    ref.set_particles(x)
    for s in (sim, ref):
        s.step_n(1e-5, 2)
    assert np.array_equal(sim.read_positions(), ref.read_positions())
    assert np.array_equal(sim.read_velocities(), ref.read_velocities())
    sim.close()
    ref.close()

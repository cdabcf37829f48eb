"""Material ids of every row move with their particles: written in the
original order, read back through the pinned path and past its line, from a
sorted layout and after a re-sort, on the host and on the device."""
import numpy as np
import pytest

from molla_amd import MpmConfig, MpmSimulation, Sand, Snow, Viscous
from molla_amd.devmem import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 257, 4099, 10000, 10001])
def test_material_ids_round_trip(n):
    G, dx = 32, 0.05
    rows = [Sand(), Snow(), Viscous(0.1, 0.2), Sand(0.4), Snow(0.03), Viscous(0.0, 0.0), Sand(0.7), Viscous(1.0, 2.0)]
    cfg = MpmConfig.sand().copy(grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx, max_particles=n,
                                materials=rows)
    rng = np.random.default_rng(n)
    x = (dx * (6.0 + 16.0 * rng.random((n, 3)))).astype(np.float32)
    v = (0.5 * rng.standard_normal((n, 3))).astype(np.float32)
    sim = MpmSimulation(cfg)
    sim.set_particles(x, v)
    sim.set_sort_interval(2)
    want = rng.permutation(np.arange(1, n + 1) % len(rows)).astype(np.uint32)
    for steps in (0, 3, 5):
        if steps:
            sim.step_n(1e-4, steps)
            assert np.array_equal(sim.read_field("material"), want)  # a sort moved them
            want = ((want + 1) % len(rows)).astype(np.uint32)
        sim.write_field("material", want)
        assert np.array_equal(sim.read_field("material"), want)
        with DeviceArray((n, 1), np.uint32) as d:
            sim.read_field_device("material", d.address)
            sim.synchronize()
            assert np.array_equal(d.download().ravel(), want)
    assert sim.read_status()["sorts"] > 1
    sim.close()

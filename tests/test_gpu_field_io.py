"""Field writes and reads on a sorted layout move every particle's words to
and from its own slot, for each field width and for counts around a block."""
import numpy as np
import pytest

from molla_amd import workloads
from molla_amd.devmem import DeviceArray
from molla_amd.mpm import FIELDS, MpmSimulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 257, 4099])
def test_fields_round_trip_through_a_sorted_layout(n):
    cfg, x, meta = workloads.elastic_cube(n, seed=n)
    sim = MpmSimulation(cfg)
    sim.set_particles(x)
    sim.step_n(meta["dt"], 3)  # the slots are in tile order now
    rng = np.random.default_rng(n)
    for name, (_, width) in FIELDS.items():
        want = rng.integers(0, 1, n).astype(np.uint32) if name == "material" else \
            (1.0 + 0.01 * rng.random((n, width))).astype(np.float32)
        sim.write_field(name, want)
        got = sim.read_field(name)
        assert np.array_equal(got.reshape(n, -1), want.reshape(n, -1)), name
        with DeviceArray((n, width), want.dtype) as d:
            sim.read_field_device(name, d.address)
            sim.synchronize()
            assert np.array_equal(d.download().reshape(n, -1), want.reshape(n, -1)), name
    sim.close()

"""Reads and rigid-body poses through the pinned mailbox, around its largest
particle count: every field comes back as written, interleaved with reads of
other widths, and a pose uploaded right after a read is the one stepped with."""
import numpy as np
import pytest

from molla_amd import MpmConfig, MpmSimulation
from molla_amd.mpm import FIELDS
from molla_amd.rigid import MpmPrescribedSolid, SolidSphere

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [9999, 10000, 10001])
def test_reads_and_poses_around_the_mailbox_line(n):
    G, dx = 32, 0.05
    cfg = MpmConfig.sand().copy(grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx, max_particles=n, max_rigid=2)
    rng = np.random.default_rng(n)
    x = (dx * (6.0 + 16.0 * rng.random((n, 3)))).astype(np.float32)

    def pose(k):
        return [MpmPrescribedSolid(SolidSphere(0.15), center=(0.6 + 0.05 * k, 0.7, 0.7), orientation=(0, 0, 0, 1.0),
                                   linear_velocity=(0.0, -1.0, 0.0), angular_velocity=(0.0, 0.0, 0.0))]

    def run(read):
        sim = MpmSimulation(cfg)
        sim.set_particles(x, np.zeros_like(x))
        sim.set_p2g_mode("fused")
        out = []
        for k in range(3):
            sim.set_prescribed_solids(pose(k))
            if read:
                assert sim.read_rigid_wrenches() == [((0.0,) * 3, (0.0,) * 3)]
            sim.step_n(1e-5, 2)
            if read or k == 2:
                out = [sim.read_field("F"), sim.read_positions(), np.array(sim.read_rigid_wrenches())]
        sim.close()
        return out

    for a, b in zip(run(True), run(False)):
        assert np.abs(np.asarray(b)).max() > 0
        if a.size > 6:  # the wrench is a sum of atomics
            assert np.array_equal(a, b)
        else:
            assert np.allclose(a, b, rtol=1e-6, atol=1e-6 * np.abs(b).max())

    sim = MpmSimulation(cfg)
    sim.set_particles(x, np.zeros_like(x))
    sim.step_n(1e-5, 2)
    want = {}
    for name, (_, width) in FIELDS.items():
        want[name] = np.zeros(n, np.uint32) if name == "material" else (1 + 0.01 * rng.random((n, width))).astype(np.float32)
        sim.write_field(name, want[name])
    for name in list(FIELDS) + list(reversed(FIELDS)):
        assert np.array_equal(sim.read_field(name).reshape(n, -1), want[name].reshape(n, -1)), name
    sim.close()

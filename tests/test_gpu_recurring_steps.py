"""Frames that a program repeats become graph replays of mpm_step_n: 160 calls,
with reads, writes, setters and other steps between them, leave the bits of a
handle whose stages are profiled, which keeps every launch eager."""
import numpy as np
import pytest

from molla_amd import MpmSimulation, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,substeps", [(1000, 8), (8192, 20), (8192, 7), (20000, 16)])
def test_replayed_frames_equal_eager_frames(n, substeps):
    cfg, x, meta = workloads.elastic_cube(n, seed=n)
    dt = 0.5 * meta["dt"]

    def run(eager):
        sim = MpmSimulation(cfg)
        sim.set_particles(x)
        sim.set_profiling(eager)
        out = []
        for k in range(160):
            sim.step_n(dt, substeps)
            if k % 40 == 39:
                out += [sim.read_field(f) for f in ("position", "velocity", "F", "C")]
                st = sim.read_status()
                out.append(np.array([st["completed_gathers"], st["sorts"], st["fault_bits"]]))
            if k == 100:  # another velocity field, and graphs dropped by a setter
                sim.write_field("velocity", 0.5 * sim.read_velocities())
                sim.set_materials(cfg.materials if cfg.materials else [cfg.rheology])
            if k == 130:
                sim.step_n(0.5 * dt, substeps)
                sim.step_n_graph(dt, substeps)
        sim.close()
        return out

    a, b = run(False), run(True)
    assert b[4][2] == 0
    for i, (p, q) in enumerate(zip(a, b)):
        assert np.array_equal(p, q), i

"""Semi-implicit sweeps one to a launch (grids of thousands of active tiles)
leave the bits of three to a launch, with legacy spheres and without, and
match the FP64 oracle."""
import numpy as np
import pytest

from molla_amd import Implicit, MpmConfig, MpmSimulation, Viscous
from tests.gpu_util import log
from tests.test_gpu_parity import _assert_errs, _compare_with_oracle

pytestmark = pytest.mark.gpu


def _scene(n, G, lo, hi, sweeps, seed):
    dx = 1.0 / 32
    rng = np.random.default_rng(seed)
    x = (dx * (lo + (hi - lo) * rng.random((n, 3)))).astype(np.float32)
    v = (0.3 * rng.standard_normal((n, 3))).astype(np.float32)
    cfg = MpmConfig.sand().copy(grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx, max_particles=n, youngs=1e5,
                                particle_mass=1e-3, particle_volume=1e-6, time_step=Implicit(sweeps), max_rigid=64)
    return cfg, x, v


@pytest.mark.parametrize("sweeps", [1, 2, 3, 4, 5, 7])
def test_a_scene_beside_a_wide_one_keeps_its_bits(sweeps):
    a, wide = _scene(3000, 32, 6.0, 24.0, sweeps, 1), _scene(20000, 96, 4.0, 90.0, sweeps, 2)
    out = []
    for scenes in ([a], [a, wide]):
        sim = MpmSimulation([s[0] for s in scenes])
        sim.set_particles_batch([s[1] for s in scenes], [s[2] for s in scenes])
        for _ in range(3):
            sim.step_n(5e-4, 6)
        st = sim.read_status()
        log(f"{len(scenes)} scenes: {st}")
        assert st["fault_bits"] == 0 and st["escapes"] == 0
        out.append([sim.read_field(f)[:3000] for f in ("position", "velocity", "C", "F")])
        sim.close()
    for p, q in zip(*out):
        assert np.array_equal(p, q)


@pytest.mark.parametrize("sweeps,spheres", [(1, 1), (3, 7), (5, 64)])
def test_spheres_stamp_the_same_cells_either_way(sweeps, spheres):
    # the first steps on the larger grid know of no sort and go one sweep per
    # launch; the particles are far from the walls of both
    rng = np.random.default_rng(spheres)
    bodies = [(tuple(0.25 + 0.5 * rng.random(3)), 0.02 + 0.05 * rng.random(), tuple(rng.standard_normal(3)))
              for _ in range(spheres)]
    out = []
    for G in (32, 72):
        cfg, x, v = _scene(4000, G, 8.0, 22.0, sweeps, 3)
        sim = MpmSimulation(cfg)
        sim.set_particles(x, v)
        sim.set_rigid_spheres(bodies)
        sim.step_n(1e-4, 4)
        st = sim.read_status()
        assert st["fault_bits"] == 0 and st["escapes"] == 0
        out.append([sim.read_field(f) for f in ("position", "velocity", "C", "F")])
        sim.close()
    assert np.abs(out[0][1] - v).max() > 0.1
    for p, q in zip(*out):
        assert np.array_equal(p, q)


@pytest.mark.parametrize("sweeps", [2, 3])
def test_thin_scenes_match_the_oracle(sweeps):
    cfg, x, v = _scene(3000, 80, 4.0, 75.0, sweeps, 4)
    errs = _compare_with_oracle(cfg.copy(rheology=Viscous(0, 0)), x, 1e-3, 6, v=v, mode="deterministic",
                                tag=f"thin implicit{sweeps}")
    _assert_errs(errs, {"x": 1e-6, "v": 1e-5, "F": 1e-5, "C": 1e-3})

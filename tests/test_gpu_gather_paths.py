"""The ordered gather's two ways to sum a tile of a thin scene, by its own wave
(up to 32 records, up to 512 candidates) and by the whole block, leave the same
bits: a particle of no mass and no volume adds nothing but moves its tiles
across the line.  So do a thin scene and a dense one, and grids of more tiles
than a launch has blocks match the oracle."""
import numpy as np
import pytest

from molla_amd import MpmConfig, MpmSimulation, Viscous
from tests.gpu_util import log
from tests.test_gpu_parity import _assert_errs, _compare_with_oracle

pytestmark = pytest.mark.gpu


def _grid(cfg, x, v, mass, vol):
    sim = MpmSimulation(cfg, max_particles=len(x))
    sim.set_particles(x, v)
    sim.write_field("mass", mass)
    sim.write_field("volume", vol)
    sim.set_p2g_mode("deterministic")
    sim.step_n(1e-4, 1)
    m, p = sim.read_grid_mass_momentum()
    sim.close()
    return m, p


def _tile(near, far):
    """`near` particles whose stencils reach tile (4, 4, 4) of a 64^3 grid, and
    `far` candidates in the tiles beside it that do not."""
    rng = np.random.default_rng(near + far)
    x = np.concatenate([16.6 + 2.8 * rng.random((near, 3)), 16.6 + 2.8 * rng.random((far, 3))])
    x[near:, 0] = 21.6 + 1.8 * rng.random(far)  # nodes from 21 on: two cells beyond it
    return x, rng.standard_normal(x.shape), 1e-3 * (1.0 + rng.random(len(x)))


def _scattered(n):
    rng = np.random.default_rng(n)
    x = 32.0 + 28.0 * rng.random((n, 3))  # three tiles away and more
    return x, rng.standard_normal(x.shape), 1e-3 * (1.0 + rng.random(n))


def _cfg(n):
    return MpmConfig.sand().copy(gravity_y=0.0, grid_origin=(0.0, 0.0, 0.0), grid_size=64, cell_size=1.0 / 64,
                                 max_particles=n)


def _run(parts, massless):
    x, v, m = (np.concatenate(q) for q in zip(*parts))
    cfg = _cfg(len(x) + massless)
    y = np.concatenate([x, np.full((massless, 3), 18.2)]) / 64.0
    vol = np.concatenate([np.full(len(x), cfg.particle_volume), np.zeros(massless)])
    f = np.float32
    return _grid(cfg, y.astype(f), np.concatenate([v, np.zeros((massless, 3))]).astype(f),
                 np.concatenate([m, np.zeros(massless)]).astype(f), vol.astype(f))


@pytest.mark.parametrize("near,far", [(1, 0), (16, 0), (17, 0), (31, 0), (32, 0), (33, 0), (32, 470), (32, 480),
                                      (20, 492), (5, 600)])
def test_both_ways_leave_the_same_bits(near, far):
    parts = [_tile(near, far), _scattered(600)]  # more than 600 active tiles, and few particles for them
    want = _run(parts, 0)
    assert want[0].max() > 0
    for extra in (1, 2, 40, 600):
        got = _run(parts, extra)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), extra
    # without the scattered ones the scene has few tiles and each takes a block
    alone = _run(parts[:1], 0)
    box = np.zeros((64, 64, 64), bool)
    box[:28, :28, :28] = True  # z, y, x: the cells of the tile and its neighbours
    box = box.ravel()
    assert np.array_equal(alone[0][box], want[0][box]) and np.array_equal(alone[1][box], want[1][box])


def test_many_thin_tiles_match_the_oracle():
    # 20^3 tiles, most of them on the active list, a few thick ones among them
    G, n = 80, 3000
    dx = 1.0 / G
    rng = np.random.default_rng(5)
    x = 4.0 + (G - 9.0) * rng.random((n, 3))
    x[:700] = 40.3 + 3.0 * rng.random((700, 3))
    x = (dx * x).astype(np.float32)
    v = (0.3 * rng.standard_normal((n, 3))).astype(np.float32)
    cfg = MpmConfig.sand().copy(rheology=Viscous(0, 0), grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx)
    errs = _compare_with_oracle(cfg, x, 1e-4, 4, v=v, mode="deterministic", tag="thin tiles")
    log(f"thin tiles: {errs}")
    _assert_errs(errs, {"x": 1e-6, "v": 1e-5, "F": 1e-5, "C": 1e-3})

"""The ordered gather's two ways to sum a tile, by its own wave (up to 32
records, up to 512 candidates) and by the whole block, leave the same bits: a
particle of no mass and no volume adds nothing but moves its tiles across the
line; grids of more tiles than a launch has blocks match the oracle."""
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


@pytest.mark.parametrize("near,far", [(1, 0), (31, 0), (32, 0), (33, 0), (32, 470), (32, 480), (20, 492), (5, 600)])
def test_both_ways_leave_the_same_bits(near, far):
    # `near` particles whose stencils reach the tile, `far` candidates in the
    # tiles beside it that do not; then one more of each without mass
    G, dx = 32, 1.0 / 32
    rng = np.random.default_rng(near + far)
    cfg = MpmConfig.sand().copy(gravity_y=0.0, grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx)
    a = 16.6 + 2.8 * rng.random((near, 3))  # in tile (4, 4, 4)
    b = 16.6 + 2.8 * rng.random((far, 3))
    b[:, 0] = 21.6 + 1.8 * rng.random(far)  # nodes from 21 on: two cells beyond it
    x = (dx * np.concatenate([a, b])).astype(np.float32)
    v = rng.standard_normal(x.shape).astype(np.float32)
    mass = (1e-3 * (1.0 + rng.random(len(x)))).astype(np.float32)
    vol = np.full(len(x), cfg.particle_volume, np.float32)
    want = _grid(cfg, x, v, mass, vol)
    assert want[0].max() > 0
    for extra in (1, 2, 40, 600):  # near the tile's middle
        y = np.concatenate([x, np.tile(np.float32(dx * 18.2), (extra, 3))])
        got = _grid(cfg, y, np.concatenate([v, np.zeros((extra, 3), np.float32)]),
                    np.concatenate([mass, np.zeros(extra, np.float32)]),
                    np.concatenate([vol, np.zeros(extra, np.float32)]))
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), extra


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

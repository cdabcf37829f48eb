"""The deterministic gather-order P2G at the edges of its kernel: a tile whose
particles outgrow the block's slot list (more than 4,096 stencils on one
tile), a list that ends inside a record batch, one particle, a ragged grid
edge, and a moved grid window.  Mass and momentum are compared with the FP64
P2G at four times the error of the oracle's f32 sum in the same order (or one
part in 1e6), and two runs agree bit for bit."""
import numpy as np
import pytest

import oracle as orc
from molla_amd import MpmConfig, MpmSimulation, Viscous
from tests.gpu_util import log, oracle_state, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,G,lo,hi,window", [
    (1, 16, 6.2, 6.3, 0),
    (5003, 16, 7.0, 9.0, 0),      # more stencils on a tile than the slot list holds
    (257, 16, 6.0, 7.5, 0),       # half a batch and one record
    (513, 16, 7.0, 8.9, 0),       # one record more than a batch
    (3001, 19, 2.6, 15.9, 0),     # ragged grid: the last tile has three cells
    (2048, 18, 4.0, 13.0, 5),     # window: grid indices start at cell 5
])
def test_gather_matches_fp64_and_repeats(n, G, lo, hi, window):
    dx = 1.0 / 16
    cfg = MpmConfig.sand().copy(youngs=2.0e4, rheology=Viscous(0, 0), grid_origin=(0.0, 0.0, 0.0), grid_size=G,
                                cell_size=dx, max_particles=n, grid_window_cells=(window,) * 3)
    rng = np.random.default_rng(n)
    x = (dx * (window + lo + (hi - lo) * rng.random((n, 3)))).astype(np.float32)
    v = rng.standard_normal((n, 3)).astype(np.float32)
    F = (np.eye(3) + 0.05 * rng.standard_normal((n, 3, 3))).astype(np.float32)
    C = (0.5 * rng.standard_normal((n, 3, 3))).astype(np.float32)
    out = []
    for _ in range(2):
        sim = MpmSimulation(cfg)
        sim.set_particles(x, v)
        sim.write_field("F", F)
        sim.write_field("C", C)
        sim.set_p2g_mode("deterministic")
        sim.step_n(1e-4, 1)
        out.append(sim.read_grid_mass_momentum())
        sim.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    st = oracle_state(cfg, x, v, F=F)
    st.C[:] = C
    gm, gp = orc.p2g(cfg, st, 1e-4)
    s32 = oracle_state(cfg, x, v, F=F, dtype=np.float32)
    s32.C[:] = C
    m32, p32 = orc.p2g_gather_f32(cfg, s32, 1e-4)
    (m, p), em32, ep32 = out[0], rel_err(m32, gm), rel_err(p32, gp)
    em, ep = rel_err(m, gm), rel_err(p, gp)
    log(f"n={n} G={G}: mass {em:.2e} momentum {ep:.2e} (f32 in the same order {em32:.2e} {ep32:.2e})")
    assert em <= max(4 * em32, 1e-6) and ep <= max(4 * ep32, 1e-6)

"""The reverse pass's gathers at the edges of their staged boxes: stencils that
hang over the low and the high border of the grid, a last chunk of one
particle, and a sheared body whose chunks outgrow the box so that its gathers
read global memory.  Against the FP64 oracle at the bound of the adjoint's
other parity cases, 1e-4 of the largest gradient entry."""
import numpy as np
import pytest

from molla_amd import workloads
from test_gpu_adjoint import _gpu_run, _oracle_run, _perturbed

from gpu_util import log, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,lo,hi,shear", [
    (257, (0.1, 4.0, 0.1), (3.9, 6.0, 2.2), 0.0),        # over the low border
    (1025, (10.0, 5.0, 11.0), (15.9, 9.0, 15.9), 0.0),   # over the high border
    (200, (1.0, 8.1, 8.1), (15.0, 11.9, 11.9), 0.4),     # one chunk, sheared to more than 1,600 cells
])
def test_gathers_at_box_edges_match_fp64(n, lo, hi, shear):
    G, dt, steps = 16, 1e-3, 12
    cfg, d, _ = workloads.diff_scene(n, seed=n, grid=G)
    rng = np.random.default_rng(n)
    lo, hi = np.array(lo), np.array(hi)
    d = dict(d)
    cells = lo + (hi - lo) * rng.random((n, 3))
    d["x"] = (np.array(cfg.grid_origin) + cfg.cell_size * cells).astype(np.float32)
    d["v"] = np.zeros((n, 3), np.float32)
    d["v"][:, 1:] = (shear / (dt * steps) * cfg.cell_size * (cells[:, :1] - 8.0)).astype(np.float32)
    d["E"] = d["E"][:1].repeat(n)
    d = _perturbed(d, n + 1)
    gx = rng.standard_normal((n, 3)).astype(np.float32)
    gv = (0.1 * rng.standard_normal((n, 3))).astype(np.float32)
    g = _gpu_run(cfg, d, dt, steps, 5, gx, gv)
    o = _oracle_run(cfg, d, dt, steps, gx, gv)
    g["x"], o["x"] = g["x"] - gx, o["x"] - gx
    errs = {k: rel_err(g[k], o[k]) for k in ("x", "v", "C", "F", "E")}
    log(f"n={n} {g['status']['escapes']} escapes: " + ", ".join(f"{k} {e:.1e}" for k, e in errs.items()))
    assert max(errs.values()) < 1e-4

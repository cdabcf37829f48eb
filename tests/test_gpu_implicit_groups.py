"""Sweep counts that need more than one launch (three sweeps each), on a grid
whose last tiles are ragged, against the FP64 oracle at f32-oracle level (the
deterministic P2G: the fused one's fixed-point momenta add their own error in
cells of tiny mass)."""
import numpy as np
import pytest

from molla_amd import Implicit, MpmConfig, Viscous
from tests.fixtures import fill_box
from tests.test_gpu_parity import _assert_errs, _compare_with_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iters", [4, 5, 6, 7])
def test_sweep_groups_match_fp64_oracle(iters):
    cfg = MpmConfig.sand_calibrated().copy(time_step=Implicit(iters), rheology=Viscous(0, 0), grid_size=46)
    x = fill_box([-1.05, 0.15, -1.05], [-0.65, 0.45, -0.65], 9, 41 + iters)  # by the floor and two walls
    v = np.tile(np.array([-0.4, -0.3, -0.2], np.float32), (len(x), 1))
    errs = _compare_with_oracle(cfg, x, 1e-3, 12, v=v, mode="deterministic", tag=f"implicit{iters}")
    _assert_errs(errs, {"x": 1e-6, "v": 1e-5, "F": 1e-5, "C": 1e-3})

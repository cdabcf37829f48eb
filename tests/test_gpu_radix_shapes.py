"""The radix sort's shapes against the oracle's stable order, whole numbers and
so equal: one and two passes, eight waves a block (digits of up to 10 bits) and
four (wider), counts around a block of 4,096 keys, and block counts on both
sides of the 512 whose rows stay in registers."""
import numpy as np
import pytest

import oracle as orc
from molla_amd import MpmConfig, MpmSimulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,G", [(1, 16), (4095, 40), (4097, 44), (4096, 64), (20001, 128), (262145, 160),
                                 (524289, 250), (2097152, 100), (2097153, 100)])
def test_key_order_equals_the_oracle(n, G):
    dx = 1.0 / G
    cfg = MpmConfig.sand().copy(grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx, max_particles=n)
    rng = np.random.default_rng(n)
    x = (dx * (3.0 + (G - 7.0) * rng.random((n, 3)))).astype(np.float32)
    x[: n // 3] = x[0]  # a long run of one key
    sim = MpmSimulation(cfg)
    sim.set_particles(x)
    keys, ids = sim.sort_keys_debug()
    want_k, want_i = orc.sorted_tile_keys(cfg, x)
    assert np.array_equal(keys, want_k) and np.array_equal(ids, want_i)
    sim.close()

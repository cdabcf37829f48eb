"""The sorted layout's shapes at the lines between them: one block for keys,
sort and lists (up to 16,384 particles and 8,192 tiles), one block for the
lists, a launch per step; one and two radix passes; scenes without particles.
The key query equals the oracle's keys and order bit for bit, the chunk list
has the modelled count, and stepping on it agrees with the unsorted
global-atomic mode to f32 rounding."""
import numpy as np
import pytest

import oracle as orc
from molla_amd import MpmConfig, MpmSimulation, Viscous
from tests.gpu_util import log, rel_err
from tests.test_gpu_parity import _model_chunk_count

pytestmark = pytest.mark.gpu


def _scene(n, G, seed):
    rng = np.random.default_rng(seed)
    cfg = MpmConfig.sand().copy(rheology=Viscous(0, 0), youngs=2.0e3, grid_size=G, cell_size=1.0 / G,
                                grid_origin=(0.0, 0.0, 0.0), max_particles=max(n, 1))
    cfg = cfg.copy(particle_volume=(0.6 ** 3) / max(n, 1), particle_mass=1000.0 * (0.6 ** 3) / max(n, 1))
    return cfg, (0.2 + 0.6 * rng.random((n, 3))).astype(np.float32)


def _chunks(scenes, cap, seg):
    total = 0
    for cfg, x in scenes:
        if len(x):
            W = (cfg.grid_size + 3) // 4
            keys, _ = orc.tile_keys(cfg, x)
            total += _model_chunk_count(np.bincount(keys.astype(np.int64), minlength=W ** 3), W, cap, seg)
    return total


@pytest.mark.parametrize("sizes", [[(16384, 32)], [(16385, 32)], [(5001, 80)], [(5001, 84)], [(70001, 64)],
                                   [(70001, 131)], [(0, 32), (300, 33), (0, 48), (2000, 64), (0, 32)],
                                   [(0, 32), (30000, 64), (17, 40)]],
                         ids=lambda s: "-".join(f"{n}@{g}" for n, g in s))
def test_layout_shapes(sizes):
    scenes = [_scene(n, g, 7 + i) for i, (n, g) in enumerate(sizes)]

    def sim():
        s = MpmSimulation([c for c, _ in scenes])
        if len(scenes) > 1:
            s.set_particles_batch([x for _, x in scenes])
        else:
            s.set_particles(scenes[0][1])
        return s

    ref = sim()
    for i, (cfg, x) in enumerate(scenes):
        if len(x):
            keys, ids = ref.sort_keys_debug(scene=i)
            okeys, oids = orc.sorted_tile_keys(cfg, x)
            assert np.array_equal(keys, okeys) and np.array_equal(ids, oids)
    ref.set_p2g_mode("global_atomic")
    ref.step_n(1e-5, 3)
    want = ref.read_positions(), ref.read_velocities()
    ref.close()
    for seg in (6, 8):
        s = sim()
        s.set_launch_config(particles_per_thread=2, segment_tiles=seg)
        s.step_n(1e-5, 3)
        st = s.read_status()
        assert st["chunks"] == _chunks(scenes, 512, seg) and st["fault_bits"] == 0
        e = rel_err(s.read_positions(), want[0]), rel_err(s.read_velocities(), want[1])
        log(f"{sizes} segment_tiles {seg}: {st['chunks']} chunks, x {e[0]:.1e} v {e[1]:.1e}")
        assert e[0] <= 1e-6 and e[1] <= 2e-5
        s.close()


@pytest.mark.parametrize("n,G,cap", [(8192, 32, 256), (131072, 64, 256), (131073, 64, 512)])
def test_default_chunk_size_follows_the_particle_count(n, G, cap):
    # one particle per thread up to 131,072 particles, two beyond; a
    # configuration that is set holds, and takes effect at the next step
    scene = _scene(n, G, 3)
    s = MpmSimulation(scene[0])
    s.set_particles(scene[1])
    s.step_n(1e-5, 1)
    assert s.read_status()["chunks"] == _chunks([scene], cap, 6)
    s.set_launch_config(particles_per_thread=2)
    s.step_n(1e-5, 1)
    st = s.read_status()
    x = s.read_positions()
    s.close()
    assert abs(st["chunks"] - _chunks([scene], 512, 6)) <= 2  # the particles have moved a little
    t = MpmSimulation(scene[0])
    t.set_particles(scene[1])
    t.set_launch_config(particles_per_thread=2)
    t.step_n(1e-5, 2)
    assert rel_err(x, t.read_positions()) <= 1e-6
    t.close()

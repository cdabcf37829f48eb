"""Particles per thread that a handle chooses by itself: reads back as chosen,
survives a change of any other launch setting and a round trip of the whole
configuration, follows the particle count; a value that is given holds, also
before the particles are there."""
import ctypes as C

import numpy as np
import pytest

from molla_amd import MpmConfig, MpmError, MpmSimulation
from molla_amd.mpm import LaunchConfig, lib

pytestmark = pytest.mark.gpu
G, CAP = 64, 140000


def _handle():
    dx = 1.0 / G
    cfg = MpmConfig.sand().copy(grid_origin=(0.0, 0.0, 0.0), grid_size=G, cell_size=dx, max_particles=CAP)
    x = (dx * (3.0 + 16.0 * np.random.default_rng(1).random((CAP, 3)))).astype(np.float32)
    return MpmSimulation(cfg), x


def _chunks(sim):
    sim.step_n(1e-6, 1)
    return sim.read_status()["chunks"]


def test_the_choice_outlives_other_settings_and_round_trips():
    sim, x = _handle()
    assert sim.launch_config()["particles_per_thread"] == 2  # no particles yet
    sim.set_launch_config(grid_blocks=2048)
    sim.set_particles(x[:20000])
    one = _chunks(sim)
    assert sim.launch_config()["particles_per_thread"] == 1
    sim.set_launch_config(sort_every=32)
    cfg = LaunchConfig()
    assert lib().mpm_get_launch_config(sim._h, C.byref(cfg)) == 0
    assert lib().mpm_set_launch_config(sim._h, C.byref(cfg)) == 0
    assert cfg.as_dict() == sim.launch_config() == {"particle_blocks": 0, "grid_blocks": 2048, "sort_every": 32,
                                                    "particles_per_thread": 1, "segment_tiles": 6}
    assert _chunks(sim) == one and sim.read_status()["sorts"] == 1  # the layout stayed
    sim.set_launch_config(particles_per_thread=2)
    two = _chunks(sim)
    assert two < one and sim.launch_config()["particles_per_thread"] == 2
    # a set above the line: two by its own choice
    sim.set_particles(x)
    given = _chunks(sim)
    sim.close()
    sim, _ = _handle()
    sim.set_particles(x[:20000])
    sim.set_launch_config(sort_every=32)
    sim.set_particles(x)
    assert _chunks(sim) == given and sim.launch_config()["particles_per_thread"] == 2
    sim.close()


@pytest.mark.parametrize("given", [1, 2])
def test_a_given_value_holds_for_later_particles(given):
    counts = {}
    for when in ("before", "small", "after"):
        sim, x = _handle()
        if when == "before":
            sim.set_launch_config(particles_per_thread=given)
        sim.set_particles(x[:20000])
        if when == "small":
            sim.set_launch_config(particles_per_thread=given)
        sim.set_particles(x)
        if when == "after":
            sim.set_launch_config(particles_per_thread=given)
        assert sim.launch_config()["particles_per_thread"] == given
        large = _chunks(sim)
        sim.set_particles(x[:20000])
        counts[when] = large, _chunks(sim)
        assert sim.launch_config()["particles_per_thread"] == given
        assert lib().mpm_set_particles_per_thread(sim._h, 0) == 0  # the handle's choice again
        assert sim.launch_config()["particles_per_thread"] == 1
        assert lib().mpm_set_particles_per_thread(sim._h, 3) != 0
        with pytest.raises(MpmError):
            sim.set_launch_config(particles_per_thread=0)
        sim.close()
    assert len(set(counts.values())) == 1, counts

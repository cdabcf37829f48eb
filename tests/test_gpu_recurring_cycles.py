"""Repeated calls whose state comes back only after a long cycle (long sort
intervals) and semi-implicit ones are replayed, and leave the bits of a handle
whose stages are profiled, which keeps every launch eager."""
import numpy as np
import pytest

from molla_amd import Implicit, MpmSimulation, workloads
from tests.gpu_util import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("interval,substeps,calls,sweeps,least", [(128, 17, 3000, 0, 250), (64, 10, 900, 0, 250),
                                                                  (16, 8, 60, 3, 30), (16, 9, 300, 4, 100)])
def test_long_cycles_and_implicit_steps_replay_the_same_bits(interval, substeps, calls, sweeps, least):
    cfg, x, meta = workloads.elastic_cube(1500, seed=interval)
    if sweeps:
        cfg = cfg.copy(time_step=Implicit(sweeps))
    dt = 0.02 * meta["dt"]

    def run(eager):
        sim = MpmSimulation(cfg)
        sim.set_particles(x, np.tile(np.float32([0.3, -0.2, 0.1]), (len(x), 1)))
        sim.set_sort_interval(interval)
        sim.set_profiling(eager)
        for _ in range(calls):
            sim.step_n(dt, substeps)
        st, got = sim.read_status(), sim.graph_stats()
        out = [sim.read_field(f) for f in ("position", "velocity", "F", "C")]
        sim.close()
        log(f"interval {interval}, {calls} calls of {substeps}: eager {eager}, {got}, escapes {st['escapes']}")
        assert st["fault_bits"] == 0 and st["escapes"] == 0
        return out, got, st["sorts"]

    a, got, sorts = run(False)
    b, none, want = run(True)
    assert none["captures"] == 0 and sorts == want
    assert got["replays"] >= least and got["captures"] <= 64
    for p, q in zip(a, b):
        assert np.array_equal(p, q)


def test_captures_that_are_not_replayed_end():
    # particles loaded anew every 24 frames drop the graphs after a replay or none
    cfg, x, meta = workloads.elastic_cube(1000, seed=3)
    sim = MpmSimulation(cfg)
    for _ in range(120):
        sim.set_particles(x)
        for _ in range(24):
            sim.step_n(0.02 * meta["dt"], 8)
    got = sim.graph_stats()
    log(f"short episodes: {got}")
    assert 0 < got["captures"] <= 64 + got["replays"] // 16
    sim.close()

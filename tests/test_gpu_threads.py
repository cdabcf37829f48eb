"""Handles of several host threads at once: repeated small frames that become
graph replays, reads through the pinned mailbox, new particles and setters in
one thread while another captures.  Each leaves the bits of a run alone."""
import threading

import numpy as np
import pytest

from molla_amd import Implicit, MpmSimulation, workloads

pytestmark = pytest.mark.gpu


def _program(k):
    cfg, x, meta = workloads.elastic_cube(600 + 900 * k, seed=k)
    if k % 2:
        cfg = cfg.copy(time_step=Implicit(3))
    out = []
    for episode in range(3):
        sim = MpmSimulation(cfg)
        sim.set_particles(x)
        for frame in range(60):
            sim.step_n(0.2 * meta["dt"], 8 + k)
            if frame % 7 == k:
                sim.read_positions()
            if frame == 30 and k == 2:
                sim.set_materials([cfg.rheology])
        out += [sim.read_field(f) for f in ("position", "velocity", "F")]
        sim.close()
    return out


def test_threads_with_a_handle_each_leave_the_bits_of_one_alone():
    alone = [_program(k) for k in range(4)]
    got, errors = [None] * 4, []

    def work(k):
        try:
            got[k] = _program(k)
        except Exception as e:  # noqa: BLE001
            errors.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    assert not errors and not any(t.is_alive() for t in threads), errors
    for a, b in zip(alone, got):
        for p, q in zip(a, b):
            assert np.array_equal(p, q)

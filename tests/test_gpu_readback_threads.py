"""Contexts of several threads whose results go through the process's pinned slots at the same time, among them ones that
come and go (-m gpu)."""
import threading

import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes

pytestmark = pytest.mark.gpu


def test_threads_read_back_side_by_side(gpu):
    print("case: four threads with contexts of their own read back", flush=True)
    shapes = [(64, 64, 67), (5, 331, 1999), (128, 128, 130), (40, 200, 301)]
    wrong = []

    def work(k):
        try:
            shape = shapes[k]
            rng = np.random.default_rng(k)
            for turn in range(3):   # a context each turn, several results from each
                sim = capi.Simulation(capi.Grid(*shape, 1.0 / 32, 0.25 / 32), scenes.params())
                for field in (capi.FIELD_U2, capi.FIELD_V2, capi.FIELD_W2):
                    want = rng.standard_normal(sim.grid.nc, np.float32)
                    sim.set_grid(field, want)
                    for _ in range(4):
                        if not np.array_equal(sim.get_grid(field), want):
                            wrong.append((k, turn, field))
                sim.close()
        except Exception as e:   # an assertion in a thread would go unseen
            wrong.append((k, repr(e)))

    team = [threading.Thread(target=work, args=(k,)) for k in range(len(shapes))]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not wrong

"""Particles in order of their ids inside every cell, for cells of every kind of sorter: up to 16, up to 64 and more
particles, many and few in a block of cells (-m gpu)."""
import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [(1, 2, 15, 16, 17, 31, 32, 33), (63, 64, 65), (17,) * 200, (64, 130, 1, 700, 40),
                                    (5000, 129, 66)])
def test_cells_hold_ascending_ids(gpu, counts):
    print(f"case: cells of {sorted(set(counts))} particles", flush=True)
    grid = capi.Grid(8, 12, 40, 1.0 / 32, 0.25 / 32)
    rng = np.random.default_rng(len(counts))
    # cells next to each other along z, a row after the other
    cells = [(1 + k // 380, 1 + k // 38 % 10, 1 + k % 38) for k in range(len(counts))]
    pos = np.concatenate([(np.array(c) + 0.1 + 0.8 * rng.random((m, 3))) / 32 for c, m in zip(cells, counts)])
    pos = pos[rng.permutation(len(pos))].astype(np.float32)
    sim = capi.Simulation(grid, scenes.params())
    sim.set_particles(pos)
    for _ in range(2):   # from the order they came in, and sorted already
        sim.run_stage(capi.STAGE_BIN)
        ids = sim.slot_ids()
        start = sim.get_grid(capi.FIELD_CELL_START)
        count = sim.get_grid(capi.FIELD_CELL_COUNT)
        assert sorted(count[count > 0]) == sorted(counts)
        assert np.array_equal(np.sort(ids), np.arange(len(pos)))
        for c in np.nonzero(count)[0]:
            part = ids[start[c]:start[c] + count[c]]
            assert np.all(np.diff(part) > 0)
            at = (pos[part].astype(np.float64) * 32).astype(int)
            assert np.all((at[:, 0] * 12 + at[:, 1]) * 40 + at[:, 2] == c)
    sim.close()

"""The tiled P2G at every tile shape that the number of blocks selects, with rows of more than one staged chunk and
particles on faces, cell centres and quarter cells, against the one-row-per-block gather (-m gpu)."""
import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes

pytestmark = pytest.mark.gpu
DX = 1.0 / 32


# 1 x 2 tiles; 2 x 2, with a last z chunk of one cell; 4 x 2, with partial tiles along x and y
@pytest.mark.parametrize("transfer", [capi.PIC, capi.APIC])
@pytest.mark.parametrize("shape", [(9, 7, 70), (29, 22, 193), (38, 41, 321)])
def test_p2g_tile_shapes_equal_row_gather(gpu, shape, transfer):
    print(f"case: P2G tiles on {shape}, transfer {transfer}", flush=True)
    grid = capi.Grid(*shape, DX, 0.25 * DX)
    rng = np.random.default_rng(sum(shape))
    # half of the particles anywhere, a quarter on the quarter-cell lattice, a quarter crowded into a few rows of
    # cells, about 25 a cell: several chunks a row
    n = 8 * grid.nc
    low, high = np.full(3, 1.3), np.array(shape) - 1.3
    cells = rng.uniform(low, high, (n, 3))
    cells[: n // 4] = np.round(4 * cells[: n // 4]) / 4
    rows = rng.integers(2, np.array(shape[:2]) - 2, (max(1, shape[0] * shape[1] // 12), 2))
    crowd = n // 4
    cells[n // 4: n // 4 + crowd, :2] = rows[rng.integers(0, len(rows), crowd)] + rng.random((crowd, 2))
    pos = (cells * DX).astype(np.float32)
    vel = rng.standard_normal((n, 3), np.float32)
    c = 4 * rng.standard_normal((n, 9), np.float32) if transfer == capi.APIC else None
    out = {}
    for rows_only in (1, 0):
        sim = capi.Simulation(grid, scenes.params(transfer=transfer))
        sim.set_option(capi.OPT_P2G_KERNEL, rows_only)
        sim.set_particles(pos, vel, c)
        sim.run_stage(capi.STAGE_P2G, scenes.DT)
        out[rows_only] = [sim.get_grid(f) for f in (capi.FIELD_U, capi.FIELD_V, capi.FIELD_W, capi.FIELD_DENSITY,
                                                    capi.FIELD_LABEL)]
        count = sim.get_grid(capi.FIELD_CELL_COUNT).reshape(shape)
        sim.close()
    assert count.reshape(-1, shape[2])[:, :66].sum(1).max() > 2 * 560   # more than two chunks in a row
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(a, b)
    assert np.count_nonzero(out[0][3]) > 0

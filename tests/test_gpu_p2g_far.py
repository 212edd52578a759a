"""P2G with particles whose positions lie outside the grid, up to beyond the range of 32-bit cell indices: the tiles
leave out what the one-row-per-block gather leaves out (-m gpu)."""
import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes

pytestmark = pytest.mark.gpu
DX = 1.0 / 32


@pytest.mark.parametrize("transfer", [capi.PIC, capi.APIC])
@pytest.mark.parametrize("shape,two_d", [((9, 7, 12), 0), ((29, 22, 193), 0), ((9, 7, 3), 1)])
def test_p2g_particles_off_the_grid_equal_row_gather(gpu, shape, two_d, transfer):
    print(f"case: P2G with particles off the grid {shape}, transfer {transfer}", flush=True)
    grid = capi.Grid(*shape, DX, 0.25 * DX, two_d=two_d, cell_d_z=DX if two_d else 0.0)
    rng = np.random.default_rng(sum(shape))
    cells = rng.uniform(0.3, np.array(shape) - 0.3, (6 * grid.nc, 3))
    inside = len(cells)
    far = [-0.6, -1.0, -1.7, -3.0, -1e3, -2.0 ** 30, -2.0 ** 31, -1e12, -1e30, -np.inf, 1e3, 2.0 ** 30, 2.0 ** 31, 1e12,
           1e30, np.inf]
    off = rng.uniform(0.3, np.array(shape) - 0.3, (3 * len(far) * 4, 3))
    for k in range(len(off)):   # one coordinate off the grid, one after the other
        off[k, k % 3] = far[k // 3 % len(far)]
    cells = np.concatenate([cells, off])
    # the largest stay FP32 numbers
    pos = np.where(np.abs(cells) > 1e29, cells, cells * DX).astype(np.float32)
    vel = rng.standard_normal((len(pos), 3), np.float32)
    out = {}
    for rows_only in (1, 0):
        sim = capi.Simulation(grid, scenes.params(transfer=transfer))
        sim.set_option(capi.OPT_P2G_KERNEL, rows_only)
        sim.set_particles(pos, vel)
        sim.run_stage(capi.STAGE_P2G, scenes.DT)
        out[rows_only] = [sim.get_grid(f) for f in (capi.FIELD_U, capi.FIELD_V, capi.FIELD_W, capi.FIELD_DENSITY)]
        assert sim.get_grid(capi.FIELD_CELL_COUNT).sum() == inside + len(off)
        sim.close()
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(a, b, equal_nan=True)
    assert np.isfinite(out[0][3]).all() and out[0][3].any()

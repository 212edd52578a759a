"""2D sweeps with a row per lane: heights around a wave's 64 rows, widths around the groups of four, water in a part of
the width, against one launch per plane (-m gpu)."""
import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes

pytestmark = pytest.mark.gpu
DT = scenes.DT


# ny - 2: less than a group of lanes, a wave, one row more, two waves, six waves and beyond (the tiles' kernel)
@pytest.mark.parametrize("nx,ny,x0,x1", [(4, 4, 1, 3), (9, 5, 2, 7), (30, 66, 0, 30), (31, 67, 5, 6), (64, 130, 13, 50),
                                         (129, 131, 3, 128), (70, 322, 0, 70), (20, 386, 0, 20),
                                         (70, 386, 0, 70), (40, 387, 0, 40)])
def test_2d_sweeps_equal_planes(gpu, nx, ny, x0, x1):
    shape = (nx, ny, 3)
    print(f"case: 2D sweeps {shape}, water in x {x0} .. {x1 - 1}", flush=True)
    grid = capi.Grid(nx, ny, 3, 1.0 / 32, 0.25 / 32, two_d=1, cell_d_z=0.1)
    rng = np.random.default_rng(nx + ny)
    lab = np.full(shape, capi.AIR, np.uint8)
    lab[x0:x1] = capi.WATER
    lab[rng.random(shape) < 0.08] = capi.AIR
    lab[rng.random(shape) < 0.04] = capi.SOLID
    lab[0], lab[-1], lab[:, 0], lab[:, :, 0], lab[:, :, -1] = (capi.SOLID,) * 5
    lab[:, -1] = np.where(lab[:, -1] == capi.WATER, capi.AIR, lab[:, -1])
    lab[min(max(x0, 1), nx - 2), 1, 1] = capi.WATER
    vec = np.where(lab == capi.WATER, rng.standard_normal(shape), 0.0).astype(np.float32).astype(np.float64)
    faces = [rng.standard_normal(shape).astype(np.float32) for _ in range(3)]
    faces[2][:] = 0
    got = {}
    for mode in (1, 0):
        sim = capi.Simulation(grid, scenes.params(tol=1e-6))
        sim.set_option(capi.OPT_SWEEP_MODE, mode)
        sim.set_grid(capi.FIELD_LABEL, lab.reshape(-1))
        z = sim.solver_apply(capi.OP_APPLY_MIC0, DT, vec)
        for f, v in zip((capi.FIELD_U2, capi.FIELD_V2, capi.FIELD_W2), faces):
            sim.set_grid(f, v.reshape(-1))
        sim.run_stage(capi.STAGE_SOLVE, DT)
        st = sim.stats()
        got[mode] = (z, sim.get_grid(capi.FIELD_PRESSURE), st.pcg_iterations, st.residual_rel_l2)
        sim.close()
    # a WATER cell between SOLID ones has no equation: its NaN ends the solve at once, with p = 0, and how far it
    # reaches in z depends on the cells that a kernel passes over
    water = (lab == capi.WATER).reshape(-1)
    if np.isfinite(got[1][0]).all():
        assert np.array_equal(got[0][0], got[1][0]) and np.count_nonzero(got[0][0]) == np.count_nonzero(vec)
    else:
        assert got[0][2] == 0 and np.isnan(got[0][0][water]).any()
    assert np.array_equal(got[0][1], got[1][1])
    assert got[0][2:] == got[1][2:]


def test_2d_solve_without_water(gpu):
    sim = capi.Simulation(capi.Grid(20, 30, 3, 1.0 / 32, 0.25 / 32, two_d=1, cell_d_z=0.1), scenes.params())
    print("case: 2D operators without water", flush=True)
    z = sim.solver_apply(capi.OP_APPLY_MIC0, DT, np.zeros(sim.grid.nc))
    assert not z.any()
    sim.close()

"""The sweeps where the rings between their waves are used again and where the 2D kernel ends, against one launch per
plane (-m gpu)."""
import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes

pytestmark = pytest.mark.gpu
DT = scenes.DT
# of the kernels: planes in a group, groups in a +z out-ring and the groups by which the +z edge runs behind its tile
GROUP, RING_Z, BEHIND = 4, 32, 15


def _labels(shape, seed):
    """WATER with holes and SOLID cells between SOLID walls, none of it enclosed by SOLID cells."""
    rng = np.random.default_rng(seed)
    lab = np.full(shape, capi.WATER, np.uint8)
    lab[rng.random(shape) < 0.08] = capi.AIR
    lab[rng.random(shape) < 0.04] = capi.SOLID
    lab[0], lab[-1], lab[:, 0], lab[:, :, 0], lab[:, :, -1] = (capi.SOLID,) * 5
    lab[:, -1] = np.where(lab[:, -1] == capi.WATER, capi.AIR, lab[:, -1])
    lab[1, 1, 1] = lab[-2, 1, 1] = capi.WATER
    pad = np.pad(lab, 1, constant_values=capi.SOLID)
    enclosed = lab == capi.WATER
    for a in range(3):
        for s in (0, 2):
            enclosed &= pad[tuple(slice(s, s + n) if k == a else slice(1, -1) for k, n in enumerate(shape))] == capi.SOLID
    lab[enclosed] = capi.AIR
    return lab


@pytest.mark.parametrize("delay", [0, 1, 8])
def test_out_rings_used_again(gpu, delay):
    """Marches of more groups than an out-ring's slots and its head start, so that the compute waves wait for the sending
    waves, and the more so the slower these are (FSIM_OPT_WAVE_SEND_DELAY); the factor and both sweeps on three tiles along
    z and two along y."""
    shape = (200, 14, 131)
    print(f"case: out-rings used again {shape}, sending waves' delay {delay}", flush=True)
    lab = _labels(shape, 3)
    water = lab == capi.WATER
    x = np.flatnonzero(water.any(axis=(1, 2)))
    full = (x[-1] + 63) // GROUP - x[0] // GROUP + 1     # march groups of a full z-tile
    part = x[-1] // GROUP - x[0] // GROUP + 1            # of the last one, a column wide, which goes first backward
    assert full > RING_Z + BEHIND + 1 and part > RING_Z + 1
    grid = capi.Grid(*shape, 1.0 / 32, 0.25 / 32)
    vec = np.where(water, np.random.default_rng(1).standard_normal(shape), 0.0).astype(np.float32).astype(np.float64)
    out = {}
    for mode in (1, 0):
        sim = capi.Simulation(grid, scenes.params())
        sim.set_option(capi.OPT_SWEEP_MODE, mode)
        sim.set_option(capi.OPT_WAVE_SEND_DELAY, delay)
        sim.set_grid(capi.FIELD_LABEL, lab.reshape(-1))
        out[mode] = (sim.solver_apply(capi.OP_FACTOR_MIC0, DT), sim.solver_apply(capi.OP_APPLY_MIC0, DT, vec))
        sim.close()
    for a, b in zip(out[0], out[1]):
        assert np.isfinite(b).all() and np.array_equal(a, b)
        assert np.count_nonzero(b) == np.count_nonzero(water)


# six waves of rows, full and not; the widest grid whose edges fit the kernel's LDS at six waves, and one plane group more
@pytest.mark.parametrize("nx,ny", [(70, 386), (70, 324), (1915, 330), (1916, 330)])
def test_2d_sweeps_of_six_waves_equal_planes(gpu, nx, ny):
    shape = (nx, ny, 3)
    print(f"case: 2D sweeps {shape}", flush=True)
    lab = _labels(shape, nx + ny)
    water = lab == capi.WATER
    grid = capi.Grid(nx, ny, 3, 1.0 / 32, 0.25 / 32, two_d=1, cell_d_z=0.1)
    rng = np.random.default_rng(2)
    vec = np.where(water, rng.standard_normal(shape), 0.0).astype(np.float32).astype(np.float64)
    faces = [rng.standard_normal(shape).astype(np.float32) for _ in range(3)]
    got = {}
    for mode in (1, 0):
        prm = scenes.params(tol=1e-6)
        prm.max_iterations = 5
        sim = capi.Simulation(grid, prm)
        sim.set_option(capi.OPT_SWEEP_MODE, mode)
        sim.set_grid(capi.FIELD_LABEL, lab.reshape(-1))
        z = sim.solver_apply(capi.OP_APPLY_MIC0, DT, vec)
        for f, v in zip((capi.FIELD_U2, capi.FIELD_V2, capi.FIELD_W2), faces):
            sim.set_grid(f, v.reshape(-1))
        sim.run_stage(capi.STAGE_SOLVE, DT)
        got[mode] = (z, sim.get_grid(capi.FIELD_PRESSURE), sim.stats().pcg_iterations)
        sim.close()
    assert np.isfinite(got[1][0]).all() and np.count_nonzero(got[1][0]) == np.count_nonzero(water)
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1]) and np.count_nonzero(got[0][1]) == np.count_nonzero(water)
    assert got[0][2] == got[1][2] == 5

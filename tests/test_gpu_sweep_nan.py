"""Sweeps over values that are not numbers: a NaN or an infinity stays on the WATER cells that depend on it, as with one
launch per plane, across the edges of waves and tiles as well (-m gpu)."""
import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes

pytestmark = pytest.mark.gpu
DT = scenes.DT
# the float of the first has every bit set, as a boundary packet's word that has not been sent
NANS = np.array([0xFFFFFFFFFFFFFFFF, 0x7FF8000000000000, 0xFFF0000000000000, 0x7FF0000000000000], np.uint64).view(np.float64)


def _labels(shape, rng):
    lab = np.full(shape, capi.WATER, np.uint8)
    lab[rng.random(shape) < 0.1] = capi.AIR
    lab[rng.random(shape) < 0.05] = capi.SOLID
    lab[:, -1] = np.where(lab[:, -1] == capi.WATER, capi.AIR, lab[:, -1])
    return lab


def _walls(lab):
    lab[0], lab[-1], lab[:, 0], lab[:, :, 0], lab[:, :, -1] = (capi.SOLID,) * 5
    return lab


def _both(grid, lab, vec):
    got = {}
    for mode in (1, 0):
        sim = capi.Simulation(grid, scenes.params())
        sim.set_option(capi.OPT_SWEEP_MODE, mode)
        sim.set_grid(capi.FIELD_LABEL, lab.reshape(-1))
        got[mode] = sim.solver_apply(capi.OP_APPLY_MIC0, DT, vec)
        sim.close()
    return got[0], got[1]


# several tiles along y and z; two columns along x; one workgroup of three waves
@pytest.mark.parametrize("shape", [(12, 20, 140), (6, 9, 67), (4, 14, 12), (40, 140, 3)])
@pytest.mark.parametrize("what", ["enclosed", "off water", "on water"])
def test_sweeps_keep_what_is_not_a_number_in_place(gpu, shape, what):
    print(f"case: sweeps {shape}, not a number {what}", flush=True)
    two_d = shape[2] == 3
    grid = capi.Grid(*shape, 1.0 / 32, 0.25 / 32, two_d=int(two_d), cell_d_z=0.1 if two_d else 0.0)
    rng = np.random.default_rng(sum(shape))
    lab = _labels(shape, rng)
    vec = rng.standard_normal(shape).astype(np.float32).astype(np.float64)
    x, z = shape[0] // 2, 1 if two_d else min(64, shape[2] - 3)
    if what == "enclosed":
        # a WATER cell between SOLID ones (its diagonal is 0, its factor infinite), AIR and WATER behind them
        lab[x - 1:x + 2, 3:6, z - 1:z + 2] = capi.SOLID
        lab[x, 4, z] = capi.WATER
        lab[x, 6] = capi.AIR
    _walls(lab)
    water = lab == capi.WATER
    if what == "off water":
        off = np.flatnonzero(~water)
        vec.reshape(-1)[off] = NANS[rng.integers(0, len(NANS), len(off))]
    if what == "on water":
        # on a tile's last row and lane, and on the row before a wave's end
        for k, v in enumerate(NANS):
            at = np.argwhere(water[:, min(6, shape[1] - 3) + (k & 1):, z - (k >> 1 & 1 & (z > 1)):])
            x1, y1, z1 = at[len(at) * k // len(NANS)]
            vec[x1, min(6, shape[1] - 3) + (k & 1) + y1, z - (k >> 1 & 1 & (z > 1)) + z1] = v
        vec[:, 6 if shape[1] > 8 else 3, z] = NANS[0]
    wave, plane = _both(grid, lab, vec)
    assert np.array_equal(wave, plane, equal_nan=True)
    assert not plane.reshape(shape)[~water].any()
    good = np.isfinite(plane.reshape(shape)[water])
    # (a WATER cell between SOLID ones can come from the random labels as well)
    enclosed = water[1:-1, 1:-1, 1:-1].copy()
    for a in range(3):
        for s in (0, 2):
            enclosed &= lab[tuple(slice(s, s + n - 2) if k == a else slice(1, -1) for k, n in enumerate(shape))] == capi.SOLID
    assert good.any() and good.all() == (what == "off water" and not enclosed.any())


# inf: a face without bound; enclosed: a WATER cell between SOLID ones, whose factor is infinite
@pytest.mark.parametrize("shape", [(12, 20, 140), (40, 140, 3)])
@pytest.mark.parametrize("what", ["enclosed", "inf"])
def test_solve_ends_on_what_is_not_a_number(gpu, shape, what):
    print(f"case: solve {shape}, {what}", flush=True)
    two_d = shape[2] == 3
    grid = capi.Grid(*shape, 1.0 / 32, 0.25 / 32, two_d=int(two_d), cell_d_z=0.1 if two_d else 0.0)
    rng = np.random.default_rng(1)
    lab = np.full(shape, capi.WATER, np.uint8)
    x, z = shape[0] // 2, 1 if two_d else 64
    lab[:, 7] = capi.AIR
    lab[:, -2] = capi.AIR
    faces = [rng.standard_normal(shape).astype(np.float32) for _ in range(3)]
    if what == "enclosed":
        lab[x - 1:x + 2, 3:6, z - 1:z + 2] = capi.SOLID
        lab[x, 4, z] = capi.WATER
    else:
        faces[0][x, 6, z] = np.inf
    _walls(lab)
    got = {}
    for mode in (1, 0):
        sim = capi.Simulation(grid, scenes.params(tol=1e-6))
        sim.set_option(capi.OPT_SWEEP_MODE, mode)
        sim.set_grid(capi.FIELD_LABEL, lab.reshape(-1))
        for f, v in zip((capi.FIELD_U2, capi.FIELD_V2, capi.FIELD_W2), faces):
            sim.set_grid(f, v.reshape(-1))
        sim.run_stage(capi.STAGE_SOLVE, DT)
        st = sim.stats()
        got[mode] = (st.pcg_iterations, st.solve_nan, sim.get_grid(capi.FIELD_PRESSURE), sim.get_grid(capi.FIELD_U2))
        sim.close()
    assert got[0][:2] == got[1][:2] == (0, 1)
    assert not got[0][2].any() and not got[1][2].any()
    assert np.array_equal(got[0][3], faces[0].reshape(-1), equal_nan=True)

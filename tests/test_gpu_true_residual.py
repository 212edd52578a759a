"""The FP64 residual of a solve, formed by columns of plane groups, against numpy on the returned pressure, at the sizes
where a column's planes wrap, end inside a group or share a tile edge (-m gpu)."""
import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes

pytestmark = pytest.mark.gpu
DT = scenes.DT


# nx: every remainder of a plane group, below, at and above the 64-lane rotation (60: 16 groups); nz: one lane, a full
# z-tile, one lane in the next, three tiles; 2D
@pytest.mark.parametrize("most", [3, 500])
@pytest.mark.parametrize("shape", [(4, 4, 4), (5, 9, 66), (6, 8, 67), (7, 13, 12), (60, 9, 67), (63, 7, 66), (64, 8, 131),
                                   (66, 20, 65), (130, 6, 70), (33, 40, 3)])
def test_residual_equals_numpy(gpu, shape, most):
    print(f"case: residual on {shape}, at most {most} iterations", flush=True)
    two_d = shape[2] == 3
    grid = capi.Grid(*shape, 1.0 / 32, 0.25 / 32, two_d=int(two_d), cell_d_z=0.1 if two_d else 0.0)
    rng = np.random.default_rng(sum(shape))
    lab = np.full(shape, capi.WATER, np.uint8)
    lab[rng.random(shape) < 0.08] = capi.AIR
    lab[rng.random(shape) < 0.04] = capi.SOLID
    lab[0], lab[-1], lab[:, 0], lab[:, :, 0], lab[:, :, -1] = (capi.SOLID,) * 5
    lab[:, -1] = np.where(lab[:, -1] == capi.WATER, capi.AIR, lab[:, -1])
    lab[1, 1, 1] = capi.WATER
    pad = np.pad(lab, 1, constant_values=capi.SOLID)

    def around(a, s):
        return tuple(slice(1 + (s if k == a else 0), n + 1 + (s if k == a else 0)) for k, n in enumerate(shape))

    sides = [(a, s) for a in range(3) for s in (-1, 1)]
    # WATER without a non-SOLID neighbour has no equation
    lab[(lab == capi.WATER) & np.all([pad[around(a, s)] == capi.SOLID for a, s in sides], axis=0)] = capi.AIR
    pad = np.pad(lab, 1, constant_values=capi.SOLID)
    water = lab == capi.WATER
    faces = [rng.standard_normal(shape).astype(np.float32) for _ in range(3)]
    prm = scenes.params(tol=1e-9)
    prm.max_iterations = most
    sim = capi.Simulation(grid, prm)
    sim.set_grid(capi.FIELD_LABEL, lab.reshape(-1))
    for f, v in zip((capi.FIELD_U2, capi.FIELD_V2, capi.FIELD_W2), faces):
        sim.set_grid(f, v.reshape(-1))
    sim.run_stage(capi.STAGE_SOLVE, DT)
    st = sim.stats()
    b = sim.get_grid(capi.FIELD_RHS).astype(np.float64).reshape(shape)
    p = sim.get_grid(capi.FIELD_PRESSURE).reshape(shape)
    sim.close()
    ppad = np.pad(p, 1)
    scale = DT / (1.0 * grid.cell_d ** 2)
    count, near, size = np.zeros(shape), np.zeros(shape), np.zeros(shape)
    for a, s in sides:
        at = around(a, s)
        count += pad[at] != capi.SOLID
        near += np.where(pad[at] == capi.WATER, ppad[at], 0.0)
        size += np.where(pad[at] == capi.WATER, np.abs(ppad[at]), 0.0)
    t = np.where(water, b - scale * (count * p - near), 0.0)
    # FP64: on either side six roundings of the diagonal, seven products and seven sums of terms below this total
    err = np.where(water, 2 * 20 * 2.0 ** -53 * (np.abs(b) + scale * (count * np.abs(p) + size)), 0.0)
    assert abs(st.residual_abs_inf - np.abs(t).max()) <= err.max()
    l2 = np.linalg.norm(t)
    # the norm's own rounding: a sum of at most that many terms, each square rounded
    assert abs(st.residual_rel_l2 * st.b_norm_l2 - l2) <= np.linalg.norm(err) + 1e-12 * l2
    assert (st.residual_rel_l2 <= 1e-9) == (most == 500) or shape == (4, 4, 4)


def test_residual_costs_little_more_than_a_product(gpu):
    """Per launch it moves 14 bytes a WATER cell, an iteration's matrix product 18: where both are bound by memory it takes
    at most half as long again (a gather cell by cell took 1.9 times as long)."""
    print("case: time of the true residual, 192^3", flush=True)
    sc = scenes.dam_break(192, capi.FLIP)
    sim = capi.Simulation(sc.grid, scenes.params(tol=1e-6))
    sim.set_particles(sc.particles())
    sim.step(DT)
    sim.set_option(capi.OPT_PROFILE, 1)
    for _ in range(4):
        sim.step(DT)
    times = sim.kernel_times()
    sim.close()
    per = {k: times[k][0] / times[k][1] for k in ("true_residual", "spmv")}
    print(per)
    assert times["true_residual"][1] >= 8 and per["true_residual"] <= 1.55 * per["spmv"]

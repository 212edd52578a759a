"""The step length of PCG: alpha = z.r / s.A s with the z and the A s that the solve uses, to FP64 rounding (-m gpu)."""
import math

import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes

pytestmark = pytest.mark.gpu
DT = scenes.DT


# one block beside the product, several, their largest number; the product's grid at its limit; 2D
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("shape", [(5, 6, 7), (12, 20, 140), (67, 40, 70), (128, 100, 130), (4, 1600, 600), (128, 128, 3)])
def test_first_step_takes_z_dot_r(gpu, shape, mode):
    """After one iteration x = alpha z with z = M^-1 b."""
    print(f"case: first step on {shape}, sweep mode {mode}", flush=True)
    two_d = shape[2] == 3
    grid = capi.Grid(*shape, 1.0 / 32, 0.25 / 32, two_d=int(two_d), cell_d_z=0.1 if two_d else 0.0)
    rng = np.random.default_rng(sum(shape))
    lab = np.full(shape, capi.WATER, np.uint8)
    lab[rng.random(shape) < 0.05] = capi.AIR
    lab[0], lab[-1], lab[:, 0], lab[:, :, 0], lab[:, :, -1] = (capi.SOLID,) * 5
    lab[:, -1] = np.where(lab[:, -1] == capi.WATER, capi.AIR, lab[:, -1])
    prm = scenes.params(tol=1e-12)
    prm.max_iterations = 1
    sim = capi.Simulation(grid, prm)
    sim.set_option(capi.OPT_SWEEP_MODE, mode)
    sim.set_grid(capi.FIELD_LABEL, lab.reshape(-1))
    for f in (capi.FIELD_U2, capi.FIELD_V2, capi.FIELD_W2):
        sim.set_grid(f, rng.standard_normal(grid.nc).astype(np.float32))
    sim.run_stage(capi.STAGE_SOLVE, DT)
    b = sim.get_grid(capi.FIELD_RHS).astype(np.float64)
    p = sim.get_grid(capi.FIELD_PRESSURE)
    z = sim.solver_apply(capi.OP_APPLY_MIC0, DT, b)
    q = sim.solver_apply(capi.OP_APPLY_A, DT, z)
    sim.close()
    # both sums are of exact FP64 products; the kernels add theirs in another order
    alpha = math.fsum(z * b) / math.fsum(z * q)
    assert np.count_nonzero(z) == np.count_nonzero(lab == capi.WATER)
    # 2^-53 for each of the 24 levels of those sums at most, relative to the sums of magnitudes
    slack = np.abs(z * b).sum() / abs(math.fsum(z * b)) + np.abs(z * q).sum() / math.fsum(z * q)
    assert np.abs(p - alpha * z).max() <= 24 * 2.0 ** -53 * slack * abs(alpha) * np.abs(z).max()

"""The network on grids whose levels end inside a tile of 16 voxels and on both sides of the rule that gives a wave one
tile, against the FP64 oracle with the same BF16 rounding points (-m gpu)."""
import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes
from oracle import learned_net as net

pytestmark = pytest.mark.gpu


# padded 8 x 8 x 8 (one voxel on the coarsest level), 16 x 24 x 8, 8 x 40 x 24, and 40 x 48 x 56, where the first and
# the last layers have more than 4096 waves' worth of tiles and the others fewer
@pytest.mark.parametrize("shape", [(8, 8, 8), (9, 24, 7), (5, 33, 24), (40, 41, 56)])
def test_network_at_level_edges(gpu, shape):
    print(f"case: network on {shape}", flush=True)
    rng = np.random.default_rng(sum(shape))
    lab = np.where(rng.random(shape) < 0.8, capi.WATER, capi.AIR).astype(np.uint8)
    lab[0], lab[-1], lab[:, 0], lab[:, :, 0], lab[:, :, -1] = (capi.SOLID,) * 5
    lab = lab.reshape(-1)
    b = np.where(lab == capi.WATER, rng.standard_normal(lab.size), 0.0).astype(np.float32)
    sim = capi.Simulation(capi.Grid(*shape, 1.0 / 32, 0.25 / 32), scenes.params())
    sim.learned_init(6)
    params = sim.learned_get_params()
    out = sim.learned_forward(b, lab).reshape(shape)
    sim.close()
    x, _, _ = net.make_input(b, lab, shape)
    ref, _ = net.forward(net.unpack(params), x, emulate_bf16=True)
    ref = ref[:shape[0], :shape[1], :shape[2]]
    # the same bound as at 16^3: FP32 sums in another order may move an activation by one BF16 step
    assert np.linalg.norm(out - ref) <= 2e-2 * np.linalg.norm(ref)

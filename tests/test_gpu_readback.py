"""Results copied to host memory in pieces by several threads (-m gpu): sizes around the pieces' and threads' edges and
destinations off their alignment, and the particles in their own order, against what was put in."""
import numpy as np
import pytest

from fluid_simulator_amd import capi, scenes

pytestmark = pytest.mark.gpu
MB = 1 << 20


# bytes of a field: below the first piece, one float around it, quarter pieces, whole ones, more than all slots
@pytest.mark.parametrize("cells,off", [(64 * 64 * 63, 0), (64 * 64 * 64, 0), (64 * 64 * 64, 3), (5 * 331 * 199, 1),
                                       (4 * 1024 * 1024 - 4 * 1024, 7), (4 * 1024 * 1024, 1), (7 * 1283 * 1501, 5)])
def test_fields_come_back_whole(gpu, cells, off):
    shape = {64 * 64 * 63: (64, 64, 63), 64 * 64 * 64: (64, 64, 64), 5 * 331 * 199: (5, 331, 199),
             4 * MB - 4 * 1024: (4, 1023, 1024), 4 * MB: (4, 1024, 1024), 7 * 1283 * 1501: (7, 1283, 1501)}[cells]
    print(f"case: field of {shape}, destination {off} floats off", flush=True)
    sim = capi.Simulation(capi.Grid(*shape, 1.0 / 32, 0.25 / 32), scenes.params())
    want = np.random.default_rng(cells).standard_normal(cells, np.float32)
    sim.set_grid(capi.FIELD_V2, want)
    out = np.full(cells + 16, np.nan, np.float32)
    for _ in range(2):
        part = out[off:off + cells]
        sim._check(sim.lib.fsim_get_grid(sim._ctx, capi.FIELD_V2, part.ctypes.data, part.nbytes))
        assert np.array_equal(part, want)
        assert np.isnan(out[:off]).all() and np.isnan(out[off + cells:]).all()
        part[:] = 0
    sim.close()


@pytest.mark.parametrize("n", [0, 1, 257, 100_003, 1_700_001])
@pytest.mark.parametrize("transfer", [capi.FLIP, capi.APIC])
def test_particles_come_back_in_their_own_order(gpu, n, transfer):
    print(f"case: {n} particles, transfer {transfer}", flush=True)
    grid = scenes.grid(32)
    rng = np.random.default_rng(n)
    lo = grid.cell_d + 1.01 * grid.particle_r
    pos = rng.uniform(lo, 1.0 - lo, (n, 3)).astype(np.float32)
    vel = rng.standard_normal((n, 3), np.float32)
    c = rng.standard_normal((n, 9), np.float32)
    sim = capi.Simulation(grid, scenes.params(transfer=transfer))
    sim.set_particles(pos, vel, c)
    for step in range(2):   # as they were put in, and sorted by cell
        got = sim.get_particles()
        assert np.array_equal(got[0], pos) and np.array_equal(got[1], vel)
        # PIC and FLIP drop C when the particles are sorted
        assert np.array_equal(got[2], c if step == 0 or transfer == capi.APIC else np.zeros_like(c))
        sim.run_stage(capi.STAGE_BIN)
    if n > 1:
        assert not np.array_equal(sim.slot_ids(), np.arange(n))
    sim.close()

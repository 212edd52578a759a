"""bench.py's algorithmic bytes of the iteration's kernels, array by array (CPU only)."""
import bench

F32, F64, LABEL = 4, 8, 1


def test_bytes_of_the_sweeps_are_those_of_the_arrays_they_use():
    # forward: r, q and the factor in, t and the new r out; no label (the factor is 0 off WATER)
    assert bench.ALGO_BYTES["sweep_fwd"] == ("f", 3 * F32 + 2 * F32)
    # backward: t and the factor in, z out; every other time x in and out with two directions and the mask
    assert bench.ALGO_BYTES["sweep_bwd"] == ("f", 2 * F32 + F32 + (2 * F64 + 2 * F32 + LABEL) / 2)
    # r update: q and r in, r out
    assert bench.ALGO_BYTES["update"] == ("f", 2 * F32 + F32)

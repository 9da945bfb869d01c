"""Particle lattices on both sides of the displacement's change of block, cut on
every axis: blocks of two x planes below 64^3 particles, of eight from there on."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [63, 65])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_positions_of_cut_blocks(gpu, oracle, M, prec):
    N, L = 32, 100.0
    print("case", N, M, prec, flush=True)
    ref = oracle.ic_run(N, L, 5, bins=8, want_density=False, M=M)
    ic = gpu.IC(gpu.ICConfig(N=N, boxlen=L, seed=5, bins=8, M=M,
                             precision=gpu.MITOS_FP64 if prec == "fp64" else gpu.MITOS_FP32))
    ic.run()
    got = [t.cpu().numpy() for t in ic.positions()]
    ic.close()
    for g, c in zip(got, "XYZ"):
        if prec == "fp64":  # the oracle's operations one by one
            assert np.array_equal(g, ref[c])
        else:  # rounding of float positions and displacement grids
            d = np.abs(g.astype(np.float64) - ref[c].astype(np.float64))
            assert np.minimum(d, L - d).max() < 1e-4 * L / N

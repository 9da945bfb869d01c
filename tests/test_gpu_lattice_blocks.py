"""Particle lattices that the displacement's 8 x 8 x 16 blocks cut: below one block,
one site over a block on every axis, coarser and finer than the grid, and the
particle-per-cell FP64 grid whose size is not a multiple of 16."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pos_err(a, b, L):
    d = np.abs(a.astype(np.float64) - b.astype(np.float64))
    return np.minimum(d, L - d).max()


@pytest.mark.parametrize("N,M,L,prec", [
    (32, 7, 128.0, "fp64"), (32, 17, 100.0, "fp64"), (32, 33, 128.0, "fp64"),
    (24, 24, 96.0, "fp64"), (32, 7, 128.0, "fp32"), (32, 17, 100.0, "fp32"),
    (48, 33, 100.0, "fp32")])
def test_positions_of_cut_lattices(gpu, oracle, N, M, L, prec):
    # FP64 moves are the oracle's operations one by one; FP32 ones stay within the
    # rounding of float positions and displacement grids (1e-4 cells)
    print("case", N, M, L, prec, flush=True)
    ref = oracle.ic_run(N, L, 11, bins=8, want_density=True, M=M)
    p = gpu.MITOS_FP64 if prec == "fp64" else gpu.MITOS_FP32
    ic = gpu.IC(gpu.ICConfig(N=N, boxlen=L, seed=11, bins=8, precision=p, M=M))
    ic.run()
    got = [t.cpu().numpy() for t in ic.positions()]
    ic.close()
    for g, c in zip(got, "XYZ"):
        assert g.size == M ** 3
        if prec == "fp64":
            assert np.array_equal(g, ref[c])
        else:
            assert _pos_err(g, ref[c], L) < 1e-4 * L / N

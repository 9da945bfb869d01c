"""The 2LPT source on FP64 lines of four values a thread: rows that share a wave
(128, 256); 512 and 1024 are in the configuration tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("N", [128, 256])
def test_solve2lpt_lines(gpu, oracle, N):
    # FP64 transforms of N^3: relative error of order 1e-16 log2(N^3), three in a row
    print("case solve2LPT lines", N, flush=True)
    L = 2.0 * N
    f = oracle.grf(N, L, 11)
    f = oracle.apply_kernel(f, L, oracle.K_SQRT_POWER_LAW, (2e5, 0.965))
    od, op, ow = oracle.Grid(N, L), oracle.Grid(N, L), oracle.Grid(N, L)
    od.fbox[:] = f
    od.box[:, :, :N] = oracle.fft_c2r(f) / L ** 3
    od.s.momentum_space = b"\x01"
    assert oracle.solve_2lpt(op, od, ow, 1.0, -3.0 / 7.0) == 0
    d, p, w = gpu.Grid(N, L), gpu.Grid(N, L), gpu.Grid(N, L)
    d.set_fbox(f)
    d.set_box(od.box)
    d.momentum_space = 1
    assert gpu.solve2LPT(p, d, w, 1.0, -3.0 / 7.0) == 0
    assert _rel(p.fbox(), op.fbox) < 1e-11
    assert _rel(w.box()[:, :, :N], ow.box[:, :, :N]) < 1e-11

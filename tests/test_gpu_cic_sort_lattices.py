"""The sorted deposit inside a realization whose particles are not the grid's (float
and double weights, one and several passes in the displacement grids) and the grids
too small for it, against the same integer sums formed on the host."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# FP32: two passes (cells cut on every axis), three passes, atomics; FP64: three
# passes, one pass, atomics on the smallest grid
@pytest.mark.parametrize("fp32,N,M", [(True, 96, 90), (True, 128, 150), (True, 16, 90),
                                      (False, 96, 150), (False, 96, 90), (False, 8, 81)])
def test_realization_deposit(gpu, host_checks, fp32, N, M):
    L = 1000.0 / 3
    print("case sorted deposit", fp32, N, M, flush=True)
    cfg = gpu.ICConfig(N=N, M=M, boxlen=L, seed=11, bins=16,
                       precision=gpu.MITOS_FP32 if fp32 else gpu.MITOS_FP64)
    ctx = gpu.IC(cfg)
    ctx.run()
    pos = [np.ascontiguousarray(t.cpu().numpy()) for t in ctx.positions()]
    delta = ctx.density().cpu().numpy()
    ctx.close()
    grid = np.zeros((N, N, N), np.uint64)
    check = host_checks.check_deposit_f if fp32 else host_checks.check_deposit_d
    check(N, ctypes.c_double(L), ctypes.c_long(M ** 3),
          *(p.ctypes.data_as(ctypes.c_void_p) for p in pos), grid.ctypes.data_as(ctypes.c_void_p))
    want = grid.astype(np.float64) * (2.0 ** (-24 if fp32 else -40) * (N ** 3 / M ** 3)) - 1
    # one rounding of the same sum to the density's type
    assert np.all(np.abs(delta - want) <= np.spacing(1 + np.abs(want).astype(delta.dtype)))


# the smallest array that is sorted on a grid of 8^3 and the largest that is not
@pytest.mark.parametrize("n", [524287, 524288])
def test_rule_edge_same_sums(gpu, n):
    import torch
    N, L = 8, 10.0
    print("case sorted deposit rule", n, flush=True)
    q = np.random.default_rng(2).random((3, n)).astype(np.float32) * np.float32(L)
    d = [torch.from_numpy(p).cuda() for p in q]
    out = [torch.empty((N, N, N), dtype=torch.float64, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    p = [t.data_ptr() for t in d]
    assert gpu.lib().mitos_cic_overdensity(N, L, n, *p, out[0].data_ptr()) == 0
    assert gpu.lib().mitos_cic_overdensity_noalloc(N, L, n, *p, out[1].data_ptr(), None) == 0
    assert torch.equal(*out)

"""The FP32 deposit of the adjoint's forward in LDS windows (one pass, two passes, far
particles, cells past the window's 32 bits) and by atomics (32^3), against the same
integer sums of the same positions formed on the host."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _noise(gpu, N, how):
    import torch
    if how == "white":
        return gpu.white_noise(N, 3, gpu.MITOS_FP32)
    # one wave along each axis: particles fall together where all three converge
    n = torch.zeros(N, N, N // 2 + 1, dtype=torch.complex64, device="cuda")
    n[1, 0, 0] = n[N - 1, 0, 0] = n[0, 1, 0] = n[0, N - 1, 0] = n[0, 0, 1] = 1.0
    return n


# cells of 1.5, whose reciprocal rounds; cells of 1/4, whose particles leave the windows
@pytest.mark.parametrize("N,L,how", [(32, 48.0, "white"), (64, 96.0, "white"),
                                     (128, 192.0, "white"), (128, 32.0, "white"),
                                     (128, 192.0, "wave")])
def test_deposit_of_the_forward(gpu, host_checks, N, L, how):
    import torch
    print("case adjoint deposit", N, L, how, flush=True)
    cfg = gpu.ICConfig(N=N, boxlen=L, seed=3, bins=8, run2lpt=int(how == "white"),
                       precision=gpu.MITOS_FP32)
    ctx = gpu.IC(cfg)
    noise = _noise(gpu, N, how)
    q = np.arange(N, dtype=np.float32)[:, None, None] * np.float32(L / N)
    torch.cuda.synchronize()
    ctx.noise_forward(cfg, noise)
    if how == "wave":
        # the amplitude at which the waves' crossings meet: L / 2 pi
        x = ctx.positions()[0].cpu().numpy().reshape(N, N, N) - q
        far = np.abs(x - L * np.round(x / L)).max()
        noise = noise * float(L / (2 * np.pi) / far)
        torch.cuda.synchronize()
        ctx.noise_forward(cfg, noise)
    pos = [np.ascontiguousarray(t.cpu().numpy()) for t in ctx.positions()]
    delta = ctx.density().cpu().numpy()
    ctx.close()
    grid = np.zeros((N, N, N), np.uint64)
    host_checks.check_deposit_t(N, ctypes.c_double(L), ctypes.c_long(N ** 3),
                                *(p.ctypes.data_as(ctypes.c_void_p) for p in pos),
                                grid.ctypes.data_as(ctypes.c_void_p))
    if how == "wave":
        assert grid.max() >= 1 << 32
    want = grid.astype(np.float64) * 2.0 ** -24 - 1
    # one rounding of the same sum to float
    assert np.all(np.abs(delta - want) <= np.spacing(1 + np.abs(want).astype(np.float32)))
    assert int(grid.sum()) == pytest.approx(N ** 3 * 2 ** 24, abs=8 * N ** 3)

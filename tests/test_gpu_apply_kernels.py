"""k-space kernels whose values come from tables (windows, spectra) and the
block decomposition of the grid, at sizes around its edges, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# fewer modes than a block, rows shorter and longer than a block's tail, odd and
# prime sizes (the apply functions take any N), and sizes that use the tables
@pytest.mark.parametrize("N", [2, 7, 8, 62, 64, 66, 101])
def test_apply_kernels_any_size(gpu, oracle, N):
    rng = np.random.default_rng(N)
    L = 150.0
    H = N // 2 + 1
    f = rng.standard_normal((N, N, H)) + 1j * rng.standard_normal((N, N, H))
    cases = [
        ("kernel_dy", {}, oracle.K_DY, ()),
        ("kernel_power_no_transfer", {"A_s": 2.1e-9, "n_s": 0.96, "k_pivot": 0.05},
         oracle.K_POWER_NO_TRANSFER, (2.1e-9, 0.96, 0.05)),
        ("kernel_undo_Hermite_window", {"order": 2, "N": N, "boxlen": L}, oracle.K_UNDO_WINDOW,
         (2, N, L)),
        ("kernel_undo_Hermite_window", {"order": 3, "N": 2 * N, "boxlen": L},
         oracle.K_UNDO_WINDOW, (3, 2 * N, L)),
        ("kernel_undo_Hermite_window", {"order": 4, "N": 2 * N, "boxlen": L},
         oracle.K_UNDO_WINDOW, (4, 2 * N, L)),
        ("kernel_sqrt_power_law", {"A": 1.5e6, "n_s": 0.965}, oracle.K_SQRT_POWER_LAW,
         (1.5e6, 0.965)),
        ("kernel_bbks_transfer", {"Gamma": 0.21}, oracle.K_BBKS, (0.21,)),
    ]
    import torch
    lib = gpu.lib()
    import ctypes
    d = torch.from_numpy(f).cuda()
    for name, kw, kid, prm in cases:
        print("case apply", N, name, flush=True)
        p = gpu.kernel_params(name, **kw)
        out = torch.empty_like(d)
        torch.cuda.synchronize()
        assert lib.fft_apply_kernel(out.data_ptr(), d.data_ptr(), N, L, gpu.kernel_ptr(name),
                                    ctypes.cast(ctypes.byref(p), ctypes.c_void_p)
                                    if p is not None else None) == 0
        ref = oracle.apply_kernel(f, L, kid, prm)
        err = np.abs(out.cpu().numpy() - ref)
        # a few roundings of the factor and of the product
        assert np.all(err <= 4e-15 * np.abs(ref) + 1e-300), name

"""k-space kernels at the sizes where their values change from formulas to tables and
a thread from one mode to four, whole grids and slabs, against the formulas."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (N, planes): below the window's table, with it, the spectra's table, four modes a
# thread, and slabs of few modes an entry that start inside the grid
@pytest.mark.parametrize("N,x0,nx", [(78, 0, 78), (82, 0, 82), (102, 0, 102), (130, 0, 130),
                                     (512, 300, 3), (512, 250, 13), (256, 120, 17)])
@pytest.mark.parametrize("name", ["window", "power", "bbks"])
def test_tables_and_formulas_agree(gpu, N, x0, nx, name):
    import torch
    print("case apply tables", N, x0, nx, name, flush=True)
    L, H = 150.0, N // 2 + 1
    kernel, kw = {"window": ("kernel_undo_Hermite_window", dict(order=3, N=N, boxlen=L)),
                  "power": ("kernel_sqrt_power_law", dict(A=1.5e6, n_s=0.965)),
                  "bbks": ("kernel_bbks_transfer", dict(Gamma=0.21))}[name]
    gen = torch.Generator(device="cuda").manual_seed(N)
    f = torch.randn(nx, N, H, dtype=torch.complex64, device="cuda", generator=gen)
    out = torch.zeros_like(f)
    p = gpu.kernel_params(kernel, **kw)
    torch.cuda.synchronize()
    assert gpu.lib().fft_apply_kernel_float_mpi(
        out.data_ptr(), f.data_ptr(), N, x0, nx, L, gpu.kernel_ptr(kernel),
        ctypes.cast(ctypes.byref(p), ctypes.c_void_p)) == 0
    i = torch.arange(N, device="cuda", dtype=torch.float64)
    i = torch.where(i > N // 2, i - N, i)
    n = [i[x0:x0 + nx, None, None], i[None, :, None], i[None, None, :H].abs()]
    dk = 2 * np.pi / L
    if name == "window":
        w = 1.0
        for m in n:
            w = w * torch.sinc(m / N)
        v = w ** -3
    else:
        k = dk * torch.sqrt(n[0] ** 2 + n[1] ** 2 + n[2] ** 2)
        if name == "power":
            v = torch.sqrt(1.5e6 * k ** 0.965)
        else:
            q = k / 0.21
            poly = 1 + 3.89 * q + (16.1 * q) ** 2 + (5.46 * q) ** 3 + (6.71 * q) ** 4
            v = torch.log1p(2.34 * q) / (2.34 * q) * poly ** -0.25
            v = torch.where(k > 0, v, torch.ones_like(v))
    want = torch.view_as_real(f).double() * v[..., None]
    got = torch.view_as_real(out).double()
    if name != "window":  # the spectra's value at k = 0 is a convention
        got, want = got.clone(), want.clone()
        if x0 == 0:
            got[0, 0, 0] = want[0, 0, 0] = 0
    # one rounding to float of a product in double
    assert torch.all((got - want).abs() <= 2.0 ** -23 * want.abs() + 1e-30)


@pytest.mark.parametrize("name,kw", [("kernel_dx", {}),
                                     ("kernel_undo_Hermite_window", dict(order=2, N=16, boxlen=9.0)),
                                     ("kernel_bbks_transfer", dict(Gamma=0.2))])
def test_empty_slab_is_refused(gpu, name, kw):
    import torch
    print("case empty slab", name, flush=True)
    f = torch.zeros(1, 16, 9, dtype=torch.complex64, device="cuda")
    torch.cuda.synchronize()
    p = gpu.kernel_params(name, **kw) if kw else None
    assert gpu.lib().fft_apply_kernel_float_mpi(
        f.data_ptr(), f.data_ptr(), 16, 0, 0, 9.0, gpu.kernel_ptr(name),
        ctypes.cast(ctypes.byref(p), ctypes.c_void_p) if p is not None else None) == 3

"""Calls of several host threads on one device: transforms of different sizes (whose
work grids grow), tables, Poisson and deposits get the results they get alone."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_threads_do_not_disturb_each_other(gpu):
    import torch
    print("case scratch threads", flush=True)
    lib = gpu.lib()
    gen = torch.Generator(device="cuda").manual_seed(8)
    L = 100.0
    jobs = []

    def job(call, shape, dtype):
        out = torch.zeros(shape, dtype=dtype, device="cuda")
        jobs.append((call, out))

    def randn(*shape, dtype=torch.float64):
        return torch.randn(*shape, dtype=dtype, device="cuda", generator=gen)

    for N in (48, 192, 96, 256, 128):
        x = randn(N, N, N)
        k = randn(N, N, N // 2 + 1, dtype=torch.complex128)
        job(lambda o, N=N, x=x: lib.mitos_fft_r2c(N, x.data_ptr(), o.data_ptr()),
            (N, N, N // 2 + 1), torch.complex128)
        job(lambda o, N=N, k=k: lib.mitos_fft_c2r(N, k.data_ptr(), o.data_ptr()),
            (N, N, N), torch.float64)
        job(lambda o, N=N, x=x: lib.solvePoisson(o.data_ptr(), x.data_ptr(), N, L),
            (N, N, N), torch.float64)
        for name, kw in (("kernel_bbks_transfer", dict(Gamma=0.21)),
                         ("kernel_undo_Hermite_window", dict(order=3, N=N, boxlen=L))):
            p = gpu.kernel_params(name, **kw)
            job(lambda o, N=N, k=k, name=name, p=p: lib.fft_apply_kernel(
                o.data_ptr(), k.data_ptr(), N, L, gpu.kernel_ptr(name),
                ctypes.cast(ctypes.byref(p), ctypes.c_void_p)),
                (N, N, N // 2 + 1), torch.complex128)
    for n in (700001, 2000003):
        q = torch.rand(3, n, device="cuda", generator=gen) * L
        for N in (64, 128):
            job(lambda o, N=N, n=n, q=q: lib.mitos_cic_overdensity(
                N, L, n, *(q[a].data_ptr() for a in range(3)), o.data_ptr()),
                (N, N, N), torch.float64)
    torch.cuda.synchronize()
    want = []
    for call, out in jobs:
        assert call(out) == 0
        want.append(out.cpu().numpy().copy())
    rc = {}

    def work(t, order):
        for i in order:
            rc[t, i] = jobs[i][0](jobs[i][1])

    for turn in range(4):
        assert lib.mitos_release_workspace() == 0
        for _, out in jobs:
            out.zero_()
        torch.cuda.synchronize()
        parts = np.array_split(np.random.default_rng(turn).permutation(len(jobs)), 6)
        threads = [threading.Thread(target=work, args=(t, [int(i) for i in part]))
                   for t, part in enumerate(parts)]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        assert len(rc) >= len(jobs) and not any(rc.values())
        for (_, out), ref in zip(jobs, want):
            assert np.array_equal(out.cpu().numpy(), ref)


def test_grids_take_scratch_back(gpu):
    """a grid that fits only without the transforms' work grid is allocated"""
    import torch
    print("case scratch given back", flush=True)
    lib = gpu.lib()
    N = 512
    x = torch.zeros(N, N, N, dtype=torch.float64, device="cuda")
    k = torch.zeros(N, N, N // 2 + 1, dtype=torch.complex128, device="cuda")
    assert lib.mitos_release_workspace() == 0
    torch.cuda.synchronize()
    assert lib.mitos_fft_r2c(N, x.data_ptr(), k.data_ptr()) == 0  # holds 1.1 GB
    torch.cuda.empty_cache()
    hog = []
    while True:  # leave half a gigabyte
        free = torch.cuda.mem_get_info()[0] - (512 << 20)
        if free < (64 << 20):
            break
        try:
            hog.append(torch.empty(free, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            break
    assert torch.cuda.mem_get_info()[0] < (1 << 30)
    g = gpu.Grid(384, 100.0)  # 0.9 GB
    g.free()
    assert lib.mitos_release_workspace() == 0
    del hog
    torch.cuda.empty_cache()

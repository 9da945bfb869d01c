"""Transforms where their work grid cannot be had: r2c runs in its output, as it
needs no scratch, with the same bits."""
import pytest

pytestmark = pytest.mark.gpu


def test_r2c_without_scratch(gpu):
    import torch
    lib = gpu.lib()
    N = 512  # work grid 1.1 GB, dense or not
    print("case r2c without scratch", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(N, N, N, dtype=torch.float64, device="cuda", generator=gen)
    want = torch.empty(N, N, N // 2 + 1, dtype=torch.complex128, device="cuda")
    got = torch.zeros_like(want)
    torch.cuda.synchronize()
    assert lib.mitos_fft_r2c(N, x.data_ptr(), want.data_ptr()) == 0
    assert lib.mitos_release_workspace() == 0
    torch.cuda.empty_cache()
    hog = []
    while True:  # leave half a work grid
        free = torch.cuda.mem_get_info()[0] - (512 << 20)
        if free < (64 << 20):
            break
        try:
            hog.append(torch.empty(free, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            break
    assert torch.cuda.mem_get_info()[0] < (1 << 30)
    torch.cuda.synchronize()
    assert lib.mitos_fft_r2c(N, x.data_ptr(), got.data_ptr()) == 0
    del hog
    torch.cuda.empty_cache()
    assert torch.equal(torch.view_as_real(got), torch.view_as_real(want))

"""The white noise drawn in segments of the stream (grids below 256^3) and in
whole rows: the oracle's draws, in any row layout."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one segment, segments cut by the grid's end, more segments than one work-group
# starts
@pytest.mark.parametrize("N", [2, 4, 6, 10, 22, 34, 50])
def test_segmented_noise_matches_oracle(gpu, oracle, N):
    L = 100.0
    print("case noise segments", N, flush=True)
    g = gpu.Grid(N, L)
    st = gpu.rand_uint64_init(11)
    assert gpu.generate_complex_grf(g, st) == 0
    got, ref = g.fbox(), oracle.grf(N, L, 11, hermitian=False)
    # the Gaussians are correctly rounded; glibc's differ by an ulp at times
    assert np.linalg.norm(got - ref) < 1e-15 * np.linalg.norm(ref)
    assert got[0, 0, 0] == 0
    g.free()


# the three segment lengths at their largest sizes, and the first sizes in rows
@pytest.mark.parametrize("N", [96, 98, 160, 162, 254, 256, 384])
def test_segments_at_large_sizes(gpu, oracle, N):
    """single modes of the stream, jumped to on the host"""
    L = 2.0 ** (1 / 3)  # sqrt(L^3 / 2) = 1
    print("case noise segments", N, flush=True)
    g = gpu.Grid(N, L)
    st = gpu.rand_uint64_init(42)
    assert gpu.generate_complex_grf(g, st) == 0
    got = g.fbox().reshape(-1)
    H = N // 2 + 1
    for m in (1, 15, 16, 17, 4095, 4096, 12345 * 7, N * N * H // 2 + 5, N * N * H - 1):
        A, B, C, D = (float(v) for v in oracle.draws(42, 4 * (m - 1), 4))
        u = [(v + 0.5) / 2.0 ** 64 for v in (A, B, C, D)]
        want = complex(np.sqrt(-2 * np.log(u[0])) * np.cos(2 * np.pi * u[1]),
                       np.sqrt(-2 * np.log(u[2])) * np.cos(2 * np.pi * u[3]))
        f = np.sqrt(L ** 3 / 2)
        assert abs(got[m] - want * f) < 1e-14 * max(1.0, abs(want)), m
    g.free()

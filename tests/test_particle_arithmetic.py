"""The index and weight arithmetic of the particle kernels, compiled for the host:
positions far from the box, at the edges of cells and of the box."""
import ctypes

import numpy as np
import pytest


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


# every compiled grid size: powers of two, whose reciprocal is exact, and 3 * 2^k
@pytest.mark.parametrize("N", [8, 16, 24, 48, 96, 256, 384, 1024, 1536])
def test_wrapped_cells_stay_in_the_grid(host_checks, N):
    rng = np.random.default_rng(N)
    near = rng.integers(-(1 << 22) + 1, 1 << 22, 200000)
    far = rng.integers(-(1 << 31), 1 << 31, 200000)
    ends = np.array([0, -1, N, N - 1, -N, -(1 << 31), (1 << 31) - 1])
    i = np.concatenate([near, far, ends]).astype(np.int32)
    out = np.empty_like(i)
    host_checks.check_wrapf(N, ctypes.c_long(i.size), _p(i), _p(out))
    assert out.min() >= 0 and out.max() < N
    assert np.array_equal(out[:near.size], np.mod(near, N))


# the deposit takes a base index in [-N, 2N) and wraps it once: positions up to far
# more box lengths than a float resolves, infinities and NaN
@pytest.mark.parametrize("N,L", [(32, 48.0), (96, 1000 / 3), (256, 500.0), (256, 512.0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_deposit_cells_stay_in_the_grid(host_checks, N, L, dtype):
    rng = np.random.default_rng(N)
    scale = 10.0 ** rng.uniform(0, 30, 200000)
    x = np.concatenate([L * scale * rng.choice([-1, 1], scale.size), L * rng.random(200000),
                        [0, L, np.nextafter(dtype(L), dtype(0)), -1e-30, np.inf, -np.inf, np.nan]])
    x = x.astype(dtype)
    base = np.empty(x.size, np.int32)
    check = host_checks.check_lattice_cell_f if dtype == np.float32 else host_checks.check_lattice_cell_d
    for site in (0, N // 2, N - 1):
        check(N, ctypes.c_double(L), ctypes.c_long(x.size), site, _p(x), _p(base))
        assert base.min() >= -N and base.max() < 2 * N


# cells of 1.5 and 2.5, whose reciprocals round, and of 2; positions everywhere and
# a few floats around every cell edge
@pytest.mark.parametrize("N,L", [(256, 384.0), (96, 240.0), (256, 512.0)])
def test_float_cell_offsets_and_mass(host_checks, N, L):
    rng = np.random.default_rng(N)
    edge = np.float32(np.arange(N) * (L / N))
    near = [edge]
    for to in (-np.inf, np.inf):
        x = edge
        for _ in range(4):
            x = np.nextafter(x, np.float32(to))
            near.append(x)
    x = np.concatenate([rng.random(1000000) * L, *near]).astype(np.float32)
    d = np.empty_like(x)
    mass = np.empty(x.size, np.uint64)
    host_checks.check_cell_mass(N, ctypes.c_double(L), ctypes.c_long(x.size), _p(x), _p(d), _p(mass))
    assert d.min() >= 0 and d.max() <= 1
    # eight weights, each from four roundings of 2^-24 of itself and one to a unit
    assert np.abs(mass.astype(np.int64) - (1 << 24)).max() <= 8


# moved coordinates are not wrapped yet: below zero, where X - floor(X) rounds, and
# on both sides of cell edges and half cells
def test_tsc_weights_have_the_reference_bits(host_checks):
    rng = np.random.default_rng(1)
    marks = np.arange(-40, 41) / 2.0
    near = [marks]
    for to in (-np.inf, np.inf):
        x = marks
        for _ in range(3):
            x = np.nextafter(x, to)
            near.append(x)
    x = np.concatenate([rng.uniform(a, b, 300000) for a, b in ((-0.5, 0), (-5, 5), (0, 300))] +
                       [-10.0 ** rng.uniform(-300, 0, 100000), *near, [1e15, -1e15, np.inf, np.nan]])
    res = []
    for check in (host_checks.check_tsc_axis, host_checks.check_tsc_axis_short):
        i, w = np.empty(x.size, np.int32), np.empty((x.size, 3))
        check(ctypes.c_long(x.size), _p(x), _p(i), _p(w))
        res.append((i, w))
    assert np.array_equal(res[0][1].view(np.uint64), res[1][1].view(np.uint64))
    inside = np.abs(x) < 1e9
    assert np.array_equal(res[0][0][inside], res[1][0][inside])

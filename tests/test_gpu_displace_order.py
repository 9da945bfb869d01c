"""The particle loop in blocks of lattice indices against memory order, and grids
past 4 GB: the order of work and the offsets' width do not change a result."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _grids(gpu, N, L, count, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        g = gpu.Grid(N, L)
        box = np.zeros((N, N, N + 2))
        box[:, :, :N] = 3.0 * L / N * rng.standard_normal((N, N, N))
        box[:, :, N:] = np.nan  # the padding is never read
        g.set_box(box)
        g.momentum_space = 0
        out.append(g)
    return out


# M^3 particles are walked in 8 x 8 x 16 blocks, M^3 + 1 in memory order; blocks
# cut on every axis, lattices coarser and finer than the grid, the smallest grid
@pytest.mark.parametrize("N,M", [(8, 16), (24, 17), (32, 31), (32, 33), (16, 40)])
@pytest.mark.parametrize("velocities", [False, True])
def test_block_order_same_bits(gpu, N, M, velocities):
    import torch
    L = 100.0 / 3
    print("case displace order", N, M, velocities, flush=True)
    grids = _grids(gpu, N, L, 6 if velocities else 3, N + M)
    lib = gpu.lib()
    n = M ** 3
    rng = np.random.default_rng(5)
    q = (np.indices((M, M, M)).reshape(3, -1) * np.float32(L / M)).astype(np.float32)
    q = np.concatenate([q, np.float32([[L], [-L], [2.5 * L]])], 1)
    far = rng.integers(0, n, 50)
    q[:, far] += np.float32(L) * rng.integers(-3, 4, (3, 50)).astype(np.float32)
    res = []
    for count in (n, n + 1):
        t = [torch.from_numpy(q[a, :count].copy()).cuda() for a in range(3)]
        v = [torch.full((count,), np.nan, device="cuda") for _ in range(3)]
        torch.cuda.synchronize()
        p = [x.data_ptr() for x in t + v]
        if velocities:
            assert lib.mitos_displace_velocity_tsc_dg(*(g.ref() for g in grids), count, *p) == 0
        else:
            assert lib.mitos_displace_tsc_dg(*(g.ref() for g in grids), count, *p[:3]) == 0
        res.append([x[:n] for x in t + (v if velocities else [])])
    for a, b in zip(*res):
        assert torch.equal(a, b) and not torch.isnan(a).any()


def test_grid_past_4_gb(gpu):
    """814^3: element offsets need more than 32 bits of bytes"""
    import torch
    N, L = 814, 814.0
    print("case displace past 4 GB", flush=True)
    g = gpu.Grid(N, L)

    class View:
        __cuda_array_interface__ = dict(data=(g.s.box, False), shape=(N, N, N + 2),
                                        typestr="<f8", strides=None, version=2)

    gen = torch.Generator(device="cuda").manual_seed(1)
    box = torch.as_tensor(View(), device="cuda")
    box.copy_(torch.randn(box.shape, generator=gen, device="cuda", dtype=torch.float64))
    g.momentum_space = 0
    n = 4099
    pos = torch.rand(3, n, generator=gen, device="cuda") * L
    pos[0, :64] = L - 0.25  # the last planes
    want = []
    cells = [pos[a].double() * N / L for a in range(3)]
    near = [torch.floor(c + 0.5) for c in cells]
    total = torch.zeros(n, dtype=torch.float64, device="cuda")
    for a in range(-1, 2):
        for b in range(-1, 2):
            for c in range(-1, 2):
                w = 1.0
                for d, (cell, at) in zip((a, b, c), zip(cells, near)):
                    u = (cell - at - d).abs()
                    w = w * torch.where(u < 0.5, 0.75 - u * u, 0.5 * (1.5 - u) ** 2)
                i = [((m + d).long() % N) for m, d in zip(near, (a, b, c))]
                total += w * box[i[0], i[1], i[2]]
    x, y, z = (pos[a].clone() for a in range(3))
    v = [torch.empty(n, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    none = None
    assert gpu.lib().mitos_displace_velocity_tsc_dg(
        none, none, none, g.ref(), g.ref(), g.ref(), n, x.data_ptr(), y.data_ptr(), z.data_ptr(),
        *(t.data_ptr() for t in v)) == 0
    for t in v:  # one rounding to float of a sum of 27 doubles
        assert (t.double() - total).abs().max() < 1e-6 * total.abs().max()
    g.free()

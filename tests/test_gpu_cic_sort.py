"""The sorted CIC deposit (particles in any order, tiles of 8 x 8 x 64 cells)
against the one-thread-per-particle atomic deposit: the same integer sums, so
the same overdensity bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _both(gpu, N, L, pos):
    """(mitos_cic_overdensity, mitos_cic_overdensity_noalloc) of positions"""
    import torch
    lib = gpu.lib()
    X, Y, Z = (torch.from_numpy(np.ascontiguousarray(p, np.float32)).cuda() for p in pos)
    out = [torch.empty((N, N, N), dtype=torch.float64, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    n = X.numel()
    assert lib.mitos_cic_overdensity(N, L, n, X.data_ptr(), Y.data_ptr(), Z.data_ptr(),
                                     out[0].data_ptr()) == 0
    assert lib.mitos_cic_overdensity_noalloc(N, L, n, X.data_ptr(), Y.data_ptr(), Z.data_ptr(),
                                             out[1].data_ptr(), None) == 0
    return out


# grids below, at and past the tile sizes, odd ones, and particle counts at the
# smallest number that is sorted, odd and at the group sizes
@pytest.mark.parametrize("N", [2, 7, 8, 9, 63, 64, 65, 96, 127, 128])
@pytest.mark.parametrize("order", ["shuffled", "lattice"])
def test_sorted_deposit_same_bits(gpu, N, order):
    import torch
    L = 100.0 / 3
    rng = np.random.default_rng(N)
    n = {2: 524288, 7: 524289, 8: 532479}.get(N, 600001)
    pos = rng.random((3, n)) * L
    if order == "lattice":  # runs along z, several particles a cell
        pos[:, :] = pos[:, np.lexsort((pos[2], np.floor(pos[1] / L * 8), np.floor(pos[0] / L * 8)))]
    pos = pos.astype(np.float32)
    # corners of the box, cell edges, positions outside it
    pos[:, :4] = np.float32([[0, L, np.nextafter(np.float32(L), np.float32(0)), -1e-3]] * 3)
    pos[0, 4:8] = np.float32([-5.5 * L, 7.25 * L, 2 * L, -L])
    print("case sorted cic N", N, order, n, flush=True)
    a, b = _both(gpu, N, L, pos)
    assert torch.equal(a, b)


def test_sorted_deposit_one_cell_and_passes(gpu):
    """every particle in one cell, and more particles than one pass holds"""
    import torch
    L, N = 64.0, 64
    print("case sorted cic one cell", flush=True)
    a, b = _both(gpu, N, L, np.full((3, 570001), 63.75))
    assert torch.equal(a, b)
    n = (1 << 26) + 1001
    print("case sorted cic passes", n, flush=True)
    rng = np.random.default_rng(3)
    pos = [rng.random(n, dtype=np.float32) * np.float32(L) for _ in range(3)]
    a, b = _both(gpu, N, L, pos)
    assert torch.equal(a, b)


def test_sorted_deposit_of_a_denser_lattice(gpu):
    """a fused realization with M != N sorts in the pipeline's own grids, which
    hold fewer particles than this lattice has: several passes"""
    import torch
    N, M, L = 64, 128, 100.0
    print("case sorted cic pipeline", N, M, flush=True)
    ctx = gpu.IC(gpu.ICConfig(N=N, M=M, boxlen=L, seed=3, bins=16, precision=gpu.MITOS_FP64))
    ctx.run()
    X, Y, Z = (t.cpu().numpy() for t in ctx.positions())
    delta = ctx.density()
    _, b = _both(gpu, N, L, (X, Y, Z))
    assert torch.equal(delta, b)
    ctx.close()

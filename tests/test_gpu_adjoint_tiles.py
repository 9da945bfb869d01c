"""The tiled particle kernels of the adjoint (LDS windows with margins, the
tiled FP64 deposit) against torch.autograd through the FP64 restatement."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# tiles cut at the grid's edge (8, 24), whole tiles and the tiled deposit (32),
# and cells so small that most particles leave the windows' margins (L = 8)
@pytest.mark.parametrize("N,L", [(8, 16.0), (24, 12.0), (32, 64.0), (32, 8.0)])
def test_tiled_adjoint_vs_autograd(gpu, N, L):
    from mitos_amd import adjoint
    from oracle import adjoint_ref as R
    ic = gpu
    print("case tiled adjoint", N, L, flush=True)
    cfg = ic.ICConfig(N=N, boxlen=L, seed=7, bins=8, precision=ic.MITOS_FP64)
    ctx = ic.IC(cfg)
    fw = R.Forward(N, L, 8, ic.sigma8_amplitude(0.965, 0.21, 0.81))
    noise = ic.white_noise(N, 7, ic.MITOS_FP64)
    nz = noise.cpu().numpy()
    r = np.random.default_rng(4).standard_normal((N, N, N))
    with torch.no_grad():
        dref = fw.density(torch.tensor(nz)).numpy()
    _, gref = R.density_gradient(fw, nz, r)
    leaf = noise.clone().requires_grad_(True)
    d = adjoint.noise_density(leaf, ctx, cfg)
    rt = torch.from_numpy(r).cuda()
    ((d * rt).sum() + 0.5 * (d * d).sum()).backward()
    # the bounds of the untiled comparison: fixed point of 2^-40, FP64 sums
    assert np.abs(d.detach().cpu().numpy() - dref).max() < 1e-9
    g = leaf.grad.cpu().numpy()
    assert np.linalg.norm(g - gref) < 1e-8 * np.linalg.norm(gref)
    # the sums do not depend on the order of the atomics
    again = noise.clone().requires_grad_(True)
    d = adjoint.noise_density(again, ctx, cfg)
    ((d * rt).sum() + 0.5 * (d * d).sum()).backward()
    assert torch.equal(torch.view_as_real(leaf.grad), torch.view_as_real(again.grad))
    ctx.close()

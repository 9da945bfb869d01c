"""The particle loop over arrays large enough for blocks of lattice indices: in
blocks, in memory order and shuffled (scattered lanes read single values) each
particle gets the same bits, and they are the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# the smallest array in blocks, blocks cut on every axis, and grids on which most
# waves wrap in z; positions below zero and past the box among them
@pytest.mark.parametrize("N,M", [(8, 64), (32, 65), (48, 71)])
@pytest.mark.parametrize("velocities", [False, True])
def test_orders_same_bits(gpu, oracle, N, M, velocities):
    import torch
    L = 100.0 / 3
    print("case displace blocks", N, M, velocities, flush=True)
    rng = np.random.default_rng(N + M)
    grids, boxes = [], []
    for _ in range(6 if velocities else 3):
        g = gpu.Grid(N, L)
        box = np.zeros((N, N, N + 2))
        box[:, :, :N] = 1.5 * L / N * rng.standard_normal((N, N, N))
        g.set_box(box)
        g.momentum_space = 0
        grids.append(g)
        boxes.append(box)
    lib = gpu.lib()
    n = M ** 3
    q = (np.indices((M, M, M)).reshape(3, -1) * np.float32(L / M)).astype(np.float32)
    far = rng.integers(0, n, 50)
    q[:, far] += np.float32(L) * rng.integers(-3, 4, (3, 50)).astype(np.float32)
    q[:, rng.integers(0, n, 50)] *= np.float32(-0.01)

    def run(pos):
        t = [torch.from_numpy(p.copy()).cuda() for p in pos]
        v = [torch.full_like(t[0], np.nan) for _ in range(3)]
        torch.cuda.synchronize()
        p = [x.data_ptr() for x in t + v]
        if velocities:
            assert lib.mitos_displace_velocity_tsc_dg(*(g.ref() for g in grids), len(pos[0]),
                                                      *p) == 0
        else:
            assert lib.mitos_displace_tsc_dg(*(g.ref() for g in grids), len(pos[0]), *p[:3]) == 0
        return np.stack([x.cpu().numpy() for x in t + (v if velocities else [])])

    blocks = run(q)
    memory = run(np.concatenate([q, q[:, :1]], 1))[:, :n]
    order = rng.permutation(n)
    shuffled = run(q[:, order])
    assert np.array_equal(blocks, memory)
    assert np.array_equal(blocks[:, order], shuffled)
    some = rng.integers(0, n, 400)
    x, y, z = (q[a, some].copy() for a in range(3))
    boxes = np.stack(boxes)
    if velocities:
        want = np.stack([x, y, z, *oracle.displace_velocity_tsc(boxes[:3], boxes[3:], L, x, y, z)])
        want[:3] = x, y, z  # moved in place
    else:
        oracle.displace_tsc(boxes, L, x, y, z)
        want = np.stack([x, y, z])
    # the oracle's operations one by one: at most the last bit of a float
    assert np.all(np.abs(blocks[:, some].astype(np.float64) - want) <= np.spacing(np.abs(want)))
    for g in grids:
        g.free()

"""The learned corrector at the edges of its kernels' voxel blocks: crops
smaller than a block, remainders along every axis at all three resolutions,
no halo, a halo wider than the tile, more crops than one and fewer than the
batch, and inference over volumes that the tiles do not divide.  Against
oracle/unet.py with BF16 rounding where the GPU stores; the two differ by
FP32 accumulation order and the BF16 roundings it flips (2^-9 relative
each), so the bars are the 2e-2 per layer gradient and 1e-2 per output that
test_gpu_corrector.py derives for one size."""
import numpy as np
import pytest

import utr_public_amd as U
from oracle import unet as N

pytestmark = pytest.mark.gpu

SCALE = 0.8


def rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("tile,halo,batch,nb", [(8, 0, 1, 1), (4, 4, 2, 2), (4, 8, 3, 2), (12, 4, 1, 1), (24, 2, 2, 1),
                                                (20, 8, 1, 1)])
def test_forward_and_gradient_at_block_edges(tile, halo, batch, nb):
    import torch
    T = tile + 2 * halo
    print("corrector tile %d halo %d batch %d crops %d" % (tile, halo, batch, nb), flush=True)
    rng = np.random.default_rng(tile * 100 + halo)
    theta = N.init(tile + halo, scale_head=0.3).astype(np.float32)
    vol = rng.normal(0, 1, (nb, T, T, T)).astype(np.float32)
    tgt = (0.5 * vol + rng.normal(0, 0.5, vol.shape)).astype(np.float32)
    c = U.Corrector(tile=tile, halo=halo, batch=batch, seed=5)
    try:
        c.set_params(theta, SCALE)
        dv, dt = torch.from_numpy(vol).cuda(), torch.from_numpy(tgt).cuda()
        out = torch.empty_like(dv)
        c.forward(dv, out)
        assert rel(out.cpu().numpy(), N.forward(theta.astype(np.float64), vol, SCALE, bf=True)[0] / SCALE) <= 1e-2
        loss, g = c.gradient(dv, dt)
        loss2, g2 = c.gradient(dv, dt)
        assert loss == loss2 and np.array_equal(g, g2)
    finally:
        c.close()
    rloss, rg = N.loss_and_grad(theta.astype(np.float64), vol, tgt, tile, halo, SCALE, bf=True)
    assert abs(loss - rloss) <= 1e-3 * rloss
    off = 0
    for ci, co in N.LAYERS:
        nw = 27 * ci * co
        assert rel(g[off:off + nw], rg[off:off + nw]) <= 2e-2, (ci, co)
        assert rel(g[off + nw:off + nw + co], rg[off + nw:off + nw + co]) <= 2e-2, (ci, co)
        off += nw + co
    assert rel(g[off:], rg[off:]) <= 2e-2


@pytest.mark.parametrize("tile,halo,batch,shape", [(8, 4, 3, (17, 8, 11)), (12, 2, 2, (5, 30, 13)), (20, 0, 1, (20, 7, 33))])
def test_apply_ragged_volumes(tile, halo, batch, shape):
    import torch
    print("corrector apply tile %d halo %d volume %s" % (tile, halo, shape), flush=True)
    rng = np.random.default_rng(tile)
    theta = N.init(3, scale_head=0.3).astype(np.float32)
    vol = rng.normal(0, 1, shape).astype(np.float32)
    c = U.Corrector(tile=tile, halo=halo, batch=batch, seed=5)
    try:
        c.set_params(theta, SCALE)
        dv = torch.from_numpy(vol).cuda()
        out = torch.full_like(dv, float("nan"))
        c.apply(dv, out)
        got = out.cpu().numpy()
    finally:
        c.close()
    nt = [-(-n // tile) for n in shape]
    pad = np.zeros([n * tile + 2 * halo for n in nt])
    pad[halo:halo + shape[0], halo:halo + shape[1], halo:halo + shape[2]] = vol
    ref = np.zeros([n * tile for n in nt])
    T = tile + 2 * halo
    for k in np.ndindex(*nt):
        a = [i * tile for i in k]
        crop = pad[a[0]:a[0] + T, a[1]:a[1] + T, a[2]:a[2] + T]
        o = N.forward(theta.astype(np.float64), crop[None], SCALE, bf=True)[0][0] / SCALE
        ref[a[0]:a[0] + tile, a[1]:a[1] + tile, a[2]:a[2] + tile] = o[halo:halo + tile, halo:halo + tile, halo:halo + tile]
    assert rel(got, ref[:shape[0], :shape[1], :shape[2]]) <= 1e-2

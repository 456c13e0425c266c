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


def assert_layers(g, rg):
    off = 0
    for ci, co in N.LAYERS:
        nw = 27 * ci * co
        assert rel(g[off:off + nw], rg[off:off + nw]) <= 2e-2, (ci, co)
        assert rel(g[off + nw:off + nw + co], rg[off + nw:off + nw + co]) <= 2e-2, (ci, co)
        off += nw + co
    assert rel(g[off:], rg[off:]) <= 2e-2


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
    assert_layers(g, rg)


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


@pytest.fixture
def gpu_convolutions(monkeypatch):
    """The oracle's convolutions by torch in FP64 on the GPU, for crops whose
    products take minutes on the CPU."""
    import torch

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a, np.float64)).cuda()

    def taps(x):
        D, H, W = x.shape[1:4]
        p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        for t in range(27):
            z, y, w = t // 9, t // 3 % 3, t % 3
            yield t, p[:, z:z + D, y:y + H, w:w + W].reshape(-1, x.shape[4])

    def conv(x, W, b=None):
        out = torch.zeros((int(np.prod(x.shape[:4])), W.shape[2]), dtype=torch.float64, device="cuda")
        Wd = dev(W)
        for t, v in taps(dev(x)):
            out.addmm_(v, Wd[t])
        out = out.cpu().numpy().reshape(x.shape[:4] + (W.shape[2],))
        return out if b is None else out + b

    def conv_back(x, W, dy):
        Wd, g = dev(W), dev(dy)
        flat = g.reshape(-1, g.shape[4])
        dW = torch.stack([v.T.contiguous() @ flat for _, v in taps(dev(x))])
        dx = torch.zeros((flat.shape[0], x.shape[4]), dtype=torch.float64, device="cuda")
        for t, v in taps(g):
            dx.addmm_(v, Wd[26 - t].T.contiguous())
        return dx.cpu().numpy().reshape(x.shape), dW.cpu().numpy(), flat.sum(0).cpu().numpy()

    monkeypatch.setattr(N, "conv", conv)
    monkeypatch.setattr(N, "conv_back", conv_back)


def blocks(n, e):
    """Blocks of 16 x 8 x 4 voxels of n cubes of edge e: the steps that at most
    768 weight-gradient work-groups share."""
    return n * -(-e // 16) * -(-e // 8) * -(-e // 4)


def test_large_batch_forward_and_gradient(gpu_convolutions):
    """A training batch as large as real ones, with remainders of the blocks at
    the two finer levels: every work-group of the finer weight gradients takes
    several voxel blocks, and thousands share the loss."""
    import torch
    tile, halo, nb = 72, 2, 4
    T = tile + 2 * halo
    assert T % 16 and T % 8 and T // 2 % 16 and T // 2 % 8 and T // 2 % 4
    assert blocks(nb, tile) > 2 * 768
    rng = np.random.default_rng(11)
    theta = N.init(11, scale_head=0.3).astype(np.float32)
    vol = rng.normal(0, 1, (nb, T, T, T)).astype(np.float32)
    tgt = (0.5 * vol + rng.normal(0, 0.5, vol.shape)).astype(np.float32)
    c = U.Corrector(tile=tile, halo=halo, batch=nb, seed=5)
    try:
        c.set_params(theta, SCALE)
        dv, dt = torch.from_numpy(vol).cuda(), torch.from_numpy(tgt).cuda()
        out = torch.empty_like(dv)
        c.forward(dv, out)
        loss, g = c.gradient(dv, dt)
    finally:
        c.close()
    print("large batch: gradient done", flush=True)
    ref = N.forward(theta.astype(np.float64), vol, SCALE, bf=True)[0] / SCALE
    print("large batch: output rel-L2 %.2e" % rel(out.cpu().numpy(), ref), flush=True)
    assert rel(out.cpu().numpy(), ref) <= 1e-2
    rloss, rg = N.loss_and_grad(theta.astype(np.float64), vol, tgt, tile, halo, SCALE, bf=True)
    print("large batch: loss %.6f, oracle %.6f, gradient rel-L2 %.2e" % (loss, rloss, rel(g, rg)), flush=True)
    assert abs(loss - rloss) <= 1e-3 * rloss
    assert_layers(g, rg)


def test_apply_four_tiles_of_64(gpu_convolutions):
    """Inference with the default tile, halo and batch: four crops of 80^3 in
    one pass."""
    import torch
    tile, halo, shape = 64, 8, (70, 60, 128)
    T = tile + 2 * halo
    rng = np.random.default_rng(12)
    theta = N.init(12, scale_head=0.3).astype(np.float32)
    vol = rng.normal(0, 1, shape).astype(np.float32)
    c = U.Corrector(tile=tile, halo=halo, batch=4, seed=5)
    try:
        c.set_params(theta, SCALE)
        dv = torch.from_numpy(vol).cuda()
        out = torch.full_like(dv, float("nan"))
        c.apply(dv, out)
        got = out.cpu().numpy()
    finally:
        c.close()
    pad = np.zeros((2 * tile + 2 * halo, tile + 2 * halo, 2 * tile + 2 * halo))
    pad[halo:halo + 70, halo:halo + 60, halo:halo + 128] = vol
    ref = np.zeros((2 * tile, tile, 2 * tile))
    for k, i in np.ndindex(2, 2):
        a, b = k * tile, i * tile
        o = N.forward(theta.astype(np.float64), pad[None, a:a + T, :, b:b + T], SCALE, bf=True)[0][0] / SCALE
        ref[a:a + tile, :, b:b + tile] = o[halo:halo + tile, halo:halo + tile, halo:halo + tile]
        print("apply: tile", k, i, flush=True)
    assert rel(got, ref[:70, :60]) <= 1e-2

"""The multislice transforms at lengths of powers of two and of the odd
radices, images wider and taller, with the columns the bandwidth limit drops,
against the FP64 oracle; tolerance on the wave as test_gpu_msct.py has it."""
import numpy as np
import pytest

import utr_public_amd as U
from oracle import msct as M
from utr_public_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,mode", [(32, 128, 0), (128, 32, 1), (96, 160, 0), (48, 64, 0), (320, 32, 0),
                                        (64, 384, 0), (512, 64, 0), (192, 256, 1)])
def test_multislice_lengths(nx, ny, mode):
    print("multislice", nx, ny, mode, flush=True)
    ctb = 19.2
    p = U.default_msct_params(nx=nx, ny=ny, ctblength=ctb, deltaz=1.6, kev=200.0, mode=mode, output=2)
    xyz, Z = synth.atoms(nx + ny, 12, "sphere", 5.0, 1.4)
    at = dict(Z=Z, occ=np.ones(len(Z), np.float32),
              **{k: (xyz[:, i] + ctb / 2).astype(np.float32) for i, k in enumerate("xyz")})
    angZ, angY, defocus = [5.0, 250.0], [33.0, 160.0], [0.0, 150.0]
    psi = U.multislice_images(p, at, angZ, angY, defocus)
    ref = M.images(dict(nx=nx, ny=ny, ctb=ctb, deltaz=1.6, kev=200.0, mode=mode), at, np.radians(angZ),
                   np.radians(angY), defocus, output="complex")
    assert np.linalg.norm(psi - ref) / np.linalg.norm(ref) < 1e-5


@pytest.mark.parametrize("nx,ny", [(16, 16), (16, 48), (32, 32), (32, 64), (48, 32), (48, 160), (64, 16)])
def test_potential_of_narrow_rows(nx, ny, monkeypatch):
    """Rows summed a pixel a thread (up to 48 pixels) and eight pixels a thread
    (64), with more atoms in a slice than a workgroup lists at once and a row
    count that the workgroups do not divide: the tile form's bits, the FP64
    oracle to 1e-5, and the oracle's Debye-Waller filter of the raw potential
    to the 1e-5 of test_gpu_msct.py."""
    print("narrow rows", nx, ny, flush=True)
    ctb = 19.2
    p = U.default_msct_params(nx=nx, ny=ny, ctblength=ctb, deltaz=9.6, kev=200.0, output=2)
    rng = np.random.default_rng(nx + 7 * ny)
    n = 600
    xyz = rng.uniform(4.0, 15.0, (3, n)).astype(np.float32)
    at = dict(Z=rng.choice([6, 8], n).astype(np.int32), x=xyz[0], y=xyz[1], z=xyz[2], occ=np.full(n, 0.05, np.float32),
              wobble=np.full(n, 0.1, np.float32))
    ang = [5.0, 250.0], [33.0, 160.0]
    psi = U.multislice_images(p, at, *ang, [0.0])
    monkeypatch.setenv("UTR_MSCT_FUSED", "0")
    assert np.array_equal(psi.view(np.uint32), U.multislice_images(p, at, *ang, [0.0]).view(np.uint32))
    monkeypatch.delenv("UTR_MSCT_FUSED")
    op = dict(nx=nx, ny=ny, ctb=ctb, deltaz=9.6, kev=200.0, mode=0)
    ref = M.images(op, at, np.radians(ang[0]), np.radians(ang[1]), [0.0], output="complex")
    assert np.linalg.norm(psi - ref) / np.linalg.norm(ref) < 1e-5
    got = U.multislice_images(dict(p, output=0, nwobble=1), at, *ang, [0.0])
    ref = M.images(dict(op, nwobble=1, temperature=300.0), at, np.radians(ang[0]), np.radians(ang[1]), [0.0])
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 1e-5


@pytest.mark.parametrize("nx,ny,na", [(384, 96, 24), (320, 128, 17), (512, 64, 33)])
def test_long_lines_of_many_and_of_single_orientations(nx, ny, na):
    """Products of long lines split over more workgroups where there are few
    of them: the orientations together and one by one give the same bits."""
    print("long lines", nx, ny, na, flush=True)
    ctb = 19.2
    p = U.default_msct_params(nx=nx, ny=ny, ctblength=ctb, deltaz=3.2, kev=200.0, output=2)
    xyz, Z = synth.atoms(nx + ny, 12, "sphere", 5.0, 1.4)
    at = dict(Z=Z, occ=np.ones(len(Z), np.float32),
              **{k: (xyz[:, i] + ctb / 2).astype(np.float32) for i, k in enumerate("xyz")})
    angZ, angY = np.linspace(0, 300, na), np.linspace(5, 170, na)
    psi = U.multislice_images(p, at, angZ, angY, [100.0])
    m = U.Multislice(p, at)
    try:
        for a in (0, na // 2, na - 1):
            one = m.images(angZ[a:a + 1], angY[a:a + 1], [100.0])
            assert np.array_equal(one[0].view(np.uint32), psi[a].view(np.uint32)), a
    finally:
        m.close()


def test_batch_is_what_a_pass_takes(monkeypatch):
    """By default a pass holds at most 200 MiB of wave and transmission planes;
    a set budget rules alone, in either direction; the images do not depend on
    it."""
    monkeypatch.delenv("UTR_MSCT_BATCH_BYTES", raising=False)
    p = U.default_msct_params(nx=512, ny=256, ctblength=38.4, deltaz=12.8, kev=200.0)
    at = dict(Z=np.array([6, 8], np.int32), x=np.array([15.0, 20.0], np.float32), y=np.array([17.0, 20.0], np.float32),
              z=np.array([10.0, 25.0], np.float32))
    plane = 512 * 256 * 8
    ang = np.linspace(0.0, 200.0, 5), np.linspace(10.0, 150.0, 5)
    per = None
    for budget in (None, 1 << 30, 2 * 10 ** 7):
        if budget:
            monkeypatch.setenv("UTR_MSCT_BATCH_BYTES", str(budget))
        m = U.Multislice(p, at)
        try:
            print("batch", budget, m.batch, flush=True)
            want = budget // (3 * plane + 2 * 32 + (m.slices + 1) * 8) if budget else (200 << 20) // (2 * plane)
            assert m.batch == want
            img = m.images(*ang, [0.0])
        finally:
            m.close()
        assert per is None or np.array_equal(per, img)
        per = img

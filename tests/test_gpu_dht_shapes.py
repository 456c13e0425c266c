"""DHT kernels at the sizes where their splitting changes, against the FP64
oracle: every transform length as image width or height, widths and heights
that differ, groups of orientations with a remainder.  Tolerance: relative
L2 <= 1e-5, the bound of the FP32 field transforms that test_gpu_dht.py uses."""
import numpy as np
import pytest

import oracle
import utr_public_amd as U

pytestmark = pytest.mark.gpu

TOL = 1e-5


def rel(a, b):
    a = np.asarray(a, np.complex128)
    b = np.asarray(b, np.complex128)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def images(rng, n, nx, ny, sigma=0.05):
    """Smooth random images about 1: noise cut at a quarter of the band."""
    f = np.fft.fft2(rng.standard_normal((n, ny, nx)))
    kx, ky = np.fft.fftfreq(nx)[None, None, :], np.fft.fftfreq(ny)[None, :, None]
    f *= np.exp(-((kx / 0.12) ** 2 + (ky / 0.12) ** 2))
    f[:, 0, 0] = 0
    g = np.fft.ifft2(f).real
    return (1 + sigma * g / g.std()).astype(np.float32)


def case(nx, ny, nz, nrows, seed, general=True, **kw):
    xst = 0.4
    p = U.default_dht_params(nx=nx, ny=ny, xst=xst, zlo=-nz * xst / 2, zhi=nz * xst / 2, **kw)
    rng = np.random.default_rng(seed)
    rows = dict(angZ=rng.uniform(0, 360, nrows) if general else np.zeros(nrows),
                angY=rng.uniform(0, 180, nrows), defocus=rng.uniform(80, 120, nrows))
    return p, rows, images(rng, nrows, nx, ny)


@pytest.mark.parametrize("nx,ny,nz,nrows,method,ap", [
    (16, 512, 5, 3, 3, 0.0), (512, 16, 5, 3, 4, 0.0), (32, 128, 9, 4, 3, 25.0), (128, 32, 8, 4, 4, 25.0),
    (64, 16, 3, 2, 4, 0.0),
    (256, 256, 33, 7, 3, 0.0),  # 17 MB an orientation: launches of five and two
    (256, 64, 35, 5, 4, 0.0),
])
def test_propagation_shapes(nx, ny, nz, nrows, method, ap):
    kw = dict(dzextra=60.0, epsilon=1.0) if method == 3 else dict(dzextra=0.0, asigma=0.06, epsilon=0.02)
    p, rows, imgs = case(nx, ny, nz, nrows, 50 + nx + ny, method=method, escc=1, aobj_mrad=ap, **kw)
    print("shape", nx, ny, nz, nrows, method, ap, flush=True)
    w = np.linspace(0.5, 1.5, nrows).astype(np.float32)  # a wrong orientation's weight shows
    got = U.dht_reconstruct(p, dict(rows, weights=w), imgs)
    assert rel(got, oracle.dht_reconstruct(p, rows, imgs, weights=w)) < TOL


@pytest.mark.parametrize("method", [1, 2])
@pytest.mark.parametrize("nx,ny", [(16, 128), (256, 32), (512, 64), (64, 512)])
def test_series_shapes(nx, ny, method):
    """Methods 1 and 2 on the register transforms, series of two and three
    images; tolerances of test_gpu_dht_series.py."""
    counts = [3, 2, 3]
    rng = np.random.default_rng(nx + ny)
    p, rows, _ = case(nx, ny, 6, 3, nx + 2 * ny, method=method, escc=1, dzextra=100.0,
                      epsilon=0.0 if method == 1 else 1e-8, itermax=6)
    rows.update(counts=counts, defocus=np.concatenate([[150.0, 230.0, 330.0][:c] for c in counts]))
    imgs = images(rng, sum(counts), nx, ny)
    print("series", nx, ny, method, flush=True)
    with U.DhtReconstructor(p, rows) as r:
        r.add_images(imgs)
        vol, waves, its = r.finalize(), r.waves(), r.iterations()
    assert rel(vol, oracle.dht_reconstruct(p, rows, imgs)) < 2e-5
    f = 0
    for a, c in enumerate(counts):
        psi, _, it = oracle.dht_retrieve(p, imgs[f:f + c], rows["defocus"][f:f + c])
        assert np.linalg.norm(waves[a] - psi) / np.linalg.norm(psi - 1) < 1e-4
        assert its[a] == (it if method == 1 else 0)
        f += c


@pytest.mark.parametrize("nx,ny,nz,method,escc", [
    (32, 16, 9, 3, 1), (16, 64, 30, 3, 0), (64, 128, 33, 4, 1), (32, 256, 7, 3, 1), (16, 512, 5, 3, 1),
])
def test_column_splat_shapes(nx, ny, nz, method, escc, monkeypatch):
    """Columns through y: lines shared by four, two and one group of waves, a
    height beyond the columns; the bricks form the same sums bit for bit."""
    kw = dict(dzextra=60.0, epsilon=1.0) if method == 3 else dict(dzextra=0.0, asigma=0.06, epsilon=0.02)
    p, rows, imgs = case(nx, ny, nz, 5, 70 + nx + ny, general=False, method=method, escc=escc, **kw)
    rows["angY"] = np.array([0.0, 90.0, 33.0, 135.0, 180.0])
    print("columns", nx, ny, nz, method, escc, flush=True)
    got = U.dht_reconstruct(p, rows, imgs)
    monkeypatch.setenv("UTR_GRID_FORM", "brick")
    brick = U.dht_reconstruct(p, rows, imgs)
    assert np.array_equal(got.view(np.uint32), brick.view(np.uint32))
    assert rel(got, oracle.dht_reconstruct(p, rows, imgs)) < TOL

"""The brick gridding's point lists at their edges: more points than one list
part (volumes much thinner than the images, where a line's points are closer
than a voxel), more rows than one chunk, one row, rows without and with
rotation about Z mixed, and a rotation centre off the grid, against the FP64
oracle at the 1e-5 of the FP32 form."""
import numpy as np
import pytest

import oracle
import utr_public_amd as U
from utr_public_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-5


def rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("name", ["thin_z", "thin_y", "rows300", "one", "mixed", "shift"])
def test_brick_gridding_point_lists(name):
    nx, ny, nz, rows, kw = {"thin_z": (96, 96, 16, 24, {}), "thin_y": (128, 16, 64, 24, {}),
                            "rows300": (32, 32, 32, 300, {}), "one": (64, 32, 32, 1, {}),
                            "mixed": (48, 48, 48, 30, {}), "shift": (48, 48, 32, 20, dict(dxc=0.7, dyc=-0.3, dzc=0.5))}[name]
    print("brick gridding", name, flush=True)
    xst = 0.4
    p = U.default_params(nx=nx, ny=ny, xst=xst, zlo=-nz * xst / 2, zhi=nz * xst / 2, escc=1, nsr=0.05, **kw)
    rng = np.random.default_rng(len(name))
    angZ = rng.uniform(0, 360, rows)
    if name == "mixed":
        angZ[::2] = 0.0
    angY = np.degrees(np.arccos(2 * rng.uniform(0, 1, rows) - 1))
    r = dict(angZ=angZ, angY=angY, defocus=np.full(rows, 300.0))
    xyz, Z = synth.atoms(3, 20, "cube", min(nx, ny, nz) * xst * 0.4, 1.0, ([6], [1.0]))
    imgs = synth.project(xyz, Z, nx, ny, xst, angZ, angY, dose=400.0, seed=3)
    got = U.reconstruct(p, r, imgs)
    ref = oracle.reconstruct(p, r, imgs)
    assert rel(got, ref) < TOL


@pytest.mark.parametrize("n,extra", [(32, 0), (48, 0), (32, 40), (32, 400)])
def test_brick_gridding_tiny_weights(n, extra, monkeypatch):
    """Rows on and a millionth of a voxel beside the grid planes, with and
    without rotation about Z, alone (more points with tiny corners than a
    brick's record holds) and under many random rows (voxels that have larger
    weights as well): the sampled voxels are the oracle's, and V3/Samp3 keeps
    its precision where only tiny weights fall (no noise filter: such voxels
    count in the volume as any other)."""
    monkeypatch.setenv("UTR_GRID_FORM", "brick")
    rng = np.random.default_rng(n + extra)
    angZ = np.concatenate([[0.0, 0.0, 0.0, 90.0, 1e-6, 90.000001, 45.0, 1e-6], rng.uniform(0, 360, extra)])
    angY = np.concatenate([[0.0, 90.0, 89.999999, 0.0, 0.0, 90.0, 89.999999, 180.000002],
                           np.degrees(np.arccos(rng.uniform(-1, 1, extra)))])
    rows = len(angZ)
    print("tiny weights", n, rows, flush=True)
    xst = 0.4
    p = U.default_params(nx=n, ny=n, xst=xst, zlo=-n * xst / 2, zhi=n * xst / 2, escc=0, nsr=0.0)
    r = dict(angZ=angZ, angY=angY, defocus=np.full(rows, 300.0))
    xyz, Z = synth.atoms(4, 20, "cube", n * xst * 0.4, 1.0, ([6], [1.0]))
    imgs = synth.project(xyz, Z, n, n, xst, angZ, angY, dose=400.0, seed=4)
    ref, S = oracle.reconstruct(p, r, imgs, samp=True)
    if extra < 400:
        assert ((S > 0) & (S < 2.0 ** -20)).sum() > 100
    with U.Reconstructor(p, r) as rec:
        rec.keep_sampling()
        rec.add_images(imgs)
        got = rec.finalize()
        S32 = rec.sampling()
    assert np.array_equal(S32 == 0, S == 0)
    low = (S > 0) & (S < 2.0 ** -20)
    assert np.abs(S32[low] / S[low] - 1.0).max(initial=0.0) < 1e-4
    assert rel(got, ref) < TOL

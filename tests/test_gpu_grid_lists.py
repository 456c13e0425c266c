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

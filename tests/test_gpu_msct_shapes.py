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

"""The gridding for every number of complex slices in a group (one to four, and a
second group) and chunks of a tile's list from one to several, against the FP64
oracle.

Tolerance: float32 2e-6 (the transforms' 1e-6 and the split products' 2^-20);
16-bit, six values rounded to storage, each at most half a unit, independent:
below sqrt(6) halves, asserted at 4 (9.8e-4 float16, 7.8e-3 bfloat16)."""
import numpy as np
import pytest
import torch

from oracle import fourierrec_fp64 as fr
from tomocupy_amd import FourierRec, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['float32', 'float16', 'bfloat16'])
@pytest.mark.parametrize('nz', [1, 2, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize('chunk', [0, 64, 1024])
def test_slices_and_chunks(dtype, nz, chunk):
    n, nproj = 128, 150
    rng = np.random.default_rng(nz)
    theta = synth.angles(nproj)
    data = rng.standard_normal((nz, nproj, n)).astype(np.float32)
    ref = fr.backprojection(data, theta)
    tdt = getattr(torch, dtype)
    rec = FourierRec(n, nproj, nz, torch.from_numpy(theta).cuda(), dtype=dtype, grid_chunk=chunk)
    obj = torch.empty((nz, n, n), device='cuda', dtype=tdt)
    rec.backprojection(obj, torch.from_numpy(data).cuda().to(tdt))
    got = obj.float().cpu().numpy()
    tol = {'float32': 2e-6, 'float16': 4 * 2.0**-12, 'bfloat16': 4 * 2.0**-9}[dtype]
    for z in range(nz):
        err = np.linalg.norm(got[z] - ref[z]) / np.linalg.norm(ref[z])
        assert err <= tol, (z, err)
    rec.free()

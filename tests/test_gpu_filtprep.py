"""The fused filter and detector transform in each of its forms (several rows a
wave, one row a wave or more, 256 threads a row, run-time sizes; a last row
group that is not full; one slice without a partner) against the FP64 filter
followed by the same plan's backprojection.

Tolerance: per side at most 16 float32 passes of about 1e-7 each of the row's
rms, random, and the same gridding and image transforms: below 1e-6, asserted at
2e-6; 'none' keeps the low frequencies and its rows are not differenced, the same."""
import numpy as np
import pytest
import torch

from oracle import filter_fp64 as ff
from tomocupy_amd import BackprojFunctions, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,nproj,nz,filt', [
    (256, 603, 7, 'ramp'), (256, 30, 2, 'none'), (512, 601, 8, 'shepp'), (512, 13, 3, 'ramp'),
    (512, 577, 8, 'none'), (768, 401, 8, 'ramp'), (768, 20, 1, 'ramp'), (1024, 385, 8, 'parzen'),
    (1024, 11, 2, 'ramp'), (1280, 9, 3, 'ramp'), (1536, 9, 2, 'none'), (2048, 7, 3, 'ramp'),
    (2304, 5, 2, 'ramp'), (2560, 5, 2, 'shepp'), (4096, 3, 1, 'ramp'), (300, 40, 3, 'ramp'),
    (1000, 9, 2, 'none'), (2448, 5, 3, 'ramp')])
def test_fused_filter(n, nproj, nz, filt):
    rng = np.random.default_rng(n + nproj)
    theta = torch.from_numpy(synth.angles(nproj)).cuda()
    data = rng.standard_normal((nz, nproj, n)).astype(np.float32)
    data += np.linspace(3, 1, n, dtype=np.float32)
    sht = rng.uniform(-2, 2, nz).astype(np.float32)
    centre = n / 2 + 0.25
    bf = BackprojFunctions(n, nproj, nz, theta, centre, 'float32', filt)
    ne = 4 * n
    rows = ff.fbp_filter_center(data, ff.calc_filter(ne, filt), ne, centre, sht)
    ref = torch.empty((nz, n, n), device='cuda')
    bf.cl_rec.backprojection(ref, torch.from_numpy(rows.astype(np.float32)).cuda())
    obj = torch.empty_like(ref)
    bf.fbp_filter_backprojection(obj, torch.from_numpy(data).cuda(),
                                 sht=torch.from_numpy(sht).cuda())
    err = float((obj - ref).norm() / ref.norm())
    print('n=%d %d angles %d slices %s %.3g' % (n, nproj, nz, filt, err))
    assert err <= 2e-6
    bf.free()

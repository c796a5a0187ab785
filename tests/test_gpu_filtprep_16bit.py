"""The fused filter and detector transform of 16-bit plans in the forms that long
scans take (several rows a wave, one row a wave; a last row group that is not full)
against the FP64 filter followed by a float32 plan's backprojection.

Tolerance: six values rounded to storage on the way (spectrum, two gridding
factors, grid, R, image), each at most half a unit (2^-12 float16, 2^-9 bfloat16)
and independent: below sqrt(6) of that, asserted at 4.  (float16 spectra hold filtered
rows; the unfiltered mean of 768 columns times their scale of 2^8 is past its range.)"""
import numpy as np
import pytest
import torch

from oracle import filter_fp64 as ff
from tomocupy_amd import BackprojFunctions, FourierRec, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,nproj,nz,filt,dtype', [
    (256, 603, 7, 'ramp', 'float16'), (256, 603, 7, 'ramp', 'bfloat16'),
    (512, 601, 8, 'shepp', 'float16'), (512, 601, 8, 'shepp', 'bfloat16'),
    (768, 401, 8, 'hann', 'float16'), (768, 401, 8, 'none', 'bfloat16'),
    (1024, 385, 8, 'parzen', 'float16'), (1024, 385, 8, 'parzen', 'bfloat16')])
def test_fused_filter(n, nproj, nz, filt, dtype):
    rng = np.random.default_rng(n + nproj)
    td = getattr(torch, dtype)
    theta = torch.from_numpy(synth.angles(nproj)).cuda()
    data = rng.standard_normal((nz, nproj, n)) + np.linspace(3, 1, n)
    data = torch.from_numpy(data.astype(np.float32)).to(td)
    centre = n / 2 + 0.25
    bf = BackprojFunctions(n, nproj, nz, theta, centre, dtype, filt)
    ne = bf.ne
    rows = ff.fbp_filter_center(data.double().numpy(), ff.calc_filter(ne, filt), ne, centre)
    ref = torch.empty((nz, n, n), device='cuda')
    FourierRec(n, nproj, nz, theta).backprojection(ref, torch.from_numpy(rows.astype(np.float32)).cuda())
    obj = torch.empty((nz, n, n), device='cuda', dtype=td)
    bf.fbp_filter_backprojection(obj, data.cuda())
    err = float((obj.float() - ref).norm() / ref.norm())
    print('n=%d %d angles %d slices %s %s %.3g' % (n, nproj, nz, filt, dtype, err))
    assert err <= 4 * (2.0**-12 if dtype == 'float16' else 2.0**-9)
    bf.free()

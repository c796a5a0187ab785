"""Column passes whose run-time plan differs from the row pass's, so that a
workgroup takes twice the columns (two, four and eight; with and without a large
prime), and compiled 16-bit ones on a column-blocked array, against the FP64 oracle.

Tolerance: as for every run-time plan, three transforms of at most five passes of
about 1e-7 of the row's rms each, random: below 1e-6, asserted at 2e-6; float16 six
values rounded to storage by at most half a unit of 2^-11: asserted at 4 halves."""
import numpy as np
import pytest
import torch

from oracle import fourierrec_fp64 as fr
from tomocupy_amd import FourierRec, synth

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


WIDTHS = [816, 840, 912, 1060, 1560, 1776, 2060, 3096, 3456]
CASES = [(n, dt) for n in WIDTHS for dt in ('float32', 'float16')]
CASES += [(n, 'float16') for n in (640, 768, 1152, 1280)]


@pytest.mark.parametrize('n,dtype', CASES)
def test_backprojection_and_projection(n, dtype):
    nproj, nz = 3, 2
    rng = np.random.default_rng(n)
    theta = synth.angles(nproj, 0.3)
    tdt = getattr(torch, dtype)
    rec = FourierRec(n, nproj, nz, torch.from_numpy(theta).cuda(), dtype=dtype)
    data = rng.standard_normal((nz, nproj, n)).astype(np.float32)
    obj = torch.empty((nz, n, n), device='cuda', dtype=tdt)
    rec.backprojection(obj, torch.from_numpy(data).cuda().to(tdt))
    e1 = _rel(obj.float().cpu().numpy(), fr.backprojection(data, theta))
    print('n=%d %s backprojection %.3g' % (n, dtype, e1))
    assert e1 <= (2e-6 if dtype == 'float32' else 4 * 2.0**-12)
    if dtype != 'float32':
        return
    img = rng.standard_normal((nz, n, n)).astype(np.float32)
    sino = torch.empty((nz, nproj, n), device='cuda')
    rec.forward(sino, torch.from_numpy(img).cuda())
    e2 = _rel(sino.cpu().numpy(), fr.forward(img, theta))
    print('n=%d projection %.3g' % (n, e2))
    assert e2 <= 2e-6

"""Every pass instance of the run-time transforms that an accepted length reaches
(test_runtime_plans.py derives them): the radices 2 .. 18 and 20 and the large
primes as first and as later pass, of the image transforms and of 16-bit rows; the
rule's radices with padded output, padded input and plain, of float32 rows.  Against
the FP64 oracle.

Tolerance: three transforms of at most five passes, a pass adding about 1e-7
relative to the row's rms (random): below 1e-6, asserted at 2e-6; rows, two
transforms, the same; bfloat16 rows are exact in storage before and rounded once
after, by at most half a unit of 2^-8: asserted at 2^-8."""
import numpy as np
import pytest
import torch

from oracle import filter_fp64 as ff
from oracle import fourierrec_fp64 as fr
from tomocupy_amd import FourierRec, synth

pytestmark = pytest.mark.gpu

WIDTHS = [20, 22, 32, 48, 128, 168, 182, 200, 270, 286, 324, 340, 494, 646, 900, 1102]
ROWS16 = [20, 24, 32, 96, 128, 196, 200, 216, 242, 250, 270, 294, 416, 442, 646, 722, 972, 1800,
          12324]
ROWS32 = [22, 26, 34, 38, 64, 76, 128, 152, 220, 304, 416, 630, 952, 1792]


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize('n', WIDTHS)
def test_images(n):
    nproj, nz = 5, 3
    rng = np.random.default_rng(n)
    theta = synth.angles(nproj, 0.3)
    rec = FourierRec(n, nproj, nz, torch.from_numpy(theta).cuda(), fft='generic')
    data = rng.standard_normal((nz, nproj, n)).astype(np.float32)
    obj = torch.empty((nz, n, n), device='cuda')
    rec.backprojection(obj, torch.from_numpy(data).cuda())
    e1 = _rel(obj.cpu().numpy(), fr.backprojection(data, theta))
    img = rng.standard_normal((nz, n, n)).astype(np.float32)
    sino = torch.empty((nz, nproj, n), device='cuda')
    rec.forward(sino, torch.from_numpy(img).cuda())
    e2 = _rel(sino.cpu().numpy(), fr.forward(img, theta))
    print('n=%d backprojection %.3g projection %.3g' % (n, e1, e2))
    assert e1 <= 2e-6 and e2 <= 2e-6


@pytest.mark.parametrize('ne,dtype', [(ne, 'bfloat16') for ne in ROWS16]
                         + [(ne, 'float32') for ne in ROWS32])
def test_rows(ne, dtype):
    from tomocupy_amd.fbp_filter import FBPFilter
    rng = np.random.default_rng(ne)
    td = getattr(torch, dtype)
    x = torch.from_numpy(rng.standard_normal((2, 3, ne)).astype(np.float32)).to(td)
    w = rng.standard_normal((2, ne // 2 + 1)) + 1j * rng.standard_normal((2, ne // 2 + 1))
    w = (w / ne).astype(np.complex64)
    flt = FBPFilter(ne, 3, 2, dtype, n_unpadded=20)
    d = x.cuda()
    flt.filter(d, torch.from_numpy(w).cuda())
    err = _rel(d.double().cpu().numpy(), ff.filter_padded(x.double().numpy(), w.astype(np.complex128)))
    print('ne=%d %s %.3g' % (ne, dtype, err))
    assert err <= (2e-6 if dtype == 'float32' else 2.0**-8)

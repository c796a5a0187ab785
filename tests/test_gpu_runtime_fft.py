"""The run-time FFT plans (widths without a compiled transform) against the FP64
oracle: every radix 2..18 and 20 as first and later pass, several butterflies
per thread, prime passes of 8 and 12 output pairs a wave, one pass only, two
equal large primes, and the column pass's interleaved transforms.

Tolerance: three transforms of at most five passes each, a pass adding about
1e-7 relative to the row's rms (twiddle and butterfly rounding, random): below
1e-6; asserted at 2e-6."""
import numpy as np
import pytest
import torch

from oracle import fourierrec_fp64 as fr
from tomocupy_amd import FourierRec, synth

pytestmark = pytest.mark.gpu

WIDTHS = [22, 38, 62, 68, 78, 126, 140, 148, 254, 300, 336, 374, 552, 836, 1000, 1444, 1566,
          2032, 2448, 2604]


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize('n', WIDTHS)
def test_backprojection_and_projection(n):
    nproj, nz = 7, 3
    rng = np.random.default_rng(n)
    theta = synth.angles(nproj, 0.3)
    th = torch.from_numpy(theta).cuda()
    rec = FourierRec(n, nproj, nz, th)
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


@pytest.mark.parametrize('n,ne', [(40, 62), (100, 254), (128, 13718), (200, 15138), (512, 15776)])
def test_filter_rows(n, ne):
    # ne beyond 4n: prime passes of 16 pairs a wave, three equal primes
    from oracle import filter_fp64 as ff
    from tomocupy_amd.fbp_filter import FBPFilter
    rng = np.random.default_rng(ne)
    data = rng.standard_normal((2, 3, ne)).astype(np.float32)
    w = (rng.standard_normal((2, ne // 2 + 1)) + 1j * rng.standard_normal((2, ne // 2 + 1)))
    w = w.astype(np.complex64)
    flt = FBPFilter(ne, 3, 2, n_unpadded=n)
    d = torch.from_numpy(data).cuda()
    flt.filter(d, torch.from_numpy(w).cuda())
    err = _rel(d.cpu().numpy(), ff.filter_padded(data.astype(np.float64), w.astype(np.complex128)))
    print('ne=%d filter %.3g' % (ne, err))
    assert err <= 2e-6

"""The column passes that exchange one component at a time (2n >= 2048), each
with its number of columns and both layouts of the array between the passes,
against the FP64 oracle.

Tolerances: float32 as a chain of three transforms of at most four passes, each
about 1e-7 of the row's rms: below 1e-6, asserted at 2e-6. 16-bit: six values
rounded to storage on the way (data, spectrum, two gridding factors, grid, R,
image), each at most half a unit (2^-12 float16, 2^-9 bfloat16) and
independent: below sqrt(6) of that, asserted at 4 units-in-the-last-place
halves (9.8e-4, 7.8e-3)."""
import numpy as np
import pytest
import torch

from oracle import fourierrec_fp64 as fr
from tomocupy_amd import FourierRec, synth

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize('n,dtype', [(1024, 'float32'), (1280, 'float32'), (1536, 'float32'),
                                     (1920, 'float32'), (2304, 'float32'), (2560, 'float32'),
                                     (512, 'float16'), (1024, 'float16'), (2048, 'float16'),
                                     (640, 'bfloat16'), (1280, 'bfloat16'), (2560, 'bfloat16')])
def test_backprojection_and_projection(n, dtype):
    nproj, nz = 5, 2
    rng = np.random.default_rng(n)
    theta = synth.angles(nproj, 0.3)
    tdt = getattr(torch, dtype)
    rec = FourierRec(n, nproj, nz, torch.from_numpy(theta).cuda(), dtype=dtype)
    data = rng.standard_normal((nz, nproj, n)).astype(np.float32)
    obj = torch.empty((nz, n, n), device='cuda', dtype=tdt)
    rec.backprojection(obj, torch.from_numpy(data).cuda().to(tdt))
    e1 = _rel(obj.float().cpu().numpy(), fr.backprojection(data, theta))
    print('n=%d %s backprojection %.3g' % (n, dtype, e1))
    assert e1 <= {'float32': 2e-6, 'float16': 4 * 2.0**-12, 'bfloat16': 4 * 2.0**-9}[dtype]
    if dtype != 'float32':
        return
    img = rng.standard_normal((nz, n, n)).astype(np.float32)
    sino = torch.empty((nz, nproj, n), device='cuda')
    rec.forward(sino, torch.from_numpy(img).cuda())
    e2 = _rel(sino.cpu().numpy(), fr.forward(img, theta))
    print('n=%d projection %.3g' % (n, e2))
    assert e2 <= 2e-6

"""The separate filter's compiled row lengths (every power of two from 256, for
float32 also those with factors 3 and 5), padded and unpadded rows, a row without
a partner, a width that is not a quarter of the length, against the FP64 oracle.

Tolerance: float32 two transforms of at most six passes, each about 1e-7 of the
row's rms, random: asserted at 1e-6.  16-bit rows are exact in storage before and
rounded once after, by at most half a unit: asserted at 2^-11 (float16) and 2^-8
(bfloat16) of the rms."""
import numpy as np
import pytest
import torch

from oracle import filter_fp64 as ff

pytestmark = pytest.mark.gpu

TOL = {'float32': 1e-6, 'float16': 2.0**-11, 'bfloat16': 2.0**-8}
CASES = [(ne, n, dt) for ne, n in ((256, 64), (512, 100), (1024, 256), (2048, 512), (4096, 1000),
                                   (8192, 2048), (16384, 4096))
         for dt in ('float32', 'float16', 'bfloat16')]
CASES += [(ne, ne // 4, 'float32') for ne in (768, 1280, 1536, 2304, 2560, 3072, 3840, 4608, 5120,
                                              6144, 7680, 9216, 10240, 12288, 15360)]


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize('ne,n,dtype', CASES)
def test_rows(ne, n, dtype):
    from tomocupy_amd.fbp_filter import FBPFilter
    rng = np.random.default_rng(ne)
    td = getattr(torch, dtype)
    nz, nproj = 2, 3
    flt = FBPFilter(ne, nproj, nz, dtype, n_unpadded=n)
    x = torch.from_numpy(rng.standard_normal((nz, nproj, ne)).astype(np.float32)).to(td)
    w = rng.standard_normal((nz, ne // 2 + 1)) + 1j * rng.standard_normal((nz, ne // 2 + 1))
    w = (w / ne).astype(np.complex64)
    d = x.cuda()
    flt.filter(d, torch.from_numpy(w).cuda())
    ref = ff.filter_padded(x.double().numpy(), w.astype(np.complex128))
    e1 = _rel(d.double().cpu().numpy(), ref)
    y = x[:, :, :n].contiguous()
    wf = (0.5 + rng.random(ne // 2 + 1)).astype(np.float32) / ne
    sht = rng.uniform(-2, 2, nz).astype(np.float32)
    d = y.cuda()
    flt.filter_center(d, torch.from_numpy(wf).cuda(), n / 2 + 0.75, torch.from_numpy(sht).cuda())
    ref = ff.fbp_filter_center(y.double().numpy(), wf.astype(np.float64), ne, n / 2 + 0.75, sht)
    e2 = _rel(d.double().cpu().numpy(), ref)
    print('ne=%d n=%d %s padded %.3g unpadded %.3g' % (ne, n, dtype, e1, e2))
    assert e1 <= TOL[dtype] and e2 <= TOL[dtype]
